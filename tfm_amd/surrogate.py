"""Contact-map surrogate: a 1-D convolutional encoder over a chain's binned
het/LAD pattern and the run's (volume fraction, eps_het, eps_lamina), with a
pairwise outer-product head for the log10 contact-probability map and a
pooled head for the radial density.

Every forward and backward step runs on the library's kernels
(include/ccpmi_nn.h): BF16 GEMMs on the matrix cores with FP32
accumulation, FP32 element-wise work, AdamW on FP32 master weights with BF16
copies. torch only allocates the device buffers and provides the stream.

Network (activations x[c, b L + l]):
  h1 = gelu(W1 * x + b1), h_k = h_{k-1} + gelu(W_k * h_{k-1} + b_k)  (conv k=3)
  U = Wu h, V = Wv h; raw[b](i, j) = U_b(:, i) . V_b(:, j) / sqrt(d)
  S = (raw + raw^T) / 2 + dist[|i - j|] + c0          (log10 P map)
  rd = Wr mean_l h + br                                (radial density)
"""
import ctypes
import math

import numpy as np
import torch

from .ccp import lib

NN_EXPORTS = (
    "ccp_nn_gemm", "ccp_nn_im2col", "ccp_nn_col2im", "ccp_nn_bias_gelu", "ccp_nn_gelu_back", "ccp_nn_pair_map",
    "ccp_nn_pair_loss", "ccp_nn_mean_pool", "ccp_nn_pool_back", "ccp_nn_rd_loss", "ccp_nn_cast_bf16", "ccp_nn_adamw",
    "ccp_nn_input", "ccp_nn_fwd", "ccp_nn_pair", "ccp_nn_pool", "ccp_nn_small", "ccp_nn_pair_bands", "ccp_nn_pair_grad",
    "ccp_nn_rd_grad", "ccp_nn_duv", "ccp_nn_back", "ccp_nn_wgrad_tiles", "ccp_nn_wgrad", "ccp_nn_wgrad_far", "ccp_nn_reduce",
    "ccp_nn_pack", "ccp_nn_adamw_flat",
)


def _struct(name, pointers, ints=(), longs=()):
    return type(name, (ctypes.Structure,), {"_fields_": [(k, ctypes.c_void_p) for k in pointers] +
                                            [(k, ctypes.c_long) for k in longs] + [(k, ctypes.c_int) for k in ints]})


FwdArgs = _struct("FwdArgs", ("A0", "A1", "X", "bias", "res", "pre", "y", "ob", "ot"),
                  ("M", "M0", "Kp", "Cs", "P", "Ps", "L", "Os", "O1"))
BackArgs = _struct("BackArgs", ("W", "G", "dpooled", "pre", "dh", "gb", "gt", "dbias"),
                   ("C", "Cs", "Cr", "Kr", "Gs", "P", "Ps", "L", "B", "V1", "keep"))
Segment = _struct("Segment", ("src", "dst"), (), ("n", "stride", "parts"))
WgradJob = _struct("WgradJob", ("G", "X", "dst0", "dst1"), ("M", "M0", "C", "taps", "P", "Ps"))
Weight = _struct("Weight", ("w", "wb", "fwd", "back"), ("M", "C", "taps", "Kp", "Cr", "Kr"))


_bound = False


def _nn():
    global _bound
    L = lib()
    if not _bound:
        vp, f, i, lg = ctypes.c_void_p, ctypes.c_float, ctypes.c_int, ctypes.c_long
        L.ccp_nn_gemm.argtypes = [vp, vp, vp, vp, i, i, i, i] + [lg] * 9 + [f, f, vp]
        L.ccp_nn_im2col.argtypes = [vp, vp, i, i, i, vp]
        L.ccp_nn_col2im.argtypes = [vp, vp, i, i, i, f, vp]
        L.ccp_nn_bias_gelu.argtypes = [vp, vp, vp, vp, vp, i, lg, vp]
        L.ccp_nn_gelu_back.argtypes = [vp, vp, vp, vp, vp, i, lg, vp]
        L.ccp_nn_pair_map.argtypes = [vp, vp, vp, vp, i, i, vp]
        L.ccp_nn_pair_loss.argtypes = [vp, vp, vp, vp, vp, vp, vp, vp, i, i, f, vp]
        L.ccp_nn_mean_pool.argtypes = [vp, vp, vp, i, i, i, vp]
        L.ccp_nn_pool_back.argtypes = [vp, vp, i, i, i, vp]
        L.ccp_nn_rd_loss.argtypes = [vp, vp, vp, vp, vp, vp, vp, i, i, f, vp]
        L.ccp_nn_cast_bf16.argtypes = [vp, vp, lg, vp]
        L.ccp_nn_adamw.argtypes = [vp, vp, vp, vp, vp, lg, f, f, f, f, f, i, vp]
        L.ccp_nn_input.argtypes = [vp, vp, vp, i, i, i, i, vp, vp]
        L.ccp_nn_fwd.argtypes = [vp, i, vp]
        L.ccp_nn_pair.argtypes = [vp, i, vp, vp, vp, i, i, f, vp]
        L.ccp_nn_pool.argtypes = [vp, vp, vp, i, i, i, i, i, i, vp]
        L.ccp_nn_small.argtypes = [vp, vp, vp, i, i, i, i, i, i, vp]
        L.ccp_nn_pair_bands.argtypes = [i]
        L.ccp_nn_pair_grad.argtypes = [vp, vp, vp, vp, vp, vp, i, i, i, f, vp]
        L.ccp_nn_rd_grad.argtypes = [vp, vp, vp, vp, vp, vp, vp, i, i, i, i, f, vp]
        L.ccp_nn_duv.argtypes = [vp, vp, vp, vp, i, i, i, i, i, i, f, vp]
        L.ccp_nn_back.argtypes = [vp, i, vp]
        L.ccp_nn_wgrad_tiles.argtypes = [i, i]
        L.ccp_nn_wgrad.argtypes = L.ccp_nn_wgrad_far.argtypes = [vp, vp, i, i, i, vp]
        L.ccp_nn_reduce.argtypes = [vp, i, vp]
        L.ccp_nn_pack.argtypes = [vp, i, vp]
        L.ccp_nn_adamw_flat.argtypes = [vp, vp, vp, vp, lg, lg, f, f, f, f, f, i, vp]
        _bound = True
    return L


def _p(t):
    """Device address of a tensor (None for none)."""
    return t.data_ptr() if t is not None else None


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _ok(rc, what):
    if rc != 0:
        raise RuntimeError(f"{what} failed ({rc})")


def gemm(A, B, M, N, K, sa, sb, sc, C=None, Cb=None, batch=1, alpha=1.0, beta=0.0):
    """Strided batched BF16 GEMM; sa = (batch, m, k) strides of A, sb = (batch,
    k, n) of B, sc = (batch, m, n) of C/Cb."""
    _ok(_nn().ccp_nn_gemm(_p(A), _p(B), _p(C), _p(Cb), M, N, K, batch, *sa, *sb, *sc, alpha, beta, _stream()),
        "gemm")


def bf16_like(t):
    return torch.empty(t.shape, dtype=torch.int16, device=t.device)


def _up(n, k):
    return (n + k - 1) // k * k


def _table(structs):
    """The structures as one device array (read by the kernels that take a table)."""
    raw = b"".join(bytes(t) for t in structs)
    return torch.frombuffer(bytearray(raw), dtype=torch.uint8).cuda()


def _at(tensors, names):
    """Addresses of the entries of a dict of tensors."""
    return [tensors[k].data_ptr() for k in names]


class Surrogate:
    """Weights (FP32 masters, BF16 copies) and buffers for batches of B
    sequences of L bins with c_in input channels.

    The parameters, their gradients and AdamW's moments are views of one flat
    array each, the weight matrices first (they alone decay). include/ccpmi_nn.h
    gives the layouts of the activations.

    An entry of p, g, m or v may be given another tensor (or another storage):
    the kernels' arguments hold addresses, so each call compares those it uses
    with the entries' and takes the new ones. As ever, new weight matrices
    reach the products at the next step, which casts them. pb is written then
    for a caller's own products; the network reads its packed copies."""

    def __init__(self, c_in=5, width=256, n_layers=6, d=64, L=128, rd_bins=32, B=64, seed=0, params=None):
        self.c_in, self.width, self.n_layers, self.d, self.L, self.rd_bins, self.B = \
            c_in, width, n_layers, d, L, rd_bins, B
        dev = torch.device("cuda")
        if params is None:
            import_seed = np.random.default_rng(seed)
            params = {"W1": import_seed.normal(0, 1 / math.sqrt(3 * c_in), (width, 3 * c_in)), "b1": np.zeros(width)}
            for k in range(2, n_layers + 1):
                params[f"W{k}"] = import_seed.normal(0, 0.5 / math.sqrt(3 * width), (width, 3 * width))
                params[f"b{k}"] = np.zeros(width)
            params["Wu"] = import_seed.normal(0, 1 / math.sqrt(width), (d, width))
            params["Wv"] = import_seed.normal(0, 1 / math.sqrt(width), (d, width))
            params["Wr"] = import_seed.normal(0, 1 / math.sqrt(width), (rd_bins, width))
            params["br"] = np.zeros(rd_bins)
            params["dist"] = np.zeros(L)
            params["c0"] = np.zeros(1)
        self.names = list(params.keys())
        host = {k: np.ascontiguousarray(v, np.float32) for k, v in params.items()}
        order = [k for k in self.names if k.startswith("W")] + [k for k in self.names if not k.startswith("W")]
        at, off = 0, {}
        for k in order:
            off[k] = at
            at += _up(host[k].size, 64)
            if k.startswith("W"):
                self._n_decay = at
        self._flat = [torch.zeros(at, dtype=torch.float32, device=dev) for _ in range(4)]
        view = lambda t: {k: t[off[k]:off[k] + host[k].size].view(host[k].shape) for k in self.names}
        self.p, self.g, self.m, self.v = (view(t) for t in self._flat)
        self._numel, self._off = {k: host[k].size for k in self.names}, off
        for k in self.names:
            self.p[k].copy_(torch.from_numpy(host[k]))
        self.pb = {k: bf16_like(v) for k, v in self.p.items() if k.startswith("W")}
        self.t = 0
        self._alloc_packed()
        self._alloc(B)
        self._cast_weights()

    # what holds addresses: left out of copies and made anew for them
    _BOUND = ("_flat_at", "_pack", "_pack_at", "_fwd", "_bias_at", "_back", "_jobs", "_seg", "_grad_at")

    def __getstate__(self):
        return {k: v for k, v in self.__dict__.items() if k not in self._BOUND}

    def __setstate__(self, state):
        self.__dict__.update(state)
        self._bind()

    def _bind(self):
        self._flat_at = [[t.data_ptr() + 4 * self._off[k] for k in self.names] for t in self._flat]
        self._bind_pack()
        self._bind_forward()
        self._bind_backward()
        self._bind_grads()

    def _own(self, group, names, dtype=torch.float32):
        """Entries whose addresses go into a kernel's arguments: whole contiguous device arrays."""
        for k in names:
            t = group[k]
            if t.dtype != dtype or not t.is_cuda or not t.is_contiguous() or t.numel() != self._numel[k]:
                raise ValueError(f"{k} must be a contiguous {dtype} cuda tensor of {self._numel[k]} entries")

    def _alloc_packed(self):
        """The packed weight copies."""
        W, C1, d, O = self.width, self.c_in, self.d, self.rd_bins
        h = lambda *s: torch.zeros(s, dtype=torch.int16, device="cuda")
        Cr, Kr, Kd = _up(W, 64), _up(W, 32), _up(d, 32)
        self._wf = {1: h(Cr, 3 * _up(C1, 16))}
        self._wt = {}
        for k in range(2, self.n_layers + 1):
            self._wf[k], self._wt[k] = h(Cr, 3 * _up(W, 16)), h(3, Cr, Kr)
        self._wf["u"], self._wf["v"] = h(d, _up(W, 64)), h(d, _up(W, 64))
        self._wt["uv"] = h(2, Cr, Kd)
        self._wf["r"], self._wt["r"] = h(O, _up(W, 64)), h(Cr, _up(O, 32))
        self._weights = [k for k in self.names if k.startswith("W")]

    def _bind_pack(self):
        """The table that fills the packed copies from p."""
        W, C1, d, O = self.width, self.c_in, self.d, self.rd_bins
        Cr, Kr, Kd = _up(W, 64), _up(W, 32), _up(d, 32)
        self._own(self.p, self._weights)
        self._own(self.pb, self._weights, torch.int16)
        tab = []
        for k in range(1, self.n_layers + 1):
            C, wt = (C1, None) if k == 1 else (W, self._wt[k])
            tab.append(Weight(_p(self.p[f"W{k}"]), _p(self.pb[f"W{k}"]), _p(self._wf[k]), _p(wt), W, C, 3,
                              3 * _up(C, 16), Cr, Kr))
        for j, k in enumerate("uv"):
            tab.append(Weight(_p(self.p["W" + k]), _p(self.pb["W" + k]), _p(self._wf[k]), _p(self._wt["uv"][j]), d, W,
                              1, _up(W, 64), Cr, Kd))
        tab.append(Weight(_p(self.p["Wr"]), _p(self.pb["Wr"]), _p(self._wf["r"]), _p(self._wt["r"]), O, W, 1,
                          _up(W, 64), Cr, _up(O, 32)))
        self._pack = _table(tab), len(tab)
        self._pack_at = _at(self.p, self._weights) + _at(self.pb, self._weights)

    def _alloc(self, B):
        self.B = B
        dev = torch.device("cuda")
        W, L, d, n = self.width, self.L, self.d, self.n_layers
        Ls, Cs, C1s, ds = _up(L, 8), _up(W, 64), _up(self.c_in, 16), _up(d, 32)
        P = B * L
        Ps = _up(P, 16)
        self._ls, self._ds, self._ps = Ls, ds, Ps
        f = lambda *s: torch.zeros(s, dtype=torch.float32, device=dev)
        h = lambda *s: torch.zeros(s, dtype=torch.int16, device=dev)
        # forward; pre and the channel rows are read by the backward pass only
        self.xb, self.xt = h(self.c_in, Ps), h(P, C1s)
        self.hs = [f(W, Ps), f(W, Ps)]
        self.ht = [h(P, Cs), h(P, Cs)]
        self.pre = {k: f(W, Ps) for k in range(1, n + 1)}
        self.hb = {k: h(W, Ps) for k in range(1, n + 1)}
        self.uvb, self.uvt = h(2 * d, Ps), h(P, 2 * ds)
        self.S = f(B, L, L)
        Bs, Or = _up(B, 16), _up(self.rd_bins, 32)
        self._bs, self._or, self._cs = Bs, Or, Cs
        self.pooledb, self.pooledt = h(W, Bs), h(B, Cs)
        self.rd = f(self.rd_bins, B)
        self._biases = [f"b{k}" for k in range(1, n + 1)]
        # backward: every layer keeps its gradient's channel rows for the weight gradients' one launch
        bands, tiles = _nn().ccp_nn_pair_bands(L), (P + 127) // 128
        self.grawb = h(B, L, Ls)
        self.duvb, self.duvt = h(2 * d, Ps), h(P, 2 * ds)
        self.dh = f(W, Ps)
        self.gb = {k: h(W, Ps) for k in range(1, n + 1)}
        self.gt = [h(P, Cs), h(P, Cs)]
        self.grdb, self.grdt = h(self.rd_bins, Bs), h(B, Or)
        self.dpooled = f(W, B)
        self.loss = f(1)
        self._gdist, self._gc0 = f(B * bands, L), f(B * bands)
        self._dbias = {k: f(tiles, W) for k in range(1, n + 1)}
        self._bind()

    def _bind_forward(self):
        """Arguments of the layers' products, with the biases of p."""
        W, L, d, n, B = self.width, self.L, self.d, self.n_layers, self.B
        C1s, Cs, ds, P, Ps = _up(self.c_in, 16), self._cs, self._ds, B * L, self._ps
        self._own(self.p, self._biases)
        self._fwd = {}
        for keep in (False, True):
            for k in range(1, n + 1):
                first = k == 1
                self._fwd[keep, k] = FwdArgs(
                    _p(self._wf[k]), None, _p(self.xt if first else self.ht[k % 2]), _p(self.p[f"b{k}"]),
                    None if first else _p(self.hs[k % 2]), _p(self.pre[k]) if keep else None,
                    _p(self.hs[(k + 1) % 2]), _p(self.hb[k]) if keep else None, _p(self.ht[(k + 1) % 2]),
                    W, W, 3 * _up(self.c_in if first else W, 16), C1s if first else Cs, P, Ps, L, Cs, 0)
            self._fwd[keep, "uv"] = FwdArgs(
                _p(self._wf["u"]), _p(self._wf["v"]), _p(self.ht[(n + 1) % 2]), None, None, None, None,
                _p(self.uvb) if keep else None, _p(self.uvt), 2 * d, d, _up(W, 64), Cs, P, Ps, L, 2 * ds, ds)
        self._bias_at = _at(self.p, self._biases)

    def _bind_backward(self):
        """Arguments of the layers' gradients."""
        W, L, d, n, B = self.width, self.L, self.d, self.n_layers, self.B
        Cs, ds, P, Ps = self._cs, self._ds, B * L, self._ps
        Cr = _up(W, 64)
        self._back = {n: BackArgs(_p(self._wt["uv"]), _p(self.duvt), _p(self.dpooled), _p(self.pre[n]), _p(self.dh),
                                  _p(self.gb[n]), _p(self.gt[n % 2]), _p(self._dbias[n]), W, Cs, Cr, _up(d, 32),
                                  2 * ds, P, Ps, L, B, ds, int(n > 1))}
        for k in range(n - 1, 0, -1):
            self._back[k] = BackArgs(_p(self._wt[k + 1]), _p(self.gt[(k + 1) % 2]), None, _p(self.pre[k]), _p(self.dh),
                                     _p(self.gb[k]), _p(self.gt[k % 2]), _p(self._dbias[k]), W, Cs, Cr, _up(W, 32),
                                     Cs, P, Ps, L, B, 0, int(k > 1))

    def _bind_grads(self):
        """Tables of the weight gradients and of the sums that go into g."""
        W, L, d, n, B = self.width, self.L, self.d, self.n_layers, self.B
        P, Ps, Bs = B * L, self._ps, self._bs
        bands, tiles = _nn().ccp_nn_pair_bands(L), (P + 127) // 128
        dev = torch.device("cuda")
        self._own(self.g, self.names)
        jobs, at = [], [0]
        for k in list(range(1, n + 1)):
            X, C = (self.xb, self.c_in) if k == 1 else (self.hb[k - 1], W)
            jobs.append(WgradJob(_p(self.gb[k]), _p(X), _p(self.g[f"W{k}"]), None, W, W, C, 3, P, Ps))
        jobs.append(WgradJob(_p(self.duvb), _p(self.hb[n]), _p(self.g["Wu"]), _p(self.g["Wv"]), 2 * d, d, W, 1,
                             P, Ps))
        jobs.append(WgradJob(_p(self.grdb), _p(self.pooledb), _p(self.g["Wr"]), None, self.rd_bins, self.rd_bins, W, 1,
                             B, Bs))
        for j in jobs:
            at.append(at[-1] + _nn().ccp_nn_wgrad_tiles(j.M, j.C))
        self._jobs = _table(jobs), torch.tensor(at, dtype=torch.int32, device=dev), len(jobs), at[-1]
        seg = [Segment(_p(self._dbias[k]), _p(self.g[f"b{k}"]), W, W, tiles) for k in range(1, n + 1)]
        seg.append(Segment(_p(self._gdist), _p(self.g["dist"]), L, L, B * bands))
        seg.append(Segment(_p(self._gc0), _p(self.g["c0"]), 1, 1, B * bands))
        self._seg = _table(seg), len(seg)
        self._grad_at = _at(self.g, self.names)

    def _cast_weights(self):
        if _at(self.p, self._weights) + _at(self.pb, self._weights) != self._pack_at:
            self._bind_pack()
        _ok(_nn().ccp_nn_pack(_p(self._pack[0]), self._pack[1], _stream()), "pack")

    # ------------------------------------------------------------ forward
    @staticmethod
    def _check_input(t, shape, name):
        if t.dtype != torch.float32 or not t.is_cuda or not t.is_contiguous() or tuple(t.shape) != tuple(shape):
            raise ValueError(f"{name} must be a contiguous float32 cuda tensor of shape {tuple(shape)}")

    def forward(self, x, keep=True):
        """x: [c_in, B L] float32 (cuda). Returns (S [B, L, L], rd [rd_bins, B]) on the device.
        keep: also store what loss_backward reads."""
        return self._forward(x, keep)

    def _forward(self, x, keep, loss=None):
        """forward, with the loss (when given) at zero behind it."""
        self._check_input(x, (self.c_in, self.B * self.L), "x")
        N = _nn()
        B, L, W, d = self.B, self.L, self.width, self.d
        if _at(self.p, self._biases) != self._bias_at:
            self._bind_forward()
        s = _stream()
        _ok(N.ccp_nn_input(_p(x), _p(self.xb) if keep else None, _p(self.xt), self.c_in, _up(self.c_in, 16), B * L,
                           self._ps, _p(loss), s), "input")
        for k in range(1, self.n_layers + 1):
            _ok(N.ccp_nn_fwd(ctypes.byref(self._fwd[keep, k]), 1, s), "conv")
        _ok(N.ccp_nn_fwd(ctypes.byref(self._fwd[keep, "uv"]), 0, s), "heads")
        # S from raw[b](i, j) = sum_c U[c, b, i] V[c, b, j] / sqrt(d)
        _ok(N.ccp_nn_pair(_p(self.uvt), self._ds, _p(self.p["dist"]), _p(self.p["c0"]), _p(self.S), L, B,
                          1.0 / math.sqrt(d), s), "pair")
        _ok(N.ccp_nn_pool(_p(self.hs[(self.n_layers + 1) % 2]), _p(self.pooledb), _p(self.pooledt), W, B, L, self._ps,
                          self._bs, self._cs, s), "pool")
        _ok(N.ccp_nn_small(_p(self._wf["r"]), _p(self.pooledt), _p(self.rd), self.rd_bins, B, self._cs, self._cs,
                           self._cs, B, s), "radial head")
        return self.S, self.rd

    def predict(self, x):
        S, rd = self.forward(x, keep=False)
        rd = rd + self.p["br"][:, None]
        return S, rd

    # ------------------------------------------------------------ backward
    def zero_grad(self):
        self._flat[1].zero_()
        for k, at in zip(self.names, self._flat_at[1]):
            if self.g[k].data_ptr() != at:
                self.g[k].zero_()

    def loss_backward(self, x, T, T_rd, w_pair=1.0, w_rd=1.0):
        """Forward, loss and gradients into self.g; returns the loss (device scalar)."""
        N = _nn()
        B, L, W, d, n = self.B, self.L, self.width, self.d, self.n_layers
        Ls, Ps = self._ls, self._ps
        s = _stream()
        self._check_input(T, (B, L, L), "T")
        self._check_input(T_rd, (self.rd_bins, B), "T_rd")
        if _at(self.g, self.names) != self._grad_at:
            self._bind_grads()
        self._forward(x, True, self.loss)
        _ok(N.ccp_nn_pair_grad(_p(self.S), _p(T), _p(self.grawb), _p(self._gdist), _p(self._gc0), _p(self.loss), L, Ls,
                               B, w_pair, s), "pair_grad")
        _ok(N.ccp_nn_rd_grad(_p(self.rd), _p(self.p["br"]), _p(T_rd), _p(self.grdb), _p(self.grdt), _p(self.g["br"]),
                             _p(self.loss), self.rd_bins, B, self._bs, self._or, w_rd, s), "rd_grad")
        _ok(N.ccp_nn_small(_p(self._wt["r"]), _p(self.grdt), _p(self.dpooled), W, B, self._or, self._or, self._or, B,
                           s), "pooled gradient")
        # dU_b = a V_b graw_b^T, dV_b = a U_b graw_b
        _ok(N.ccp_nn_duv(_p(self.uvb), _p(self.grawb), _p(self.duvb), _p(self.duvt), d, self._ds, L, Ls, B, Ps,
                         1.0 / math.sqrt(d), s), "duv")
        for k in range(n, 0, -1):
            _ok(N.ccp_nn_back(ctypes.byref(self._back[k]), int(k == n), s), "back")
        wgrad = N.ccp_nn_wgrad if Ps < 1 << 26 else N.ccp_nn_wgrad_far
        _ok(wgrad(_p(self._jobs[0]), _p(self._jobs[1]), self._jobs[2], self._jobs[3], L, s), "wgrad")
        _ok(N.ccp_nn_reduce(_p(self._seg[0]), self._seg[1], s), "reduce")
        return self.loss

    def step(self, lr=1e-3, b1=0.9, b2=0.999, eps=1e-8, wd=1e-4):
        self.t += 1
        groups = self.p, self.g, self.m, self.v
        if [_at(t, self.names) for t in groups] == self._flat_at:
            p, g, m, v = (_p(t) for t in self._flat)
            _ok(_nn().ccp_nn_adamw_flat(p, g, m, v, self._flat[0].numel(), self._n_decay, lr, b1, b2, eps, wd, self.t,
                                        _stream()), "adamw")
        else:
            for t in groups:
                self._own(t, self.names)
            for k in self.names:
                p, g, m, v = (_p(t[k]) for t in groups)
                _ok(_nn().ccp_nn_adamw(p, g, m, v, None, self._numel[k], lr, b1, b2, eps,
                                       wd if k.startswith("W") else 0.0, self.t, _stream()), "adamw")
        self._cast_weights()

    def state_dict(self):
        return {k: v.detach().cpu().numpy() for k, v in self.p.items()}
