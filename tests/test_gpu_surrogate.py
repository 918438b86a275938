"""GPU parity of the surrogate's kernels: the strided batched BF16 GEMM on the
matrix cores against float64 products of the same bfloat16 values, and the
network's forward pass and every gradient against the numpy oracle with the
same bfloat16 rounding points; then a short training run."""
import copy
import math
import pickle

import numpy as np
import pytest
import torch

import surrogate_oracle as so
from gpu_common import step
from tfm_amd import surrogate as sg

pytestmark = pytest.mark.gpu


def to_bf16_dev(a):
    """float array -> (device int16 words of its bfloat16 rounding, float64 values)."""
    r = so.bf16(a)
    words = (r.astype(np.float32).view(np.uint32) >> 16).astype(np.uint16).view(np.int16)
    return torch.tensor(words, device="cuda"), r


@pytest.mark.parametrize("M,N,K,batch,layout", [(64, 64, 16, 1, "nn"), (70, 33, 19, 1, "nn"), (128, 96, 200, 1, "nt"),
                                                (45, 130, 77, 1, "tn"), (32, 40, 24, 5, "nn"), (17, 17, 9, 3, "tt")])
def test_gemm_matches_float64(M, N, K, batch, layout):
    step(f"gemm {M}x{N}x{K} batch {batch} {layout}")
    rng = np.random.default_rng(M * N + K)
    a = rng.normal(size=(batch, M, K)) if layout[0] == "n" else rng.normal(size=(batch, K, M))
    b = rng.normal(size=(batch, K, N)) if layout[1] == "n" else rng.normal(size=(batch, N, K))
    A, av = to_bf16_dev(a)
    B, bv = to_bf16_dev(b)
    Am = av if layout[0] == "n" else av.transpose(0, 2, 1)
    Bm = bv if layout[1] == "n" else bv.transpose(0, 2, 1)
    want = 0.5 * np.einsum("bmk,bkn->bmn", Am, Bm) + 2.0
    sa = (M * K, K, 1) if layout[0] == "n" else (M * K, 1, M)
    sb = (K * N, N, 1) if layout[1] == "n" else (K * N, 1, K)
    C = torch.full((batch, M, N), 1.0, dtype=torch.float32, device="cuda")
    Cb = torch.zeros((batch, M, N), dtype=torch.int16, device="cuda")
    sg.gemm(A, B, M, N, K, sa, sb, (M * N, N, 1), C=C, Cb=Cb, batch=batch, alpha=0.5, beta=2.0)
    torch.cuda.synchronize()
    got = C.cpu().numpy().astype(np.float64)
    scale = 0.5 * np.einsum("bmk,bkn->bmn", np.abs(Am), np.abs(Bm)) + 2.0
    assert np.all(np.abs(got - want) <= 1e-6 * scale + 1e-6)
    gotb = (Cb.cpu().numpy().view(np.uint16).astype(np.uint32) << 16).view(np.float32)
    assert np.array_equal(gotb, so.bf16(got).astype(np.float32))


def cfg():
    return dict(c_in=5, width=32, n_layers=3, d=8, L=16, rd_bins=8, B=3)


def problem(seed=0):
    c = cfg()
    rng = np.random.default_rng(seed)
    p = so.init_params(c["c_in"], c["width"], c["n_layers"], c["d"], c["L"], c["rd_bins"], seed=seed)
    for k in p:
        p[k] = (p[k] + 0.05 * rng.normal(size=p[k].shape)).astype(np.float32).astype(np.float64)
    x = rng.normal(size=(c["c_in"], c["B"] * c["L"])).astype(np.float32).astype(np.float64)
    T = rng.normal(size=(c["B"], c["L"], c["L"]))
    T = (0.5 * (T + T.transpose(0, 2, 1))).astype(np.float32).astype(np.float64)
    T_rd = rng.normal(size=(c["rd_bins"], c["B"])).astype(np.float32).astype(np.float64)
    return c, p, x, T, T_rd


def rel(a, b):
    return np.linalg.norm(np.ravel(a) - np.ravel(b)) / max(np.linalg.norm(np.ravel(b)), 1e-30)


def test_forward_and_gradients_match_oracle():
    step("surrogate forward/backward vs oracle")
    c, p, x, T, T_rd = problem()
    net = sg.Surrogate(params=p, **c)
    dev = lambda a: torch.tensor(np.asarray(a, np.float32), device="cuda")
    net.zero_grad()
    loss = net.loss_backward(dev(x), dev(T), dev(T_rd), w_pair=1.0, w_rd=0.5)
    torch.cuda.synchronize()
    want_loss, g, S, rd = so.loss_and_grads(p, x, T, T_rd, c["B"], c["L"], c["n_layers"], 1.0, 0.5,
                                            round_bf16=True)
    assert rel(net.S.cpu().numpy(), S) < 1e-3
    assert rel(net.rd.cpu().numpy(), rd) < 1e-3
    assert float(loss.item()) == pytest.approx(want_loss, rel=1e-3)
    for k in p:
        err = rel(net.g[k].cpu().numpy(), g[k])
        step(f"  grad {k}: rel err {err:.2e}")
        assert err < 2e-2, k


@pytest.mark.parametrize("c", [dict(c_in=3, width=36, n_layers=2, d=5, L=13, rd_bins=7, B=5),
                               dict(c_in=5, width=100, n_layers=3, d=33, L=50, rd_bins=33, B=3),
                               dict(c_in=17, width=65, n_layers=1, d=16, L=40, rd_bins=1, B=1),
                               dict(c_in=1, width=256, n_layers=2, d=64, L=129, rd_bins=32, B=2)])
def test_ragged_sizes_match_oracle(c):
    # channels, positions, samples and heads off every tile size: outputs and
    # every gradient against the oracle, with the tolerances above
    step(f"surrogate sizes {c}")
    rng = np.random.default_rng(c["width"])
    p = so.init_params(c["c_in"], c["width"], c["n_layers"], c["d"], c["L"], c["rd_bins"], seed=1)
    for k in p:
        p[k] = (p[k] + 0.05 * rng.normal(size=p[k].shape)).astype(np.float32).astype(np.float64)
    x = rng.normal(size=(c["c_in"], c["B"] * c["L"])).astype(np.float32).astype(np.float64)
    T = rng.normal(size=(c["B"], c["L"], c["L"])).astype(np.float32)
    T = (0.5 * (T + T.transpose(0, 2, 1))).astype(np.float64)
    T_rd = rng.normal(size=(c["rd_bins"], c["B"])).astype(np.float32).astype(np.float64)
    net = sg.Surrogate(params=p, **c)
    dev = lambda a: torch.tensor(np.asarray(a, np.float32), device="cuda")
    S0, rd0 = (t.clone() for t in net.predict(dev(x)))
    net.zero_grad()
    loss = net.loss_backward(dev(x), dev(T), dev(T_rd), w_pair=1.0, w_rd=0.5)
    want_loss, g, S, rd = so.loss_and_grads(p, x, T, T_rd, c["B"], c["L"], c["n_layers"], 1.0, 0.5, round_bf16=True)
    assert torch.equal(S0, net.S) and torch.equal(rd0, net.rd)
    assert rel(net.S.cpu().numpy(), S) < 1e-3 and rel(net.rd.cpu().numpy(), rd) < 1e-3
    assert float(loss.item()) == pytest.approx(want_loss, rel=1e-3)
    for k in p:
        assert rel(net.g[k].cpu().numpy(), g[k]) < 2e-2, k


def test_training_reduces_loss():
    step("surrogate training")
    c, p, x, T, T_rd = problem(3)
    net = sg.Surrogate(params=p, **c)
    dev = lambda a: torch.tensor(np.asarray(a, np.float32), device="cuda")
    X, TT, TR = dev(x), dev(T), dev(T_rd)
    losses = []
    for it in range(300):
        net.zero_grad()
        losses.append(float(net.loss_backward(X, TT, TR).item()))
        net.step(lr=3e-3)
    assert np.isfinite(losses).all()
    assert losses[-1] < 0.2 * losses[0]


def test_loss_outlives_a_forward_pass():
    # the returned loss is a buffer that the next loss_backward fills; a
    # forward pass or a prediction in between leaves it alone
    step("surrogate loss after a forward pass")
    c, p, x, T, T_rd = problem(4)
    net = sg.Surrogate(params=p, **c)
    dev = lambda a: torch.tensor(np.asarray(a, np.float32), device="cuda")
    loss = net.loss_backward(dev(x), dev(T), dev(T_rd))
    first = loss.item()
    assert first > 0
    net.forward(dev(2 * x))
    net.predict(dev(x))
    assert loss.item() == first
    assert net.loss_backward(dev(x), dev(T), dev(T_rd)).item() == pytest.approx(first, rel=1e-6)


@pytest.mark.parametrize("how", ["entry", "storage", "dict"])
def test_replaced_tensors_are_the_ones_used(how):
    # a parameter, gradient or moment given as another tensor (an entry of its
    # dict, its storage, a whole dict) is what the kernels read and write: two
    # steps are bit for bit those of a net that was built with the values
    step(f"surrogate with replaced tensors ({how})")
    c, p, x, T, T_rd = problem(5)
    _, q, _, _, _ = problem(6)
    dev = lambda a: torch.tensor(np.asarray(a, np.float32), device="cuda")
    want, net = sg.Surrogate(params=q, **c), sg.Surrogate(params=p, **c)
    given = {}
    for group in ("p", "g", "m", "v"):
        new = {k: torch.full((2 * v.numel() + 1,), -9.0, device="cuda")[1:1 + v.numel()].view(v.shape)
               for k, v in getattr(net, group).items()}
        for k, t in new.items():
            t.copy_(getattr(want, group)[k])
            if how == "entry":
                getattr(net, group)[k] = t
            elif how == "storage":
                getattr(net, group)[k].data = t
        if how == "dict":
            setattr(net, group, new)
        given[group] = new
    for n in (want, net):
        n.step(lr=0.0)  # casts the weights
        n.t = 0
    for _ in range(2):
        for n in (want, net):
            n.zero_grad()
            n.loss_backward(dev(x), dev(T), dev(T_rd))
            n.step(lr=3e-3)
    assert torch.equal(net.forward(dev(x))[0], want.forward(dev(x))[0])
    for group, new in given.items():
        for k, t in new.items():
            assert torch.equal(t, getattr(want, group)[k]), (group, k)
    assert all(np.array_equal(a, b) for a, b in zip(net.state_dict().values(), want.state_dict().values()))
    net.p["b1"] = dev(np.zeros(3))
    with pytest.raises(ValueError, match="b1 must be"):
        net.predict(dev(x))


@pytest.mark.parametrize("L,B", [(3, 65536), (16, 65535 + 70)])
def test_more_samples_than_a_grid_dimension(L, B):
    # the pair map and its gradients go out in several launches: outputs and
    # gradients against the oracle, with the tolerances above
    step(f"surrogate with {B} samples of {L} bins")
    c = dict(c_in=2, width=8, n_layers=1, d=4, L=L, rd_bins=3, B=B)
    rng = np.random.default_rng(L)
    p = so.init_params(c["c_in"], c["width"], c["n_layers"], c["d"], c["L"], c["rd_bins"], seed=2)
    f32 = lambda a: a.astype(np.float32).astype(np.float64)
    p = {k: f32(v + 0.05 * rng.normal(size=v.shape)) for k, v in p.items()}
    # the last samples weigh as much in the loss as all others
    scale = np.where(np.arange(B) >= 65535, math.sqrt(65535 / (B - 65535)), 1.0)
    x = f32(rng.normal(size=(c["c_in"], B * L)))
    T = rng.normal(size=(B, L, L)) * scale[:, None, None]
    T = f32(0.5 * (T + T.transpose(0, 2, 1)))
    T_rd = f32(rng.normal(size=(c["rd_bins"], B)))
    net = sg.Surrogate(params=p, **c)
    dev = lambda a: torch.tensor(np.asarray(a, np.float32), device="cuda")
    net.zero_grad()
    loss = net.loss_backward(dev(x), dev(T), dev(T_rd), w_pair=1.0, w_rd=0.5)
    want_loss, g, S, rd = so.loss_and_grads(p, x, T, T_rd, B, L, c["n_layers"], 1.0, 0.5, round_bf16=True)
    got = net.S.cpu().numpy()
    assert rel(got, S) < 1e-3 and rel(got[65535:], S[65535:]) < 1e-3 and rel(net.rd.cpu().numpy(), rd) < 1e-3
    assert float(loss.item()) == pytest.approx(want_loss, rel=1e-3)
    for k in p:
        err = rel(net.g[k].cpu().numpy(), g[k])
        step(f"  grad {k}: rel err {err:.2e}")
        assert err < 2e-2, k


@pytest.mark.parametrize("taps,L", [(1, 64), (3, 64), (3, 13)])
@pytest.mark.parametrize("Ps", [96, (1 << 26) + 5 * (1 << 20)])
def test_weight_gradients_of_long_rows(taps, L, Ps):
    # rows so long that the last of a tile of 32 lie more than 32 bits of bytes
    # behind the first: small whole numbers in the first P columns, exact sums
    step(f"weight gradients, {taps} taps, samples of {L}, rows of {Ps}")
    M, C, P = 33, 34, 64
    rng = np.random.default_rng(taps * L)
    far = Ps >= 1 << 26
    G, X = (torch.empty((n, Ps), dtype=torch.int16, device="cuda") for n in (M, C))
    g, x = rng.integers(-4, 5, (M, P)).astype(float), rng.integers(-4, 5, (C, P)).astype(float)
    for t, v in ((G, g), (X, x)):
        t[:, :96] = 0
        t[:, :P] = to_bf16_dev(v)[0]
    dst = torch.full((M, taps * C), 3.0, device="cuda")
    nn = sg._nn()
    n_tiles = nn.ccp_nn_wgrad_tiles(M, C)
    tab = sg._table([sg.WgradJob(G.data_ptr(), X.data_ptr(), dst.data_ptr(), None, M, M, C, taps, P, Ps)])
    first = torch.tensor([0, n_tiles], dtype=torch.int32, device="cuda")
    run = nn.ccp_nn_wgrad_far if far else nn.ccp_nn_wgrad
    assert run(tab.data_ptr(), first.data_ptr(), 1, n_tiles, L, sg._stream()) == 0
    want = np.full((M, C, taps), 3.0)
    for t in range(taps):
        for p in range(P):
            q = p + t - 1 if taps == 3 else p
            if 0 <= q < P and q // L == p // L:
                want[:, :, t] += np.outer(g[:, p], x[:, q])
    assert np.array_equal(dst.cpu().numpy(), want.reshape(M, taps * C))
    del G, X
    torch.cuda.empty_cache()


def single_operations(net, x, T, T_rd, w_pair, w_rd):
    """The network's step from the library's single operations (an im2col matrix
    and one product a layer): outputs, loss and gradients. Weights as net's."""
    N, B, L, W, d, n, O = sg._nn(), net.B, net.L, net.width, net.d, net.n_layers, net.rd_bins
    P, st = B * L, sg._stream()
    f = lambda *s: torch.zeros(s, dtype=torch.float32, device="cuda")
    h = lambda *s: torch.zeros(s, dtype=torch.int16, device="cuda")
    a = lambda *t: [None if v is None else v.data_ptr() if torch.is_tensor(v) else v for v in t]

    def call(name, *args):
        assert getattr(N, "ccp_nn_" + name)(*a(*args), st) == 0, name

    pb = {k: h(*net.p[k].shape) for k in net.names if k.startswith("W")}
    for k, t in pb.items():
        call("cast_bf16", net.p[k], t, t.numel())
    xb = h(*x.shape)
    call("cast_bf16", x, xb, x.numel())
    inp, res, c = xb, None, net.c_in
    cols, pre = {}, {}
    for k in range(1, n + 1):
        cols[k], pre[k], y, yb = h(3 * c, P), f(W, P), f(W, P), h(W, P)
        call("im2col", inp, cols[k], c, B, L)
        sg.gemm(pb[f"W{k}"], cols[k], W, P, 3 * c, (0, 3 * c, 1), (0, P, 1), (0, P, 1), C=pre[k])
        call("bias_gelu", pre[k], net.p[f"b{k}"], res, y, yb, W, P)
        inp, res, c = yb, y, W
    U, V, raw, S = h(d, P), h(d, P), f(B, L, L), f(B, L, L)
    for k, t in (("Wu", U), ("Wv", V)):
        sg.gemm(pb[k], inp, d, P, W, (0, W, 1), (0, P, 1), (0, P, 1), Cb=t)
    alpha = 1.0 / math.sqrt(d)
    sg.gemm(U, V, L, L, d, (L, 1, P), (L, P, 1), (L * L, L, 1), C=raw, batch=B, alpha=alpha)
    call("pair_map", raw, net.p["dist"], net.p["c0"], S, L, B)
    pooled, pooledb, rd = f(W, B), h(W, B), f(O, B)
    call("mean_pool", res, pooled, pooledb, W, B, L)
    sg.gemm(pb["Wr"], pooledb, O, B, W, (0, W, 1), (0, B, 1), (0, B, 1), C=rd)
    g, loss = {k: f(*net.p[k].shape) for k in net.names}, f(1)
    gS, graw, grawb, grd, grdb = f(B, L, L), f(B, L, L), h(B, L, L), f(O, B), h(O, B)
    call("pair_loss", S, T, gS, graw, grawb, g["dist"], g["c0"], loss, L, B, w_pair)
    call("rd_loss", rd, net.p["br"], T_rd, grd, grdb, g["br"], loss, O, B, w_rd)
    dU, dV, dh = h(d, P), h(d, P), f(W, P)
    sg.gemm(V, grawb, d, L, L, (L, P, 1), (L * L, 1, L), (L, P, 1), Cb=dU, batch=B, alpha=alpha)
    sg.gemm(U, grawb, d, L, L, (L, P, 1), (L * L, L, 1), (L, P, 1), Cb=dV, batch=B, alpha=alpha)
    for k, t in (("Wu", dU), ("Wv", dV)):
        sg.gemm(t, inp, d, W, P, (0, P, 1), (0, 1, P), (0, W, 1), C=g[k], beta=1.0)
    sg.gemm(pb["Wu"], dU, W, P, d, (0, 1, W), (0, P, 1), (0, P, 1), C=dh)
    sg.gemm(pb["Wv"], dV, W, P, d, (0, 1, W), (0, P, 1), (0, P, 1), C=dh, beta=1.0)
    sg.gemm(grdb, pooledb, O, W, B, (0, B, 1), (0, 1, B), (0, W, 1), C=g["Wr"], beta=1.0)
    dpooled = f(W, B)
    sg.gemm(pb["Wr"], grdb, W, B, O, (0, 1, W), (0, B, 1), (0, B, 1), C=dpooled)
    call("pool_back", dpooled, dh, W, B, L)
    gp, gpb, dcols = f(W, P), h(W, P), f(3 * W, P)
    for k in range(n, 0, -1):
        call("gelu_back", pre[k], dh, gp, gpb, g[f"b{k}"], W, P)
        K = 3 * (net.c_in if k == 1 else W)
        sg.gemm(gpb, cols[k], W, K, P, (0, P, 1), (0, 1, P), (0, K, 1), C=g[f"W{k}"], beta=1.0)
        if k > 1:
            sg.gemm(pb[f"W{k}"], gpb, K, P, W, (0, 1, K), (0, P, 1), (0, P, 1), C=dcols)
            call("col2im", dcols, dh, W, B, L, 1.0)
    return S, rd, loss, g


@pytest.mark.parametrize("c", [cfg(), dict(c_in=3, width=36, n_layers=2, d=5, L=13, rd_bins=7, B=5),
                               dict(c_in=5, width=100, n_layers=4, d=33, L=64, rd_bins=33, B=9)])
def test_single_operations_give_the_networks_numbers(c):
    # the library's single operations and the network's fused kernels contract
    # in the same order: outputs and weight gradients bit for bit, the sums over
    # positions (biases, distance terms) as FP32 sums in two orders, and one step
    # of AdamW tensor by tensor
    step(f"single operations, sizes {c}")
    rng = np.random.default_rng(c["width"])
    p = so.init_params(c["c_in"], c["width"], c["n_layers"], c["d"], c["L"], c["rd_bins"], seed=3)
    p = {k: v + 0.05 * rng.normal(size=v.shape) for k, v in p.items()}
    dev = lambda a: torch.tensor(np.asarray(a, np.float32), device="cuda")
    x, T_rd = dev(rng.normal(size=(c["c_in"], c["B"] * c["L"]))), dev(rng.normal(size=(c["rd_bins"], c["B"])))
    T = rng.normal(size=(c["B"], c["L"], c["L"]))
    T = dev(0.5 * (T + T.transpose(0, 2, 1)))
    net = sg.Surrogate(params=p, **c)
    S, rd, loss, g = single_operations(net, x, T, T_rd, 1.0, 0.5)
    net.zero_grad()
    got = net.loss_backward(x, T, T_rd, w_pair=1.0, w_rd=0.5)
    assert torch.equal(net.S, S) and torch.equal(net.rd, rd)
    assert got.item() == pytest.approx(loss.item(), rel=1e-5)
    for k in net.names:
        if k.startswith("W"):
            assert torch.equal(net.g[k], g[k]), k
        else:
            assert rel(net.g[k].cpu().numpy(), g[k].cpu().numpy()) < 1e-5, k
    for k in net.names:
        w, m, v, wb = net.p[k].clone(), torch.zeros_like(g[k]), torch.zeros_like(g[k]), sg.bf16_like(g[k])
        grad = net.g[k].contiguous()
        args = [t.data_ptr() for t in (w, grad, m, v, wb)]
        assert sg._nn().ccp_nn_adamw(*args, w.numel(), 1e-3, 0.9, 0.999, 1e-8, 1e-4 if k.startswith("W") else 0.0, 1,
                                     sg._stream()) == 0
        p[k] = w, wb
    net.step()
    for k in net.names:
        assert torch.equal(net.p[k], p[k][0]), k
        if k.startswith("W"):
            assert torch.equal(net.pb[k], p[k][1]), k


@pytest.mark.parametrize("how", ["deepcopy", "pickle"])
def test_a_copied_net_is_a_net_of_its_own(how):
    # a copy trains on its own tensors, bit for bit as a net built from the same
    # parameters, and leaves the original's alone
    step(f"surrogate copied by {how}")
    c, p, x, T, T_rd = problem(7)
    dev = lambda a: torch.tensor(np.asarray(a, np.float32), device="cuda")
    X, TT, TR = dev(x), dev(T), dev(T_rd)
    net, want = sg.Surrogate(params=p, **c), sg.Surrogate(params=p, **c)

    def train(n):
        n.zero_grad()
        n.loss_backward(X, TT, TR)
        n.step(lr=3e-3)

    train(net)
    train(want)
    before = net.state_dict()
    out = net.predict(X)[0].clone()
    other = copy.deepcopy(net) if how == "deepcopy" else pickle.loads(pickle.dumps(net))
    for n in (other, want):
        for _ in range(2):
            train(n)
    for group in ("p", "g", "m", "v"):
        for k in net.names:
            assert torch.equal(getattr(other, group)[k], getattr(want, group)[k]), (group, k)
    assert torch.equal(other.predict(X)[0], want.predict(X)[0])
    assert all(np.array_equal(a, b) for a, b in zip(net.state_dict().values(), before.values()))
    assert torch.equal(net.predict(X)[0], out)
