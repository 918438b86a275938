"""GPU parity of the analysis kernels (ccp's chrana.cu per-frame work) with
the oracle: frame observables and radial density (FP64 sums, tolerance in
the test), d(s)/P(s) and ccp's packed 4-bead contact map (ccp's FP32
arithmetic, bit-exact), including the two-copy averages at N = 30386."""
import os

import numpy as np
import pytest

import pyoracle as po
import tfm_amd
from gpu_common import step
from helpers import radius_for, walk

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))
CHR_LIM = [0, 2284, 4599, 6687, 9338, 12508, 15193, 17477, 19792, 21880, 24531, 27701, 30386]


def sim_with(N, R_n, r, flags, **kw):
    p = {"number_of_particles": N, "nucleus_radius": repr(float(R_n)), "number_of_lbs": 0, "seed": 1}
    p.update(kw)
    sim = tfm_amd.Simulation(p)
    sim.flags = flags
    sim.positions = np.ascontiguousarray(r, np.float32)
    return sim


@pytest.mark.parametrize("N,n_b", [(1024, 64), (16384, 64), (4096, 7)])
def test_observables_match_oracle(N, n_b):
    step(f"observables N={N} n_b={n_b}")
    R_n = radius_for(N, 0.2)
    r = walk(N, R_n, seed=N + n_b)
    flags = (np.random.default_rng(N).random(N) < 0.4).astype(np.uint8)
    sim = sim_with(N, R_n, r, flags)
    r32 = sim.positions.astype(np.float64)
    sc, rcd = sim.observables(n_b)
    R_nf, R_of = float(np.float32(R_n)), float(sim.info.R_o)
    nod = float(np.float32(np.sqrt(R_nf * R_nf - R_of * R_of)))
    want, want_rcd = po.observables(r32, flags, R_nf, nod=nod, n_b=n_b)
    # FP64 sums in another order: relative 1e-9 (rg2 by <r^2> - <r>^2 loses
    # a few digits more to cancellation than the oracle's two-pass form)
    assert np.allclose(sc, want, rtol=1e-9, atol=1e-9), (sc, want)
    assert np.allclose(rcd, want_rcd, rtol=1e-9, atol=1e-10)
    # the radial density integrates to the bead volume
    shell = 4 / 3 * np.pi * float(np.float32(R_n)) ** 3 / n_b
    vb = 4 / 3 * np.pi * (float(np.float32(1.154701)) / 2) ** 3
    assert rcd[2].sum() * shell == pytest.approx(N * vb, rel=1e-9)
    sim.close()


def test_distance_contact_bit_exact():
    step("d(s), P(s) N=2048")
    N = 2048
    R_n = radius_for(N, 0.2)
    sim = sim_with(N, R_n, walk(N, R_n, seed=3, chain_off=[0, 700, N]), np.zeros(N, np.uint8),
                   chain_lengths="700,1348")
    sd, cp = sim.distance_contact(0)
    wsd, wcp = po.sd_cp(sim.positions, 0)
    assert sd.shape == (1024,)
    assert np.array_equal(sd, wsd) and np.array_equal(cp, wcp)
    with pytest.raises(tfm_amd.CcpError, match="no such chromosome"):
        sim.distance_contact(1)
    sim.close()


def test_distance_contact_two_copies():
    step("d(s), P(s) N=30386")
    N = 30386
    R_n = radius_for(N, 0.2)
    sim = tfm_amd.Simulation({"nucleus_radius": repr(float(R_n)), "sequence_file": os.path.join(HERE, "golden",
                              "sequence.txt"), "seed": 4, "number_of_lbs": 0})
    sim.positions = walk(N, R_n, seed=21, chain_off=CHR_LIM).astype(np.float32)
    for c in range(6):
        sd, cp = sim.distance_contact(c)
        wsd, wcp = po.sd_cp(sim.positions, c)
        assert sd.shape == ((CHR_LIM[c + 1] - CHR_LIM[c]) // 2,)
        assert np.array_equal(sd, wsd) and np.array_equal(cp, wcp), c
        assert cp[0] == 1000.0
    sim.close()


def test_frame_contact_map_bit_exact():
    step("ccp frame contact map N=1024")
    N = 1024
    R_n = radius_for(N, 0.3)
    sim = sim_with(N, R_n, walk(N, R_n, seed=8), np.zeros(N, np.uint8))
    r32 = sim.positions
    got = sim.frame_contact_map()
    want = po.ccp_contact_map(r32)
    assert got.shape == want.shape == (256 * 257 // 2,)
    assert np.array_equal(got, want)
    diag = got[np.cumsum(np.arange(1, 257)) - 1]  # a pixel of a bead block with itself
    assert (diag >= 10 * 1000.0 / 16).all()  # 4 self pairs and 6 bonded pairs, both orders
    sim.close()


def test_frame_contact_map_two_copies():
    step("ccp frame contact map N=30386")
    seq = os.path.join(HERE, "golden", "sequence.txt")
    N = 30386
    R_n = radius_for(N, 0.2)
    sim = tfm_amd.Simulation({"nucleus_radius": repr(float(R_n)), "sequence_file": seq, "seed": 4,
                              "number_of_lbs": 0})
    sim.positions = walk(N, R_n, seed=12, chain_off=CHR_LIM).astype(np.float32)
    got = sim.frame_contact_map()
    want = po.ccp_contact_map(sim.positions)
    cms = (N // 2) // 4
    assert got.shape == (cms * (cms + 1) // 2,)
    assert np.array_equal(got, want)
    sim.close()


@pytest.mark.parametrize("N", [8, 64, 65, 66, 127, 258, 1089, 4223])
def test_distance_contact_tile_edges(N):
    # separations and starting beads at the edges of tiles of 32 x 64:
    # one separation, a tile and one more or less, many ragged tiles
    step(f"d(s), P(s) N={N}")
    R_n = radius_for(N, 0.2)
    sim = sim_with(N, R_n, walk(N, R_n, seed=N), np.zeros(N, np.uint8))
    sd, cp = sim.distance_contact(0)
    wsd, wcp = po.sd_cp(sim.positions, 0)
    assert np.array_equal(sd, wsd) and np.array_equal(cp, wcp)
    sim.close()


@pytest.mark.parametrize("N", [8, 60, 68, 1027, 1028, 4164])
def test_frame_contact_map_tile_edges(N):
    # map sides at the edges of the kernel's blocks (256 columns x 16 rows),
    # with beads past the last whole pixel
    step(f"frame contact map N={N}")
    R_n = radius_for(N, 0.3)
    sim = sim_with(N, R_n, walk(N, R_n, seed=N + 1), np.zeros(N, np.uint8))
    assert np.array_equal(sim.frame_contact_map(), po.ccp_contact_map(sim.positions))
    sim.close()


def test_frame_contact_map_rounded_rows():
    # rows long enough that ccp's FP32 root of the packed index leaves the
    # row: every pixel of some rows against ccp's index arithmetic in numpy
    N = 57400
    step(f"frame contact map N={N}")
    R_n = radius_for(N, 0.2)
    sim = sim_with(N, R_n, walk(N, R_n, seed=5), np.zeros(N, np.uint8))
    r = sim.positions
    got = sim.frame_contact_map()
    cms = N // 4
    rows = np.array([cms - 1, cms - 2, cms - 700])
    moved = 0
    for row in rows:
        ia = row * (row + 1) // 2 + np.arange(row + 1)
        ix = np.minimum((np.sqrt((2.0 * ia + 0.25).astype(np.float32)).astype(np.float64) - 0.5).astype(np.int64),
                        cms - 1)
        iy = np.clip((ia - ix * (ix + 1.0) / 2.0).astype(np.int64), 0, cms - 1)
        moved += int((ix != row).sum())
        n = np.zeros(len(ia), np.int64)
        for p in range(4):
            for q in range(4):
                d = r[4 * ix + p] - r[4 * iy + q]
                n += ((d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1]) + d[:, 2] * d[:, 2]) < np.float32(4.0)
        assert np.array_equal(got[ia], (1000 * n / 16).astype(np.float32)), row
    assert moved > 0
    sim.close()


@pytest.mark.parametrize("N", [33, 34, 113, 114, 128, 129, 226, 241])
def test_distance_contact_ragged_tiles(N):
    # a last separation and a last starting bead on either side of the edges
    # of tiles of 8 and 16 separations x 112 beads
    step(f"d(s), P(s) N={N}")
    R_n = radius_for(N, 0.2)
    sim = sim_with(N, R_n, walk(N, R_n, seed=N), np.zeros(N, np.uint8))
    sd, cp = sim.distance_contact(0)
    wsd, wcp = po.sd_cp(sim.positions, 0)
    assert np.array_equal(sd, wsd) and np.array_equal(cp, wcp)
    sim.close()


@pytest.mark.parametrize("N,scale,pixels", [(2048, 1.0, "whole"), (4092, 1.0, "whole"), (4096, 1.0, "list"),
                                            (8190, 1.0, "list"), (8190, 0.45, "long list"), (8190, 0.05, "whole")])
def test_frame_contact_map_lists(N, scale, pixels):
    # nearly empty maps, which reach the host as a list of nonzero pixels (one
    # copy up to 32768 of them, then a second), and small or dense ones (more
    # than an eighth), which are copied whole; into an array of other values
    step(f"frame contact map N={N} scale={scale}")
    R_n = radius_for(N, 0.3)
    sim = sim_with(N, R_n, walk(N, R_n, seed=5) * np.float32(scale), np.zeros(N, np.uint8))
    want = po.ccp_contact_map(sim.positions)
    n, lcm = int((want != 0).sum()), want.size
    listed = lcm >= 1 << 19 and n <= lcm // 8
    assert pixels == ("whole" if not listed else "list" if n <= 32768 else "long list")
    got = np.full(lcm, np.nan, np.float32)
    lib, ptr = tfm_amd.ccp.lib(), tfm_amd.ccp._ptr
    assert lib.ccp_frame_contact_map(sim.h, ptr(got, tfm_amd.ccp.ctypes.c_float), lcm) == 0
    assert np.array_equal(got, want)
    sim.close()


@pytest.mark.parametrize("N,scale", [(140000, 1.0), (140000, 0.01), (340000, 1.0), (340002, 1.0)])
def test_distance_contact_long_chain(N, scale):
    # more contacts at a separation than 2^27 / 1000: ccp's FP32 sum of 1000 per
    # contact rounds at each addition from there on (bonded neighbours, and
    # every separation of the shrunk chain), against sums in order in numpy; and
    # both sides of 170000 separations, above which a lane takes each
    step(f"d(s), P(s) N={N} scale={scale}")
    R_n = radius_for(N, 0.2)
    sim = sim_with(N, R_n, walk(N, R_n, seed=6) * np.float32(scale), np.zeros(N, np.uint8))
    r = sim.positions
    sd, cp = sim.distance_contact(0)
    assert len(sd) == N // 2
    over = 0
    for s in (1, 2, 3, 8, 9, 112, 5000, N // 2 - 1, N // 2):
        d = r[s:] - r[:-s]
        d = np.sqrt((d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1]) + d[:, 2] * d[:, 2])
        a = np.add.accumulate(d, dtype=np.float32)[-1] / np.float32(N - s)
        hit = np.where(d < np.float32(2.0), np.float32(1000.0), np.float32(0.0))
        c = np.add.accumulate(hit, dtype=np.float32)[-1] / np.float32(N - s)
        over += int((d < 2.0).sum() > 134217)
        assert sd[s - 1] == a and cp[s - 1] == c, s
    assert over >= (1 if scale == 1.0 else 6)
    sim.close()


@pytest.mark.parametrize("N,scale", [(1000, 0.3), (4095, 0.3), (4096, 0.3), (4100, 1.0), (4124, 1.0), (4128, 0.3),
                                     (4132, 1.0), (6000, 0.1)])
def test_frame_contact_map_rows_of_a_block(N, scale):
    # one row a block below 1024 rows and eight from there on, whole and ragged
    # last blocks, with few and with many pixels in contact
    step(f"frame contact map N={N} scale={scale}")
    R_n = radius_for(N, 0.3)
    sim = sim_with(N, R_n, walk(N, R_n, seed=N) * np.float32(scale), np.zeros(N, np.uint8))
    assert np.array_equal(sim.frame_contact_map(), po.ccp_contact_map(sim.positions))
    sim.close()


@pytest.mark.parametrize("N,n_b", [(700, 1024), (700, 1025), (300, 4096), (5, 2500)])
def test_observables_of_many_bins(N, n_b):
    # up to 1024 bins the workgroup holds the shells' radii in a table, above
    # each is computed where it is used; the tolerances above
    step(f"observables N={N} n_b={n_b}")
    R_n = max(radius_for(N, 0.2), 4.0)
    r = walk(N, R_n, seed=N + n_b)
    flags = (np.random.default_rng(N).random(N) < 0.4).astype(np.uint8)
    sim = sim_with(N, R_n, r, flags)
    sc, rcd = sim.observables(n_b)
    R_nf, R_of = float(np.float32(R_n)), float(sim.info.R_o)
    nod = float(np.float32(np.sqrt(R_nf * R_nf - R_of * R_of)))
    want, want_rcd = po.observables(sim.positions.astype(np.float64), flags, R_nf, nod=nod, n_b=n_b)
    assert np.allclose(sc, want, rtol=1e-9, atol=1e-9), (sc, want)
    assert np.allclose(rcd, want_rcd, rtol=1e-9, atol=1e-10)
    sim.close()
