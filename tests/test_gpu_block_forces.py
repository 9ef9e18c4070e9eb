"""The block-per-64-particles force kernel at the sizes where it changes what
it does, bit for bit against the CPU oracle (the sums have one defined order,
so no tolerance): a pair list longer than its LDS slots, runs of more than 64
candidates (taken 64 at a time), runs too long to stage, the smallest periodic
box, a last block with one particle, whole cells and x slabs, and walls."""
import sys

import numpy as np
import pytest

import oracle as O
from oracle import rbc as R
from oracle import wall as W

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover - CPU container
    pytest.skip("no GPU", allow_module_level=True)

from ctc_amd import udx as U  # noqa: E402

DT = 1e-4


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def ctx():
    return U.Context()


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


def particles(L, n, seed, clump=0.0):
    """n uniform particles, a share of them in one corner cell and its
    neighbours across the periodic boundary"""
    rng = np.random.default_rng(seed)
    pp = np.zeros((n, 6), np.float32)
    pp[:, :3] = rng.uniform(-0.5, 0.5, (n, 3)) * np.array(L)
    k = int(clump * n)
    half = np.array(L) / 2
    pp[:k, :3] = (rng.uniform(-0.9, 0.9, (k, 3)) + 2 * half) % (2 * half) - half
    pp[:, :3] = np.clip(pp[:, :3], -half, np.nextafter(half.astype(np.float32), np.float32(0)))
    pp[:, 3:] = rng.normal(0, 0.5, (n, 3))
    return pp


# box, particles, share of them around the corner
CASES = [((3, 3, 3), 81, 0.0),          # every pair wraps or nearly so
         ((9, 8, 7), 65 * 3, 0.0),      # last block: 3 of 64
         ((4, 5, 6), 1, 0.0),
         ((8, 8, 8), 8 * 8 * 8 * 20 + 1, 0.0),    # 64 x 84 pairs a block: two windows; unions above 128
         ((5, 4, 6), 5 * 4 * 6 * 70, 0.0),        # 210 candidates a run
         ((12, 11, 13), 12 * 11 * 13 * 2, 0.3)]   # sparse box, one dense corner across the boundary


@pytest.mark.parametrize("L,n,clump", CASES)
@pytest.mark.parametrize("spow", [0.25, 1.0])
def test_step_bit_exact(ctx, L, n, clump, spow):
    say("block forces", L, n, clump, spow)
    pp = particles(L, n, 3, clump)
    par = (25.0, 4.5, O.dpd_sigma(0.5, 4.5, 1e-3), spow)
    seeds = O.seeds_table(2)
    flu = U.Flu(ctx, L, n, U.PairDpd(*par), DT)
    d = torch.as_tensor(pp).cuda()
    flu.set_pp(d)
    flu.run(2, seeds)
    out = torch.zeros_like(d)
    flu.get_pp(out)
    got, npair = host(out), flu.pairs()
    flu.close()
    ref, total = pp, 0
    for k in range(2):
        ref, p = O.flu_step(L, ref, par, seeds[k], DT, nthreads=8)
        total += p
    assert npair == total
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("L,rho", [((11, 12, 12), 24), ((12, 12, 12), 24), ((9, 8, 9), 63), ((9, 8, 9), 64),
                                   ((23, 20, 20), 14), ((24, 20, 20), 18), ((60, 41, 40), 1)])
@pytest.mark.parametrize("slabs", [True, False])
def test_line_bit_exact(ctx, L, rho, slabs):
    """boxes on both sides of the line between the block kernel and the
    lane-per-particle kernel, which falls with the candidates of a run in dense
    boxes and with their lack in sparse ones"""
    n = rho * L[0] * L[1] * L[2]
    say("line", L, rho, n, slabs)
    pp, seeds = particles(L, n, 5), O.seeds_table(1)
    par = (2.5, 4.5, O.dpd_sigma(0.05, 4.5, 5e-4), 0.25)
    if slabs:
        flu = U.Flu(ctx, L, n, U.PairDpd(*par), DT)
        d = torch.as_tensor(pp).cuda()
        flu.set_pp(d)
        flu.run(1, seeds)
        flu.get_pp(d)
        got, npair = host(d), flu.pairs()
        flu.close()
        want, total = O.flu_step(L, pp, par, seeds[0], DT, nthreads=8)
    else:
        starts, counts, srt, _ = O.clist_build(L, pp)
        want, total = O.dpd_forces(L, srt, starts, counts, par, seeds[0], nthreads=8)
        f = U.FluForces(ctx, L, n)
        sd, ff = torch.as_tensor(starts).cuda(), torch.zeros((n, 3), device="cuda")
        f.prepare(torch.as_tensor(srt).cuda())
        f.apply(U.PairDpd(*par), U._ptr(sd), ff, seeds=seeds[0])
        got, npair, total = host(ff), f.pairs(), total // 2
        f.close()
    assert npair == total
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("L,n,clump", CASES[1:])
@pytest.mark.parametrize("periodic", [True, False])
def test_whole_cells_bit_exact(ctx, L, n, clump, periodic):
    """the module binding: no slab starts, forces added to AoS; periodic boxes
    also with the lane-per-particle kernels (split halo forced)"""
    say("block forces, whole cells", L, n, clump, periodic)
    starts, counts, srt, _ = O.clist_build(L, particles(L, n, 4, clump))
    par = (25.0, 4.5, O.dpd_sigma(0.5, 4.5, 1e-3), 0.25)
    seeds = O.seeds_table(1)[0]
    f0 = np.random.default_rng(5).normal(0, 1, (n, 3)).astype(np.float32)
    want, total = O.dpd_forces(L, srt, starts, counts, par, seeds, periodic=periodic, nthreads=8, ff=f0)
    f = U.FluForces(ctx, L, n)
    sd, pd = torch.as_tensor(starts).cuda(), torch.as_tensor(srt).cuda()
    try:
        for edges in (1 << 20, 0) if periodic else (1 << 20,):
            U.set_split_edges(edges)
            f.prepare(pd)
            ff = torch.as_tensor(f0).cuda()
            f.pairs(reset=True)
            f.apply(U.PairDpd(*par), U._ptr(sd), ff, periodic=periodic, seeds=seeds)
            assert f.pairs() == total // 2
            assert np.array_equal(host(ff).view(np.uint32), want.view(np.uint32))
    finally:
        U.set_split_edges(1 << 20)
        f.close()


@pytest.mark.parametrize("rho", [3, 45])
def test_walls_bit_exact(ctx, rho):
    """shearing walls; at density 45 a wall run holds 135 candidates"""
    L, h = (7, 6, 16), 4.0
    say("block forces, walls", rho)
    ext, N = np.array(L, np.float32), (48, 48, 48)
    D = W.plane_channel_sdf(L, 48, h)
    q, ref = U.Sdf(ctx, L, ext=ext, N=N, D=D), W.Sdf(L, ext, N, D.ravel())
    pp = particles(L, rho * 7 * 6 * 16, 6)
    d = torch.as_tensor(pp).cuda()
    w = U.Wall(ctx, q, d)
    n = w.n_solvent
    cur = host(d)[:n].copy()
    _, frozen = ref.freeze(pp)
    wst, _, wpp, _ = O.clist_build(W.margin_box(L), W.wall_images(L, frozen), sub=1)
    par = (25.0, 4.5, O.dpd_sigma(0.5, 4.5, 1e-3), 0.25)
    seeds = np.concatenate([O.seeds_table(2), O.kiss_fill(42, 42, 42, 42, 2)[:, None]], axis=1)
    flu = U.Flu(ctx, L, n, U.PairDpd(*par), DT, 1.0, (0.1, 0.0, 0.0))
    flu.set_pp(d[:n].contiguous())
    flu.set_wall(w)
    flu.run(2, seeds)
    out = torch.zeros((n, 6), device="cuda")
    flu.get_pp(out)
    got, gw = host(out), flu.wall_pairs()
    flu.close()
    tw = 0
    for k in range(2):
        cur, _, nw = W.flu_wall_step(L, cur, par, seeds[k], DT, ref, wpp, wst, accel=(0.1, 0.0, 0.0), nthreads=8)
        tw += nw
    assert gw == tw and tw > 0
    assert np.array_equal(got.view(np.uint32), cur.view(np.uint32))
    w.close()
    q.close()


@pytest.mark.parametrize("rho,nv", [(60, 40), (60, 1), (12, 300), (2, 15)])
def test_vertex_side_bit_exact(ctx, rho, nv):
    """solvent-vertex pairs at densities where a vertex's rows hold 180
    candidates and a wave's pairs fill its list several times over, last waves
    with one vertex, vertices outside the box on every side"""
    L = (6, 4, 8)
    say("vertex side", rho, nv)
    starts, _, srt, _ = O.clist_build(L, particles(L, rho * 6 * 4 * 8, 8))
    rng = np.random.default_rng(9)
    opp = np.zeros((nv, 6), np.float32)
    opp[:, :3] = rng.uniform(-0.65, 0.65, (nv, 3)) * np.array(L)
    opp[:, 3:] = rng.normal(0, 0.1, (nv, 3))
    par = (2.6666667, 8.0, O.dpd_sigma(0.0444, 8.0, 5e-4), 0.25)
    seeds = np.array([0.31, 0.77], np.float32)
    fo0, fs0 = np.ones((nv, 3), np.float32), np.zeros((len(srt), 3), np.float32)
    fo, fs, n = R.fsi_forces(L, srt, starts, opp, par, seeds, fo0, fs0)
    f = U.Fsi(ctx, L, nv, exact=True)
    sd, fd, st = torch.as_tensor(srt).cuda(), torch.as_tensor(fs0).cuda(), torch.as_tensor(starts).cuda()
    f.bind_solvent(sd, fd, U._ptr(st))
    od = torch.as_tensor(fo0).cuda()
    f.apply(U.PairDpd(*par), torch.as_tensor(opp).cuda(), od, seeds=seeds)
    assert f.pairs() == n and n > 0
    assert np.array_equal(host(od).view(np.uint32), fo.view(np.uint32))
    assert np.array_equal(host(fd).view(np.uint32), fs.view(np.uint32))
    f.close()


@pytest.mark.parametrize("first", [(1 << 27) - 300, (1 << 28) - 300])
def test_vertex_side_large_indices(ctx, first):
    """solvent indices on both sides of 2^27 and of 2^28: the particles before
    the first cell are in no cell (their positions, the box centre, are out of
    every vertex's reach)"""
    L = (8, 8, 8)
    say("vertex side, first solvent particle", first)
    starts, _, srt, _ = O.clist_build(L, particles(L, 5000, 8))
    starts = (starts + first).astype(np.int32)
    rng = np.random.default_rng(3)
    opp = np.zeros((40, 6), np.float32)
    opp[:, :3] = rng.uniform(2.1, 5, (40, 3)) * rng.choice([-1, 1], (40, 3))
    par = (2.6666667, 8.0, O.dpd_sigma(0.0444, 8.0, 5e-4), 0.25)
    seeds = np.array([0.31, 0.77], np.float32)
    n = first + len(srt)
    pp = np.zeros((n, 6), np.float32)   # pages that are never touched take no memory
    pp[first:] = srt
    fo, fs, npair = R.fsi_forces(L, pp, starts, opp, par, seeds)
    del pp
    pd = torch.zeros((n, 6), device="cuda")
    pd[first:] = torch.as_tensor(srt).cuda()
    fd, st, od = torch.zeros((n, 3), device="cuda"), torch.as_tensor(starts).cuda(), torch.zeros((40, 3), device="cuda")
    f = U.Fsi(ctx, L, 40)
    f.bind_solvent(pd, fd, U._ptr(st))
    f.apply(U.PairDpd(*par), torch.as_tensor(opp).cuda(), od, seeds=seeds)
    assert f.pairs() == npair and npair > 0
    assert np.array_equal(host(od).view(np.uint32), fo.view(np.uint32))
    assert np.array_equal(host(fd[first:]).view(np.uint32), fs[first:].view(np.uint32))
    assert not bool(fd[:first].any())
    f.close()


@pytest.mark.parametrize("L,n", [((2, 3, 4), 257), ((6, 4, 8), 64), ((6, 4, 8), 1500), ((1, 5, 2), 65), ((16, 16, 16), 1)])
def test_contact_bit_exact(ctx, L, n):
    """membrane contact: rows of cells with none, one and many points (four are
    loaded at a time), boxes thinner than a block of cells, vertices on the
    faces and outside the box on every side, last waves with one vertex"""
    say("contact", L, n)
    rng = np.random.default_rng(n)
    pp = np.zeros((n, 6), np.float32)
    pp[:, :3] = rng.uniform(-0.7, 0.7, (n, 3)) * np.array(L)
    for c in range(3):
        pp[c::11, c] = L[c] // 2
        pp[c + 3::11, c] = -(L[c] // 2)
    pp[:, 3:] = rng.normal(0, 0.3, (n, 3))
    if n > 9:
        pp[n - 1, :3] = pp[0, :3]
    par, sb, sh = (20.0, 8.0, 3.0, 0.25, 0.3, 1.0), np.float32(0.123), np.float32(0.456)
    ff = rng.normal(0, 1, (n, 3)).astype(np.float32)
    want, npair = R.cnt_forces(L, pp, par, sb, sh, ff=ff.copy())
    c = U.Cnt(ctx, L, n)
    fd = torch.as_tensor(ff).cuda()
    c.apply(U.PairDpdLj(*par), torch.as_tensor(pp).cuda(), fd, seeds=(sb, sh))
    assert c.pairs() == npair and (npair > 0 or n == 1)
    assert np.array_equal(host(fd).view(np.uint32), want.view(np.uint32))
    c.close()


@pytest.mark.parametrize("nan", [0x7FC00000, 0xFFC00000])
@pytest.mark.parametrize("c", [0, 1, 2])
def test_not_a_number_hits_nothing(ctx, nan, c):
    """a particle whose position is not a number, of either sign, acts on no
    other one: their forces are those with the particle far away"""
    L, rho, k = (8, 6, 8), 8, 1500
    say("not a number", hex(nan), c)
    starts, _, srt, _ = O.clist_build(L, particles(L, rho * 8 * 6 * 8, 4))
    sd, out = torch.as_tensor(starts).cuda(), []
    for bits in (np.float32(1e6).view(np.uint32), np.uint32(nan)):
        pp = srt.copy()
        pp.view(np.uint32)[k, c] = bits
        f = U.FluForces(ctx, L, len(pp))
        f.prepare(torch.as_tensor(pp).cuda())
        ff = torch.zeros((len(pp), 3), device="cuda")
        f.apply(U.PairDpd(25.0, 4.5, O.dpd_sigma(0.5, 4.5, 1e-3), 0.25), U._ptr(sd), ff,
                seeds=O.seeds_table(1)[0])
        out.append((np.delete(host(ff), k, 0), f.pairs()))
        f.close()
    assert np.isfinite(out[0][0]).all() and out[0][1] > 0
    assert out[0][1] == out[1][1]
    assert np.array_equal(out[0][0].view(np.uint32), out[1][0].view(np.uint32))


@pytest.mark.parametrize("L,split", [((8, 6, 8), False), ((26, 26, 26), False), ((26, 26, 26), True)])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_no_position_no_force(ctx, L, split, bad):
    """a particle whose position is not finite has no pairs: nothing is added
    to its own force (the block kernel, the lane-per-particle kernel and its
    split passes), and its stress stays"""
    rho, k = 8, 1500
    n = rho * L[0] * L[1] * L[2]
    say("no position", L, split, bad)
    starts, _, srt, _ = O.clist_build(L, particles(L, n, 4))
    srt[k, 1] = bad
    par, seeds = U.PairDpd(25.0, 4.5, O.dpd_sigma(0.5, 4.5, 1e-3), 0.25), O.seeds_table(1)[0]
    f = U.FluForces(ctx, L, n)
    pd, sd = torch.as_tensor(srt).cuda(), torch.as_tensor(starts).cuda()
    f.prepare(pd)
    try:
        if split:
            U.set_split_edges(0.0)
        ff = torch.ones((n, 3), device="cuda")
        f.apply(par, U._ptr(sd), ff, seeds=seeds)
    finally:
        U.set_split_edges(1048576.0)
    assert host(ff[k]).tolist() == [1.0, 1.0, 1.0]
    assert bool(torch.isfinite(ff).all())
    ff, ss = torch.ones((n, 3), device="cuda"), torch.ones((n, 6), device="cuda")
    f.apply_stress(par, U._ptr(sd), ff, ss, seeds=seeds)
    assert host(ff[k]).tolist() == [1.0] * 3 and host(ss[k]).tolist() == [1.0] * 6
    f.close()


@pytest.mark.parametrize("rho,order", [(3, "cells"), (30, "cells"), (30, "shuffled"), (45, "cells"), (45, "one")])
def test_wall_rows_bit_exact(ctx, rho, order):
    """wall forces by a launch of their own: rows that a wave stages and rows
    too long for it (density 45: 135 candidates a run; particles out of cell
    order), runs of more than 64, one particle"""
    L = (7, 6, 16)
    say("wall rows", rho, order)
    ext, N = np.array(L, np.float32), (48, 48, 48)
    D = W.plane_channel_sdf(L, 48, 4.0)
    q, ref = U.Sdf(ctx, L, ext=ext, N=N, D=D), W.Sdf(L, ext, N, D.ravel())
    pp = particles(L, rho * 7 * 6 * 16, 6)
    d = torch.as_tensor(pp).cuda()
    w = U.Wall(ctx, q, d)
    _, frozen = ref.freeze(pp)
    wst, _, wpp, _ = O.clist_build(W.margin_box(L), W.wall_images(L, frozen), sub=1)
    _, _, srt, _ = O.clist_build(L, host(d)[:w.n_solvent])
    if order == "shuffled":
        srt = srt[np.random.default_rng(1).permutation(len(srt))]
    if order == "one":
        srt = srt[np.argmax(srt[:, 2])][None]
    par = (25.0, 4.5, O.dpd_sigma(0.5, 4.5, 1e-3), 0.25)
    ff = np.ones((len(srt), 3), np.float32)
    want, npair = W.wall_forces(L, srt, ref, wpp, wst, par, np.float32(0.37), ff.copy())
    fd = torch.as_tensor(ff).cuda()
    w.force(U.PairDpd(*par), torch.as_tensor(np.ascontiguousarray(srt)).cuda(), fd, seed=np.float32(0.37))
    assert w.pairs() == npair and npair > 0
    assert np.array_equal(host(fd).view(np.uint32), want.view(np.uint32))
    w.close()
    q.close()
