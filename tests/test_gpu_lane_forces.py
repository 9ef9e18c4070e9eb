"""The lane-per-particle force kernel, bit for bit against the CPU oracle, in
boxes above the line up to which a block takes 64 particles: more than 196608
particles with x slabs, more than 131072 without, about half of that in sparse
boxes, or more than 40960 where a run of three cells holds 48 candidates or
more.  Forces alone (periodic, not
periodic, the halo pass inside and as a launch of its own), the step that
moves the particles (eager and captured) and the step with walls."""
import sys

import numpy as np
import pytest

import oracle as O
from oracle import wall as W

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover - CPU container
    pytest.skip("no GPU", allow_module_level=True)

from ctc_amd import udx as U  # noqa: E402

DT = 5e-4


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def ctx():
    return U.Context()


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


def same(a, b):
    return np.array_equal(a.view(np.uint32), b.view(np.uint32))


def particles(L, n, seed):
    rng = np.random.default_rng(seed)
    half = np.array(L, np.float32) / 2
    pp = np.zeros((n, 6), np.float32)
    pp[:, :3] = rng.uniform(-0.5, 0.5, (n, 3)) * np.array(L)
    pp[:, :3] = np.clip(pp[:, :3], -half, np.nextafter(half, np.float32(0)))
    pp[:, 3:] = rng.normal(0, 0.3, (n, 3))
    return pp


# box, particles, spow
BOXES = [((52, 51, 50), 132600, 0.5),       # density 1
         ((70, 63, 65), 71663, 0.25),       # density 1/4, just above the line of sparse boxes
         ((7, 5, 1301), 136605 + 1, 1.0),   # thin and long, a last block with one particle
         ((3, 40, 139), 133440, 0.25),      # three cells across: every pair wraps along x or nearly so
         ((12, 11, 13), 41184, 0.25),       # density 24: runs staged in several chunks
         ((3, 4, 5), 41013, 0.25)]          # density 683: a queue generation every row


@pytest.mark.parametrize("L,n,spow", BOXES)
@pytest.mark.parametrize("periodic", [True, False])
def test_forces_bit_exact(ctx, L, n, spow, periodic):
    say("lane forces", L, n, spow, periodic)
    starts, counts, srt, _ = O.clist_build(L, particles(L, n, 2))
    par, seeds = (2.5, 4.5, O.dpd_sigma(0.05, 4.5, DT), spow), O.seeds_table(2)[1]
    f0 = np.random.default_rng(1).normal(0, 1, (n, 3)).astype(np.float32)
    want, total = O.dpd_forces(L, srt, starts, counts, par, seeds, periodic=periodic, nthreads=8, ff=f0)
    sd, pd = torch.as_tensor(starts).cuda(), torch.as_tensor(srt).cuda()
    try:
        for mode in (U.MODE_FAST, U.MODE_EXACT):
            f = U.FluForces(ctx, L, n, mode=mode)
            f.prepare(pd)
            for split in ((1e30, 0.0) if periodic else (1e30,)):
                U.set_split_edges(split)
                ff = torch.as_tensor(f0).cuda()
                f.apply(U.PairDpd(*par), U._ptr(sd), ff, periodic=periodic, seeds=seeds)
                assert f.pairs(reset=True) == total // 2
                assert same(host(ff), want), (mode, split)
            f.close()
    finally:
        U.set_split_edges(1048576.0)


@pytest.mark.parametrize("L,n,spow,steps", [((41, 40, 41), 197000, 0.25, 6), ((31, 29, 44), 197780, 1.0, 4),
                                            ((12, 11, 13), 41184, 0.5, 6)])
@pytest.mark.parametrize("graph", [False, True])
def test_steps_bit_exact(ctx, L, n, spow, steps, graph):
    """the gather that moves the particles and counts the next step's cells"""
    say("lane steps", L, n, spow, graph)
    pp, seeds, accel = particles(L, n, 3), O.seeds_table(steps), (0.3, 0.0, -0.1)
    par = (2.5, 4.5, O.dpd_sigma(0.05, 4.5, DT), spow)
    flu = U.Flu(ctx, L, n, U.PairDpd(*par), DT, 1.0, accel)
    flu.graph(graph)
    d = torch.as_tensor(pp).cuda()
    flu.set_pp(d)
    ref, done, total = pp, 0, 0
    for m in (steps - 2, 2):   # a replay after eager work and a synchronisation
        flu.run(m, seeds[done:done + m])
        flu.get_pp(d)
        for k in range(done, done + m):
            ref, p = O.flu_step(L, ref, par, seeds[k], DT, accel=accel, nthreads=8)
            total += p
        done += m
        assert same(host(d), ref)
    assert flu.pairs() == total
    flu.close()


@pytest.mark.parametrize("spow", [0.25, 0.5])
@pytest.mark.parametrize("graph", [False, True])
def test_walls_bit_exact(ctx, spow, graph):
    """sheared walls: the gather adds the wall forces, moves and bounces"""
    L, rho, steps = (12, 12, 18), 25, 4
    say("lane walls", spow, graph)
    ext, N = np.array(L, np.float32), (48, 48, 48)
    D = W.plane_channel_sdf(L, 48, 6.0)
    q, ref = U.Sdf(ctx, L, ext=ext, N=N, D=D), W.Sdf(L, ext, N, D.ravel())
    pp = particles(L, rho * 12 * 12 * 18, 6)
    d = torch.as_tensor(pp).cuda()
    w = U.Wall(ctx, q, d)
    n = w.n_solvent
    assert n > 40960
    cur = host(d)[:n].copy()
    _, frozen = ref.freeze(pp)
    wst, _, wpp, _ = O.clist_build(W.margin_box(L), W.wall_images(L, frozen), sub=1)
    par = (2.5, 4.5, O.dpd_sigma(0.05, 4.5, DT), spow)
    seeds = np.concatenate([O.seeds_table(steps), O.kiss_fill(42, 42, 42, 42, steps)[:, None]], axis=1)
    flu = U.Flu(ctx, L, n, U.PairDpd(*par), DT, 1.0, (0.1, 0.0, 0.0))
    flu.graph(graph)
    flu.set_pp(d[:n].contiguous())
    w.set_vel(U.wall_vel("shear", gdot=0.3, vdir=0, gdir=2))
    flu.set_wall(w)
    flu.run(steps, seeds)
    out = torch.zeros((n, 6), device="cuda")
    flu.get_pp(out)
    got, gp, gw = host(out), flu.pairs(), flu.wall_pairs()
    flu.close()
    tp = tw = 0
    for k in range(steps):
        cur, p, nw = W.flu_wall_step(L, cur, par, seeds[k], DT, ref, wpp, wst, accel=(0.1, 0.0, 0.0), nthreads=8,
                                     wv=W.wvel("shear", gdot=0.3, vdir=0, gdir=2))
        tp += p
        tw += nw
    assert gp == tp and gw == tw and tw > 0
    assert same(got, cur)
    w.close()
    q.close()
