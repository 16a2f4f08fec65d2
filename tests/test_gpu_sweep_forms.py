"""The sweep kernel's forms at the sizes where their rules change, one RHS
evaluation each against the oracle (NaiverStokesData3d::solve,
src/NaiverStokes3d.cpp:37-73).  The bars are those of test_gpu_rhs.py: 1e-11
relative per conserved variable, and for the schemes with cancelling 7-point
indicators three times the oracle's own change under +-1 ulp of its input."""
import numpy as np
import pytest

import nuc3d_amd as G
import oracle as O
from test_gpu_rhs import ILL_CONDITIONED, _ulp_floor

pytestmark = pytest.mark.gpu

CASES = [
    # n, rank grid, scheme, viscous scheme, splitting
    # hccs explicit rows inside the row loop (lines of several blocks, and of two
    # rows a lane); 10 cells is the shortest block
    ((10, 20, 30), (1, 2, 3), G.HCCS, G.CD6, G.AUSM),
    ((30, 10, 20), (3, 1, 2), G.HCCS, G.CD8, G.LF),
    ((12, 66, 33), (1, 3, 3), G.HCCS, G.CD6, G.AUSMP),
    # one WENO7-Z evaluation for both kinds of row
    ((10, 20, 30), (1, 2, 3), G.HCCS77, G.CD6, G.AUSM),
    ((10, 20, 30), (1, 2, 3), G.HCCS78, G.CD8, G.LF),
    # two waves per line (257-512 cells): one cell more than a wave holds, the
    # ends of each row count, tails of the lines per workgroup (2 in x, 4 or 2
    # in y and z), a compact segment of 511 cells
    ((257, 11, 12), (1, 1, 1), G.CRWENO5, G.CD8, G.LF),
    ((11, 320, 13), (1, 1, 1), G.HCCS, G.CD6, G.AUSM),
    ((13, 11, 321), (1, 1, 1), G.WENO5Z, G.CD6, G.AUSM),
    ((384, 12, 10), (2, 1, 1), G.HCCS77, G.CD6, G.LF),
    ((11, 385, 10), (1, 1, 1), G.WENO7JS, G.CD8, G.AUSMP),
    ((10, 511, 11), (1, 1, 1), G.CRWENO5, G.CD6, G.AUSM),
    ((512, 10, 11), (1, 1, 1), G.HCCS, G.CD6, G.LF),
    ((12, 10, 512), (1, 1, 4), G.CRWENO5, G.CD8, G.LF),
    ((1022, 10, 11), (2, 1, 1), G.CRWENO5, G.CD6, G.LF),
    # compact lines of one block (explicit rows ahead of the row loop): the
    # shortest and longest line of each row count, with and without tails
    ((65, 96, 97), (1, 1, 1), G.CRWENO5, G.CD6, G.AUSM),
    ((65, 96, 97), (1, 1, 1), G.HCCS, G.CD8, G.LF),
    ((128, 12, 160), (1, 1, 1), G.CRWENO5, G.CD8, G.LF),
    ((129, 128, 12), (1, 1, 1), G.HCCS, G.CD6, G.AUSMP),
    ((12, 161, 192), (1, 1, 1), G.CRWENO5, G.CD6, G.AUSMP),
    ((192, 12, 193), (1, 1, 1), G.HCCS, G.CD6, G.LF),
    ((193, 256, 12), (1, 1, 1), G.CRWENO5, G.CD8, G.LF),
    ((256, 12, 193), (1, 1, 1), G.HCCS, G.CD8, G.AUSM),
]


def _state(oc, seed):
    """Taylor-Green with a seeded 3-D perturbation: every variable of order one."""
    q = O.init_tgv(oc)
    N = oc.nx * oc.ny * oc.nz
    rng = np.random.default_rng(seed)
    q = q.reshape(5, N)
    q[3] += 0.2 * np.sin(np.linspace(0, 40, N) + rng.random())
    q[0] *= 1.0 + 0.01 * rng.standard_normal(N)
    return q.ravel().copy()


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}-{c[1]}-s{c[2]}-v{c[3]}-r{c[4]}")
def test_rhs_matches_oracle(case):
    n, npr, scheme, vis, rie = case
    print(f"sweep form {case}", flush=True)
    kw = dict(n=n, npr=npr, scheme=scheme, vis=vis, riemann=rie, model=G.NAVIERSTOKES3D)
    gc, oc = G.make_config(**kw), O.make_config(**kw)
    oc.nthreads = 8
    q = _state(oc, 11)
    N = oc.nx * oc.ny * oc.nz
    s = O.Solver(oc)
    s.set_state(q)
    ref, dt_ref = s.rhs()
    with G.Context(gc) as ctx:
        ctx.upload(q)
        got, dt = ctx.rhs()
    ref, got = ref.reshape(5, N), got.reshape(5, N)
    err = np.abs(got - ref).max(axis=1) / np.abs(ref).max(axis=1)
    tol = np.full(5, 1e-11)
    if scheme in ILL_CONDITIONED:
        tol = np.maximum(tol, 3.0 * _ulp_floor(oc, q, 0))
    print("rel err", err, "tol", tol, flush=True)
    assert np.all(err <= tol), (err, tol)
    assert abs(dt - dt_ref) <= 1e-14 * dt_ref


@pytest.mark.parametrize("scheme,precision", [(G.CRWENO5, G.FP64), (G.CRWENO5, G.MIXED), (G.HCCS, G.FP64)])
def test_pack_of_one_block_and_rank_grid(scheme, precision):
    """A pack whose members' lines are one block in some and several in others:
    each member bit for bit as it runs alone."""
    boxes = [((72, 66, 80), (1, 1, 1)), ((96, 70, 68), (1, 2, 1)), ((66, 96, 72), (1, 1, 1))]
    cfgs = [G.make_config(n=n, npr=npr, scheme=scheme, vis=G.CD6, riemann=G.LF, model=G.NAVIERSTOKES3D,
                          precision=precision) for n, npr in boxes]
    qs = [_state(O.make_config(n=n, npr=npr), 20 + k) for k, (n, npr) in enumerate(boxes)]
    alone = []
    for c, q in zip(cfgs, qs):
        with G.Context(c) as ctx:
            ctx.upload(q)
            ctx.step(2)
            alone.append(ctx.download())
    for members in ([0, 1, 2], [0, 2]):
        ctxs = [G.Context(cfgs[k]) for k in members]
        for ctx, k in zip(ctxs, members):
            ctx.upload(qs[k])
        with G.Pack(ctxs) as p:
            p.step_async(2)
            for ctx in ctxs:
                ctx.sync()
            got = [ctx.download() for ctx in ctxs]
        for ctx in ctxs:
            ctx.close()
        for k, g in zip(members, got):
            assert np.array_equal(g, alone[k]), (members, boxes[k])
