"""The stage kernels' body for blocks without cut or solid cells, against the oracle, and the per-case
extrema of more blocks than a workgroup has threads."""
import numpy as np
import pytest

import ffvhc
from helpers import G, N, OracleGrid, geometry
from test_gpu_step import BC, ctx, run_case, trees  # noqa: F401 (ctx is a fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cut_blocks", [0, 1])
@pytest.mark.parametrize("name", ["flat", "two_level"])
@pytest.mark.parametrize("implicit", [None, (0.5, 1.0, 1e-30, 8)])
def test_whole_blocks_match_oracle(ctx, name, cut_blocks, implicit):  # noqa: F811
    """Bit for bit (explicit U; BiCGSTAB of the implicit one to rounding) with no cut block and with one
    among whole ones."""
    tree = trees()[name]
    og = OracleGrid(tree)
    geo = geometry(og, np.random.default_rng(11))
    c, cid, pid = (x.copy() for x in geo)
    for f in range(6):
        c[f][cut_blocks:] = 1.0
        cid[f][cut_blocks:] = 0
    pid[cut_blocks:] = 1
    run_case(ctx, name, solver=0, omega=1.2, count_max=20, eps=1e-30, tol=0.0 if implicit is None else 1e-9, nsteps=1,
             implicit=implicit, tree=tree, geo=(c, cid, pid))


@pytest.mark.parametrize("where", [0, 255, 256, -1])
def test_stats_of_many_blocks(where):
    """Extrema that lie in the first, the last of the first round, the next and the last block."""
    tree = ffvhc.Tree(root=(8, 6, 6), root_length=1.0)
    assert tree.nblk > 256
    ctx = ffvhc.Context(max_blocks=tree.nblk)
    try:
        cid = ctx.add_case(tree, ffvhc.case_params(bc=BC))
        f = ctx.field(8)
        x = np.random.default_rng(3).uniform(0.5, 1.0, (tree.nblk, N, N, N))
        x[where, 3, 5, 7], x[where, 15, 0, 15] = 2.0, -3.0
        x[where, 0, 0, 0] = 1e-9
        ctx.upload(f, cid, np.pad(x, ((0, 0),) + ((G, G),) * 3))
        got = ctx.stats(f, ncases=1)[0]
        assert list(got[1:]) == [2.0, -3.0, 3.0, 1e-9]
    finally:
        ctx.close()


@pytest.mark.parametrize("ids", [[2, 0], [0, 1, 3], [3, 2, 1, 0]])
def test_parameters_of_selected_cases(ids):
    """Each selected case steps with its own dt, whatever runs of ids the selection makes."""
    tree = ffvhc.Tree(root=(2, 1, 1), root_length=1.0)
    ctx = ffvhc.Context(max_blocks=4 * tree.nblk)
    try:
        F = ctx.step_fields()
        rng = np.random.default_rng(8)
        start = {f: rng.standard_normal((tree.nblk,) + (N + 2 * G,) * 3) for f in (F.ux, F.uy, F.uz)}
        cids = [ctx.add_case(tree, ffvhc.case_params(mu=0.01, dt=0.001 * (1 + q), bc=BC)) for q in range(4)]

        def go(sel):
            for q in sel:
                for f in (F.p, F.lapp, *F.v, *F.uc, *F.ucp, *F.ud, *F.udp):
                    ctx.upload(f, cids[q], np.zeros_like(start[F.ux]))
                for f, x in start.items():
                    ctx.upload(f, cids[q], x)
                ctx.set_step(cids[q], 0, 0)
            ctx.select([cids[q] for q in sel])
            _, _, rc = ctx.step(F, solver=0, omega=1.2, count_max=3, eps=0.0, ncases=len(sel))
            assert rc == 0
            return {q: ctx.download(F.ux, cids[q]) for q in sel}

        together = go(ids)
        for q in ids:
            assert np.array_equal(together[q], go([q])[q])
        assert len({together[q].tobytes() for q in ids}) == len(ids)
    finally:
        ctx.close()


def test_results_of_many_cases():
    """More cases than the page-locked buffers hold at first: parameters, statistics and solves of each."""
    tree = ffvhc.Tree(root=(1, 1, 1), root_length=1.0)
    ctx = ffvhc.Context(max_blocks=150)
    try:
        f = ctx.field(8)
        cids = []
        for q in range(150):
            cids.append(ctx.add_case(tree, ffvhc.case_params(dt=0.001 * (1 + q), bc=BC)))
            ctx.upload(f, cids[-1], np.full((1,) + (N + 2 * G,) * 3, 1.0 + q))
            if q in (63, 64, 149):
                ctx.select(cids)
                assert [s[1] for s in ctx.stats(f, ncases=q + 1)] == [1.0 + c for c in range(q + 1)]
                cfl, _ = ctx.cfl(f, ncases=q + 1)
                want = [(1.0 + c) * 0.001 * (1 + c) / 1.0 for c in range(q + 1)]
                assert np.allclose(cfl, want, rtol=1e-14, atol=0.0)
    finally:
        ctx.close()
