"""Solves of at most 256 blocks run in one launch whose blocks stay on the chip; with that on (default) and
off (one launch per stage) every solver gives the same bits, counts and residuals."""
import threading

import numpy as np
import pytest

import ffvhc
from helpers import OracleGrid
from test_gpu_class_rows import SOLVE
from test_gpu_core import BC, class_uniform_system

pytestmark = pytest.mark.gpu

BC_PERIODIC = dict(BC)
BC_PERIODIC[ffvhc.BC_P] = [(9, 0.0), (9, 0.0), (1, 0.0), (0, 0.5), (-1, 0.0), (1, 0.25)]
BC_PERIODIC[ffvhc.BC_NULL] = [(9, 0.0), (9, 0.0)] + [(1, 0.0)] * 4

TREES = {
    "one": dict(root=(1, 1, 1)),
    "odd": dict(root=(5, 3, 1)),
    "three_level": dict(root=(2, 2, 2), regions=[dict(kind="ball", a=(0.9, 1.1, 1.05), r=0.2, level=2)]),
    "most": dict(root=(8, 8, 4)),
    "wrapped": dict(root=(2, 1, 3), periodic=(1, 1, 0)),
}


def mixed(method):
    return lambda c, x, A, b, n: c.solve_mixed(method, x, A, b, ffvhc.BC_P, 1.4, n, 1e-12, 0.5)


SOLVERS = {k: v for k, v in SOLVE.items() if k != "fixed_average"}
SOLVERS.update(mixed23=mixed(23), mixed26=mixed(26), mixed28=mixed(28))


def load(ctx, tree, bc, prec, n_other, seed, fields=None):
    """A case with a system of its own; n_other blocks get a cell that differs from its class."""
    params = ffvhc.case_params(bc=bc)
    cid = ctx.add_case(tree, params)
    og = OracleGrid(tree)
    t = [params.bct[ffvhc.BC_P][q] if params.bct[ffvhc.BC_P][q] in (0, 1) else 1 for q in range(6)]
    A, b, _ = class_uniform_system(og, np.random.default_rng(seed), t, [0.0] * 6, n_other)
    dtype = np.float64 if prec == 8 else np.float32
    f = fields or [ctx.field(prec) for _ in range(9)]
    for fld, v in zip(f, A + [b]):
        ctx.upload(fld, cid, v.astype(dtype))
    return cid, f, dtype


def both(ctx, cids, f, dtype, run):
    got = []
    for on in (True, False):
        ctx.set_resident(on)
        ctx.fill(f[8], 0.25)
        ctx.ghost_fill(f[8], ffvhc.BC_P)
        out = run()
        got.append([np.asarray(v).tolist() for v in out] + [ctx.download(f[8], c, dtype=dtype) for c in cids])
    ctx.set_resident(True)
    k = len(out)
    assert got[0][:k] == got[1][:k]
    for a, b in zip(got[0][k:], got[1][k:]):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("name", sorted(TREES))
@pytest.mark.parametrize("how,prec", [(h, 8) for h in sorted(SOLVERS)] + [("rbgs", 4), ("jacobi", 4), ("cg", 4)])
def test_resident_bit_identical(how, prec, name):
    """Cut off after 3 and 20 iterations; blocks with and without cells of their own."""
    tree = ffvhc.Tree(root_length=1.0, **TREES[name])
    ctx = ffvhc.Context(max_blocks=tree.nblk + 3)
    try:
        cid, f, dtype = load(ctx, tree, BC if name != "odd" else BC_PERIODIC, prec, min(tree.nblk, 3), 11)
        for n in (3, 20):
            both(ctx, [cid], f, dtype, lambda: SOLVERS[how](ctx, f[8], f[:7], f[7], n))
    finally:
        ctx.close()


@pytest.mark.parametrize("how", ["bicgstab", "cg", "mixed26", "rbgs"])
def test_resident_cases_of_one_launch(how):
    """Three cases of different sizes in one launch end at different iterations (countMax 4,000, beyond
    one launch's turns for RBGS)."""
    trees = [ffvhc.Tree(root_length=1.0, **TREES[k]) for k in ("odd", "three_level", "one")]
    ctx = ffvhc.Context(max_blocks=sum(t.nblk for t in trees))
    try:
        f = [ctx.field(8) for _ in range(9)]
        cids = [load(ctx, t, BC, 8, 0 if how == "cg" else min(k, t.nblk), 5 + k, f)[0] for k, t in enumerate(trees)]
        run = {"bicgstab": lambda: ctx.bicgstab(f[8], f[:7], f[7], ffvhc.BC_P, 1.0, 1, 4000, 1e-9),
               "cg": lambda: ctx.cg(f[8], f[:7], f[7], ffvhc.BC_P, 1.0, 1, 300, 1e-9),
               "mixed26": lambda: ctx.solve_mixed(26, f[8], f[:7], f[7], ffvhc.BC_P, 1.4, 4000, 1e-11, 0.5),
               "rbgs": lambda: ctx.rbgs(f[8], f[:7], f[7], ffvhc.BC_P, 1.2, 4000, 0.0)}[how]
        both(ctx, cids, f, np.float64, run)
    finally:
        ctx.close()


def test_resident_solves_of_two_threads():
    """Two contexts on two threads, together more blocks than the chip holds at once."""
    tree = ffvhc.Tree(root=(8, 5, 4), root_length=1.0)
    ctxs, out, errors = [ffvhc.Context(max_blocks=tree.nblk) for _ in range(2)], {}, []
    try:
        loaded = [load(c, tree, BC, 8, 3, 21 + k) for k, c in enumerate(ctxs)]

        def work(k, tag):
            try:
                cid, f, _ = loaded[k]
                for q in range(4):
                    ctxs[k].fill(f[8], 0.0)
                    ctxs[k].solve_mixed(26, f[8], f[:7], f[7], ffvhc.BC_P, 1.4, 500, 1e-10, 0.5)
                out[k, tag] = ctxs[k].download(f[8], cid)
            except Exception as e:  # shown below
                errors.append(e)

        for k in range(2):
            work(k, "alone")
        threads = [threading.Thread(target=work, args=(k, "beside")) for k in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not errors
        for k in range(2):
            assert np.array_equal(out[k, "alone"], out[k, "beside"])
    finally:
        for c in ctxs:
            c.close()
