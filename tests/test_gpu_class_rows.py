"""The reference's solvers (RBGS, Jacobi, RBGS with fixed average, CG, BiCGSTAB, FP64 and FP32) read
the bands of class-uniform blocks from 27 rows; the solve is bit-identical with the rows on (default)
and off."""
import numpy as np
import pytest

import ffvhc
from helpers import OracleGrid
from test_gpu_core import BC, class_uniform_system, trees

pytestmark = pytest.mark.gpu

SOLVE = {
    "rbgs": lambda c, x, A, b, n: c.rbgs(x, A, b, ffvhc.BC_P, 1.2, n, 0.0, ncases=1),
    "jacobi": lambda c, x, A, b, n: c.jacobi(x, A, b, ffvhc.BC_P, 0.8, n, 0.0, ncases=1),
    "fixed_average": lambda c, x, A, b, n: c.rbgs_fixed_average(x, A, b, ffvhc.BC_P, 1.2, n, 0.0, ncases=1),
    "cg": lambda c, x, A, b, n: c.cg(x, A, b, ffvhc.BC_P, 1.0, 1, n, 0.0, ncases=1),
    "bicgstab": lambda c, x, A, b, n: c.bicgstab(x, A, b, ffvhc.BC_P, 1.0, 1, n, 0.0, ncases=1),
}


@pytest.mark.parametrize("name,n_other", [("flat", 0), ("flat", 5), ("three_level", 3)])
@pytest.mark.parametrize("prec", [8, 4])
@pytest.mark.parametrize("how", sorted(SOLVE))
def test_class_rows_bit_identical(how, prec, name, n_other):
    """2 iterations (below the limit from which the rows are made) and 9, on systems without and with
    blocks that are not class-uniform."""
    tree = trees()[name]
    params = ffvhc.case_params(bc=BC)
    ctx = ffvhc.Context(max_blocks=tree.nblk)
    try:
        cid = ctx.add_case(tree, params)
        og = OracleGrid(tree)
        bct = [params.bct[ffvhc.BC_P][q] for q in range(6)]
        bcv = [params.bcv[ffvhc.BC_P][q] for q in range(6)]
        A, b, _ = class_uniform_system(og, np.random.default_rng(5), bct, bcv, n_other)
        dtype = np.float64 if prec == 8 else np.float32
        fa = [ctx.field(prec) for _ in range(7)]
        fb, fx = ctx.field(prec), ctx.field(prec)
        for f, v in zip(fa + [fb], A + [b]):
            ctx.upload(f, cid, v.astype(dtype))
        for n in (2, 9):
            got = []
            for classes in (True, False):
                ctx.set_classes(classes)
                ctx.fill(fx, 0.25)
                ctx.ghost_fill(fx, ffvhc.BC_P)
                cnt, res, rc = SOLVE[how](ctx, fx, fa, fb, n)
                got.append((cnt[0], res[0], rc, ctx.download(fx, cid, dtype=dtype)))
            assert got[0][:3] == got[1][:3]
            assert np.array_equal(got[0][3], got[1][3])
    finally:
        ctx.close()
