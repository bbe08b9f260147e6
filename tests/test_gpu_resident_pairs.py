"""Solves of 257 to 512 blocks run resident with two workgroups a compute unit: the same bits, counts and
residuals as with one launch per stage."""
import numpy as np
import pytest

import ffvhc
from test_gpu_core import BC
from test_gpu_resident import BC_PERIODIC, SOLVERS, both, load

pytestmark = pytest.mark.gpu

TREES = {
    "least": (dict(root=(257, 1, 1)), BC_PERIODIC, 257),
    "three_level": (dict(root=(6, 5, 4), regions=[dict(kind="ball", a=(2.1, 2.4, 1.9), r=0.6, level=1),
                                                  dict(kind="ball", a=(2.1, 2.4, 1.9), r=0.2, level=2)]), BC, None),
    "most": (dict(root=(8, 8, 8)), BC, 512),
    "beyond": (dict(root=(19, 9, 3)), BC, 513),
}
HOW = [(h, 8) for h in ("bicgstab", "cg", "jacobi", "rbgs", "mixed26")] + [("rbgs", 4), ("jacobi", 4), ("cg", 4)]


@pytest.mark.parametrize("name", sorted(TREES))
@pytest.mark.parametrize("how,prec", HOW)
def test_pairs_bit_identical(how, prec, name):
    """Cut off after 3 and 11 iterations; three blocks have a cell of their own."""
    spec, bc, nblk = TREES[name]
    tree = ffvhc.Tree(root_length=1.0, **spec)
    assert tree.nblk == nblk or (nblk is None and 256 < tree.nblk <= 512)
    ctx = ffvhc.Context(max_blocks=tree.nblk + 1)
    try:
        cid, f, dtype = load(ctx, tree, bc, prec, 3, 31)
        for n in (3, 11):
            both(ctx, [cid], f, dtype, lambda: SOLVERS[how](ctx, f[8], f[:7], f[7], n))
    finally:
        ctx.close()


@pytest.mark.parametrize("how", ["bicgstab", "cg", "jacobi"])
def test_pairs_of_cases(how):
    """Cases of 300 and 100 blocks in one launch, each to its own end; Jacobi beyond one launch's turns."""
    trees = [ffvhc.Tree(root_length=1.0, root=r) for r in ((10, 6, 5), (5, 5, 4))]
    ctx = ffvhc.Context(max_blocks=sum(t.nblk for t in trees))
    try:
        f = [ctx.field(8) for _ in range(9)]
        cids = [load(ctx, t, BC, 8, 0 if how == "cg" else 2, 5 + k, f)[0] for k, t in enumerate(trees)]
        run = {"bicgstab": lambda: ctx.bicgstab(f[8], f[:7], f[7], ffvhc.BC_P, 1.0, 1, 4000, 1e-9),
               "cg": lambda: ctx.cg(f[8], f[:7], f[7], ffvhc.BC_P, 1.0, 1, 300, 1e-9),
               "jacobi": lambda: ctx.jacobi(f[8], f[:7], f[7], ffvhc.BC_P, 0.8, 2500, 0.0)}[how]
        both(ctx, cids, f, np.float64, run)
    finally:
        ctx.close()
