"""The sweep kernel's forms (all blocks from class rows, few or many blocks per cell, all per cell) give
the same bits as the per-cell form, with one launch per stage."""
import numpy as np
import pytest

import ffvhc
from test_gpu_core import BC
from test_gpu_resident import load, mixed

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_other", [0, 1, 2, 3, 30])
@pytest.mark.parametrize("method", [13, 20, 26, 29])
def test_forms_bit_identical(method, n_other):
    """30 blocks: two per cell are at most a twelfth, three are more; 30 cells that differ leave few or no
    blocks uniform."""
    tree = ffvhc.Tree(root=(5, 3, 2), root_length=1.0)
    ctx = ffvhc.Context(max_blocks=tree.nblk)
    try:
        ctx.set_resident(False)
        cid, f, _ = load(ctx, tree, BC, 8, n_other, 17)
        n_irr = ctx.stencil_classes(f[:7])[1]
        assert n_irr == n_other if n_other < 30 else 12 * n_irr > tree.nblk
        got = []
        for on in (True, False):
            ctx.set_classes(on)
            ctx.fill(f[8], 0.25)
            ctx.ghost_fill(f[8], ffvhc.BC_P)
            out = mixed(method)(ctx, f[8], f[:7], f[7], 12)
            got.append([np.asarray(v).tolist() for v in out] + [ctx.download(f[8], cid).tobytes()])
        assert got[0] == got[1]
    finally:
        ctx.close()
