"""A single tile of rows computes only the 16-row blocks that M has: every block
count of the 32-, 64- and 128-row tiles (variants 9, 8, 7), at the edges of a
block, with ragged N, one and several splits, against the same plan variant's
two-tile result: x stacked past the tile's rows goes through the full tile,
whose outputs are formed by the same products in the same order, so the two
are equal bit for bit."""
import numpy as np
import pytest
import torch

from kernels import _native
from kernels.awq_gemm import awq_gemm_forward_ex
from oracle import awq_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant,rows", [(7, 128), (8, 64), (9, 32)])
@pytest.mark.parametrize("k,n", [(1024, 776), (128, 256), (1280, 1032)])
def test_tile_row_blocks(gpu, variant, rows, k, n):
    x, qw, qz, s = O.make_inputs(2 * rows, k, n, seed=variant + n)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)  # noqa: E731
    xt, op = t(x), (t(qw), t(qz), t(s))
    y_ref = O.awq_gemm_oracle(x, qw, qz, s)
    for split in (1, 2, 5):
        try:
            p2 = _native.plan_tile(2 * rows, n, k, variant, split)
        except _native.AwqNativeError:
            continue
        full = awq_gemm_forward_ex(xt, *op, plan_obj=p2)
        assert O.max_rel_err(full.cpu().numpy(), y_ref) <= 1e-2
        for m in sorted({1, 15, 16, 17, rows - 17, rows - 16, rows - 15, rows - 1, rows, *range(16, rows + 1, 16)}):
            if not 1 <= m <= rows:
                continue
            print(f"tile rows variant={variant} K={k} N={n} split={split} M={m}", flush=True)
            y = awq_gemm_forward_ex(xt[:m], *op, plan_obj=_native.plan_tile(m, n, k, variant, split))
            assert torch.equal(y, full[:m])
