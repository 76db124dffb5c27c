"""Every block shape of the prefill matmul (prefill.hip shape_for) at the sizes
where it can go wrong, against the CPU oracle on some of the tokens: both sides
of each token limit, rows one past a wave's and a block's, an odd number of
256-value chunks between the groups of K, and (32-value kinds) a last chunk of
one 64-value stage.  Gate: tests/test_gpu_prefill.py's.
"""

import numpy as np
import pytest

import oracle
from tests.test_gpu_kernels import assert_matvec_close, dequant_abs
from tests.test_gpu_prefill import K_QUANTS, KINDS, ctx, run  # noqa: F401 (ctx is a fixture)

pytestmark = pytest.mark.gpu

SHAPES = [
    # rows, K-quant cols, 32-value cols, tokens
    (129, 512, 448, 32),      # one token tile, chunks in two groups of K
    (129, 768, 576, 33),      # the small shape, three chunks in two groups
    (257, 1280, 1344, 65),    # its second block of tokens
    (300, 14592, 14400, 897),  # the large shapes: 57 chunks, ragged rows and tokens
]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("rows,k_cols,b_cols,tokens", SHAPES)
def test_prefill_block_shapes(ctx, kind, rows, k_cols, b_cols, tokens):  # noqa: F811
    cols = k_cols if kind in K_QUANTS else b_cols
    blob, x, got = run(ctx, kind, rows, cols, tokens, 700 + kind)
    some = sorted({0, 31, tokens // 2, tokens - 2, tokens - 1})
    x, got = x.reshape(tokens, cols)[some], got.reshape(tokens, rows)[some]
    want = oracle.matvec(kind, blob, rows, cols, np.ascontiguousarray(x), threads=8)
    assert_matvec_close(got.reshape(-1), want, dequant_abs(kind, blob, rows, cols), x.reshape(-1))
