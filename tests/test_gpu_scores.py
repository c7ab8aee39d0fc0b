"""Block scores on the fp32 matrix instructions against the canonical fmaf
chain of the oracle (k ascending from +0), bit for bit: sizes around the 32, 64
and 128-block tiles, both tile sizes, every column chunking, wide exponents,
denormal products, infinities, the invalid-key fill."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.test_gpu_parity import bits_equal, dev, host, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("BH,Nq,Nk,D", [(1, 1, 1, 16), (2, 31, 33, 48), (1, 64, 65, 64), (3, 63, 130, 128),
                                        (1, 129, 127, 96), (1, 2900, 2890, 32), (2, 2049, 2050, 48)], ids=str)
def test_scores_equal_the_canonical_chain(BH, Nq, Nk, D):
    from prism_amd import ops
    say("scores", (BH, Nq, Nk, D))
    rng = np.random.default_rng(Nq + D)
    q, k = (rng.standard_normal((BH, n, D)).astype(np.float32) for n in (Nq, Nk))
    q[:, ::3] *= np.float32(2.0) ** rng.integers(-60, 60, (BH, len(range(0, Nq, 3)), D)).astype(np.float32)
    k[:, ::5] *= np.float32(2.0 ** -75)  # denormal products and sums
    count = (rng.random(Nk) < 0.9).astype(np.int32)
    got = host(ops.block_scores(dev(q), dev(k), dev(count)))
    rows = np.unique(np.concatenate([np.arange(min(Nq, 5)), rng.integers(0, Nq, 12), [Nq - 1]]))
    for bh in range(BH):
        want = O.block_scores(q[bh:bh + 1, rows], k[bh:bh + 1], None)[0]
        want[:, count == 0] = -np.inf
        assert bits_equal(got[bh, rows], want), bh
    # infinities and NaN as fmaf has them, only in their own row and column
    q[0, 0, 0], k[0, -1, D - 1] = np.inf, np.nan
    odd = host(ops.block_scores(dev(q), dev(k), None))
    full = host(ops.block_scores(dev(np.nan_to_num(q, posinf=1.0)), dev(np.nan_to_num(k)), None))
    assert np.isnan(odd[0, :, -1]).all() and not np.isfinite(odd[0, 0]).any()
    assert bits_equal(odd[:, 1:, :-1], full[:, 1:, :-1])
