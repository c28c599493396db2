"""GPU parity of the prefill kernels at the sizes where their staging ends unevenly: short last stages, ragged tiles, small
and large shapes of each dispatch rule.  Against the CPU oracle, within 1e-5 * sum |terms| per output (the summation order is
all that differs), as the other matmul tests."""
import numpy as np
import pytest

import common
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    import cactus_amd
    return cactus_amd.Device(0)


def check(y, ref, what):
    err = np.abs(y.astype(np.float64) - ref["y"].astype(np.float64))
    bound = 1e-5 * ref["sum_abs"]
    assert (err <= bound).all(), "%s: worst error is %.3g x the tolerance" % (what, float((err / np.maximum(bound, 1e-300)).max()))


# (K, N, n): one stage that is short itself; one whole and one short; eight; split over workgroups with the short stage in the
# last slice; 64 x 128 tiles; 128 x 128 tiles
@pytest.mark.parametrize("wt", (O.Q4_0, O.Q8_0, O.Q5_0, O.IQ4_NL, O.Q4_1, O.Q5_1), ids=lambda t: O.TYPE_NAMES[t])
@pytest.mark.parametrize("K,N,n", [(64, 5, 49), (192, 131, 64), (960, 70, 133), (4160, 300, 130), (192, 4100, 1030), (320, 8200, 770)])
def test_block32_rows_with_a_short_last_stage(dev, orc, wt, K, N, n):
    rng = np.random.default_rng(K + N + wt)
    wq = orc.quantize_weights(wt, common.weights_f32(K + N, N, K))
    x = common.activations_f32(K + n, n, K)
    x[3] = 0
    x[5] = -np.abs(x[5])                      # negative sums: NaN bit patterns in the plane that follows the scales
    y = dev.mul_mat(wt, wq, x)
    rows = np.unique(np.concatenate([[0, N - 1], rng.choice(N, min(N, 200), replace=False)]))
    toks = np.unique(np.concatenate([[0, 3, 5, n - 1], rng.choice(n, min(n, 64), replace=False)]))
    ref = orc.mul_mat(wt, wq[rows], x[toks], nthreads=8, want=("sum_abs",))
    check(y[np.ix_(toks, rows)], ref, "short last stage")
    assert np.isfinite(y).all()
