"""GPU parity of the prefill kernels at the sizes where their staging ends unevenly: short last stages, ragged tiles, small
and large shapes of each dispatch rule.  Against the CPU oracle, within 1e-5 * sum |terms| per output (the summation order is
all that differs), as the other matmul tests."""
import numpy as np
import pytest

import common
import oracle as O
from test_gpu_routes import group_kernels, group_launches, mul_mat_id_launches, mul_mat_kernels, mul_mat_launches

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


# ---- Q3_K, Q2_K and IQ4_XS on the matrix cores ----
LOW_BIT = (O.Q3_K, O.Q2_K, O.IQ4_XS)


def random_rows(wt, rng, N, nsb):
    """Raw super-blocks: random bytes (every scale and quant occurs), d = dmin = 1; the first rows saturated."""
    w = rng.integers(0, 256, (N, nsb, O.BLOCK_BYTES[wt]), dtype=np.uint8)
    for r, fill in enumerate((0xFF, 0x00, 0x80, 0x7F)):
        w[r] = fill
    one = np.array([1.0], np.float16).view(np.uint8)
    w[..., slice(108, 110) if wt == O.Q3_K else slice(80, 82) if wt == O.Q2_K else slice(0, 2)] = one
    if wt == O.Q2_K:
        w[..., 82:84] = one
    return w.reshape(N, -1)


# (K, N, n): one super-block; ragged tiles; K split over workgroups with uneven slices; the GEMV passes that 9 tokens take on few
# short rows; 128 x 128 tiles; many tokens, few rows; the GEMM at the fewest tokens it is taken from; the staging kernel
@pytest.mark.parametrize("wt", LOW_BIT, ids=lambda t: O.TYPE_NAMES[t])
@pytest.mark.parametrize("K,N,n", [(256, 5, 41), (1024, 131, 65), (2304, 131, 70), (4096, 300, 9), (512, 4100, 1030), (768, 33, 1100),
                                   (14336, 70, 9), (2304, 8200, 70), (1280, 8100, 33), (512, 300, 96), (768, 131, 33), (2304, 12000, 70)])
def test_low_bit_kquant_gemm(dev, orc, wt, K, N, n):
    rng = np.random.default_rng(K + N + wt)
    w = random_rows(wt, rng, N, K // 256)
    x = common.activations_f32(K + n, n, K)
    x[3] = 0
    x[4] = 127.0
    x[5] = -127.0
    x[4:6, ::256] = -127.0
    if N == 12000:
        assert ("gemm_kq_kernel" in mul_mat_kernels(dev, wt, w, x)[1]) == (wt != O.Q2_K)
    y = dev.mul_mat(wt, w, x)
    rows = np.unique(np.concatenate([[0, 1, 2, 3, N - 1], rng.choice(N, min(N, 200), replace=False)]))
    toks = np.unique(np.concatenate([[0, 3, 4, 5, n - 1], rng.choice(n, min(n, 64), replace=False)]))
    ref = orc.mul_mat(wt, w[rows], x[toks], nthreads=8, want=("sum_abs",))
    check(y[np.ix_(toks, rows)], ref, "low-bit k-quant gemm")


# The GEMM whose waves expand their own rows, (K, N, n): two workgroups a CU, ragged rows and tokens; two k groups over an odd number
# of super-blocks; uneven slices and a last tile of one token (at 33 tokens by waves that share a tile); two k groups in two slices of different
# length (Q2_K, IQ4_XS) and unsplit
@pytest.mark.parametrize("wt", (O.Q4_K, O.Q5_K, O.Q6_K) + LOW_BIT, ids=lambda t: O.TYPE_NAMES[t])
@pytest.mark.parametrize("K,N,n", [(512, 4200, 1100), (1280, 4100, 260), (2816, 131, 33), (8448, 4100, 130), (2816, 131, 65), (8448, 4100, 200)])
def test_kquant_row_gemm(dev, orc, wt, K, N, n):
    rng = np.random.default_rng(K + N + wt)
    w = rng.integers(0, 256, (N, K // 256, O.BLOCK_BYTES[wt]), dtype=np.uint8)
    for r, fill in enumerate((0xFF, 0x00, 0x80, 0x7F)):
        w[r] = fill
    half = np.array([1.0], np.float16).view(np.uint8)
    for at in {O.Q4_K: (0, 2), O.Q5_K: (0, 2), O.Q6_K: (208,), O.Q3_K: (108,), O.Q2_K: (80, 82), O.IQ4_XS: (0,)}[wt]:
        w[..., at:at + 2] = half
    w = w.reshape(N, -1)
    x = common.activations_f32(K + n, n, K)
    x[3] = 0
    x[4] = 127.0
    x[5] = -127.0
    names = mul_mat_kernels(dev, wt, w, x)
    staged = wt in (O.Q6_K, O.Q3_K)
    if N == 131:
        assert ("gemm_kq_few" if n == 33 else "gemm_kq_kernel" if staged else "gemm_kr_kernel") in names[1] and len(names) == (2 if n == 33 else 3)
    elif K == 8448 and not (staged and n == 130):
        assert ("gemm_kq_kernel" if wt == O.Q6_K else "gemm_kr_kernelILi%dELi2ELi2E" % wt) in names[1]
    y = dev.mul_mat(wt, w, x)
    rows = np.unique(np.concatenate([[0, 1, 2, 3, N - 1], rng.choice(N, min(N, 150), replace=False)]))
    toks = np.unique(np.concatenate([[0, 3, 4, 5, n - 1], rng.choice(n, min(n, 48), replace=False)]))
    ref = orc.mul_mat(wt, w[rows], x[toks], nthreads=8, want=("sum_abs",))
    check(y[np.ix_(toks, rows)], ref, "k-quant row gemm")
    assert np.isfinite(y).all()


# K in eight slices of seven super-blocks that give each CU a workgroup of this kernel, tokens one past its 32-token walk and one short of it
@pytest.mark.parametrize("n", (31, 33))
@pytest.mark.parametrize("wt", (O.Q6_K, O.Q3_K), ids=lambda t: O.TYPE_NAMES[t])
def test_kquant_row_gemm_over_slices(dev, orc, wt, n):
    K, N = 14336, 4096
    w = np.tile(orc.quantize_weights(wt, common.weights_f32(wt, 128, K)), (N // 128, 1))
    w[4001] = w[3]
    x = common.activations_f32(K + n, n, K)
    assert mul_mat_launches(dev, wt, w, x) == 3
    y = dev.mul_mat(wt, w, x)
    ref = orc.mul_mat(wt, w[:128], x, nthreads=8, want=("sum_abs",))
    check(y[:, :128], ref, "slices")
    same = np.tile(y[:, :128], (1, N // 128))
    same[:, 4001] = y[:, 3]
    assert y.tobytes() == same.tobytes()


# Rows so far apart that a tile spans more than 2^32 bytes, and more than 2^32 bytes apart each: (type, stride, rows, tokens).  One whole tile
# and a ragged one; K split (3584 values at 20 tokens); rows that lie alone; 8 to 12 tokens, which the matrix-core GEMVs take of closer rows; 8 to 24
# tokens, which tiles of 32 rows take of closer rows, 2^32 bytes from a tile's first row to its last and just below that of a tile of 16
@pytest.mark.parametrize("wt,K,stride,N,n", [(O.Q4_K, 512, 140 << 20, 40, 70), (O.Q2_K, 3584, 150 << 20, 33, 20), (O.IQ4_XS, 256, (4 << 30) + 64, 3, 60),
                                             (O.Q5_K, 3584, (2 << 30) + 16, 5, 80), (O.Q4_K, 512, 300 << 20, 20, 8), (O.Q5_K, 512, 300 << 20, 20, 16),
                                             (O.Q4_0, 512, 300 << 20, 20, 9), (O.Q8_0, 512, 300 << 20, 20, 12),
                                             (O.Q4_K, 512, 140 << 20, 40, 8), (O.Q4_K, 512, 250 << 20, 40, 16), (O.Q6_K, 512, 250 << 20, 40, 12),
                                             (O.Q4_K, 512, 140 << 20, 40, 24), (O.Q3_K, 1024, 140 << 20, 40, 40), (O.IQ4_XS, 1024, 270 << 20, 20, 12)],
                         ids=lambda v: O.TYPE_NAMES[v] if isinstance(v, int) and v in O.TYPE_NAMES else None)
def test_rows_far_apart(dev, orc, wt, K, stride, N, n):
    L = dev.lib
    w = orc.quantize_weights(wt, common.weights_f32(K + N, N, K))
    x = common.activations_f32(K + n, n, K)
    dW, dx, dy = dev.alloc((N - 1) * stride + w.shape[1]), dev.to_device(x), dev.alloc(2 * n * N * 4)
    for r in range(N):
        dW.upload(w[r], r * stride)
    wsz = max(L.chip_mul_mat_workspace_size_n(wt, K, N, n), L.chip_mul_mat_id_workspace_size(wt, K, 1, 1, n, 1))
    ws, ids = dev.alloc(wsz), dev.to_device(np.zeros(n, np.int32))
    ref = orc.mul_mat(wt, w, x, nthreads=8, want=("sum_abs",))
    y2 = dy.ptr + n * N * 4
    for call in (lambda: L.chip_mul_mat(wt, dW.ptr, stride, K, N, dx.ptr, K, n, dy.ptr, N, ws.ptr, wsz, None),
                 lambda: L.chip_mul_mat_pair(wt, dW.ptr, dW.ptr, stride, K, N, dx.ptr, K, n, dy.ptr, y2, N, ws.ptr, wsz, None),
                 lambda: L.chip_mul_mat_id(wt, dW.ptr, stride, N * stride, K, N, 1, dx.ptr, K, 1, ids.ptr, 1, 1, n, dy.ptr, N, ws.ptr, wsz, None)):
        dev.check(L.chip_memset(dy.ptr, 0xFF, 2 * n * N * 4, None))
        dev.check(call())
        dev.sync()
        y = dy.download(np.float32, 2 * n * N).reshape(2, n, N)
        check(y[0], ref, "rows far apart")
        assert np.isnan(y[1]).all() or y[1].tobytes() == y[0].tobytes()


# The same rows beside a matrix that alone takes tiles of 32 rows, in one launch: 16 rows a tile for both
def test_rows_far_apart_in_a_group(dev, orc):
    import cactus_amd as ca
    L, wt, K, n, stride, N, near = dev.lib, O.Q4_K, 2048, 24, 140 << 20, 40, 8000
    w = orc.quantize_weights(wt, common.weights_f32(3, 160, K))
    x = common.activations_f32(4, n, K)
    dW, dV, dx, dy = dev.alloc((N - 1) * stride + w.shape[1]), dev.to_device(np.tile(w, (near // 160, 1))), dev.to_device(x), dev.alloc(n * (N + near) * 4)
    for r in range(N):
        dW.upload(w[r], r * stride)
    mats = (ca.Mat * 2)(ca.Mat(wt, dW.ptr, stride, N, dy.ptr, N, None, 0), ca.Mat(wt, dV.ptr, w.shape[1], near, dy.ptr + 4 * n * N, near, None, 0))
    wsz = max(L.chip_mul_mat_workspace_size_n(wt, K, m, n) for m in (N, near))
    ws = dev.alloc(wsz)
    dev.check(L.chip_mul_mat_group(mats, 2, K, dx.ptr, K, n, ws.ptr, wsz, None))
    dev.sync()
    y = dy.download(np.float32, n * (N + near))
    check(y[:n * N].reshape(n, N), orc.mul_mat(wt, w[:N], x, nthreads=8, want=("sum_abs",)), "far member")
    assert np.array_equal(y[n * N:].reshape(n, -1, 160)[:, :, :N], np.repeat(y[:n * N].reshape(n, 1, N), near // 160, axis=1))


@pytest.mark.parametrize("wt", LOW_BIT, ids=lambda t: O.TYPE_NAMES[t])
def test_low_bit_kquant_integer_sums_bit_exact(dev, orc, wt):
    """d = dmin = 1 and activation scale 1: the output of one super-block is the integer sumi - summ itself (below 2^24)."""
    K, N, n = 256, 150, 56
    rng = np.random.default_rng(77 + wt)
    w = random_rows(wt, rng, N, 1)
    x = rng.integers(-127, 128, (n, K)).astype(np.float32)
    x[:, 0] = -127.0
    x[7, 1:] = 0.0
    aq = orc.quantize_activation(O.Q8_K, x)
    y = dev.mul_mat(wt, w, x)
    want = np.zeros((n, N), np.int64)
    for t in range(n):
        for i in range(N):
            _, isum, imin = orc.vec_dot(wt, K, w[i], aq[t], want_sums=True)
            want[t, i] = int(isum.sum()) - (int(imin.sum()) if wt == O.Q2_K else 0)
    assert np.abs(want).max() < 2 ** 24
    assert np.array_equal(y.astype(np.int64), want)


@pytest.mark.parametrize("n_tokens", (90, 700))
@pytest.mark.parametrize("wt", LOW_BIT, ids=lambda t: O.TYPE_NAMES[t])
def test_low_bit_kquant_expert_groups(dev, orc, wt, n_tokens):
    """64 pairs and more, an expert nobody picks: a GEMV per pair while that is ahead (90 tokens here), then the pairs grouped by
    expert and run through the GEMM (700 tokens; ragged groups of several token tiles)."""
    K, N, n_as, n_used = 512, 70, 5, 2
    rng = np.random.default_rng(wt)
    experts = np.stack([random_rows(wt, rng, N, K // 256) for _ in range(n_as)])
    x = common.activations_f32(wt, n_tokens, K).reshape(n_tokens, 1, K)
    ids = np.stack([rng.permutation(4)[:n_used] for _ in range(n_tokens)]).astype(np.int32)
    ref = orc.mul_mat_id(wt, experts, x, ids, want=("sum_abs",))
    check(dev.mul_mat_id(wt, experts, x, ids), ref, "expert groups")


# ---- attention matmuls of a prompt: head size, heads, KV heads, tokens, cached positions ----
# one 64-row tile by 64 and by 32 columns; 96 and 256 rows (a ragged and two row tiles); 3 KV heads; K no multiple of a stage;
# kq with 128 x 128 tiles and with n_kv below and above the fp32 rule's 256 rows
@pytest.mark.parametrize("hd,nh,nkv,n,kv", [(64, 32, 8, 512, 1064), (64, 15, 5, 133, 160), (96, 24, 8, 260, 104), (256, 6, 3, 75, 264),
                                            (128, 8, 8, 257, 2056), (128, 4, 2, 70, 256)])
def test_attention_matmuls_of_a_prompt(dev, orc, hd, nh, nkv, n, kv):
    rng = np.random.default_rng(hd + n + kv)
    q = rng.standard_normal((nh, n, hd)).astype(np.float32)
    kc = rng.standard_normal((nkv, kv, hd)).astype(np.float16)
    vt = rng.standard_normal((nkv, hd, kv)).astype(np.float16)
    p = rng.random((nh, n, kv)).astype(np.float32)
    toks = np.unique(np.concatenate([[0, n - 1], rng.choice(n, 40, replace=False)]))
    for w, x in ((kc, q), (vt, p)):
        y = dev.mul_mat_f16_batched(w, x)
        ref = orc.mul_mat_f16_batched(w, np.ascontiguousarray(x[:, toks]), want=("sum_abs",))
        check(y[:, toks], ref, "attention matmul")


# ---- F16 weights: the loads run one to three stages of 64 values ahead of the products ----
# multiples of four stages (K is a multiple of 256), every remainder of three among them; odd stage counts of the two-deep form come
# with the cached positions of the attention test above.  Ragged 64 x 64 tiles three and two stages ahead; 128 x 128 tiles one and two
@pytest.mark.parametrize("N,n", [(131, 70), (1300, 1290), (2050, 2049), (2041, 2035)])
@pytest.mark.parametrize("K", (256, 512, 768, 1280))
def test_f16_gemm_stage_counts(dev, orc, K, N, n):
    rng = np.random.default_rng(K + N)
    w = orc.quantize_weights(O.F16, common.weights_f32(K + N, N, K))
    x = common.activations_f32(K + n, n, K)
    y = dev.mul_mat(O.F16, w, x)
    rows = np.unique(np.concatenate([[0, N - 1], rng.choice(N, min(N, 200), replace=False)]))
    toks = np.unique(np.concatenate([[0, n - 1], rng.choice(n, min(n, 64), replace=False)]))
    ref = orc.mul_mat(O.F16, w[rows], x[toks], nthreads=8, want=("sum_abs",))
    check(y[np.ix_(toks, rows)], ref, "F16 gemm, %d stages" % (K // 64))


# (K, N, n): 64 x 32 tiles with one token in the last, and two stages of 128 values; 64 x 64 tiles of one to two workgroups a CU; more
@pytest.mark.parametrize("K,N,n", [(256, 70, 33), (1280, 1030, 97), (768, 2050, 520), (512, 8200, 333)])
def test_f16_gemm_by_the_tiles_a_cu_gets(dev, orc, K, N, n):
    rng = np.random.default_rng(K + N)
    w = orc.quantize_weights(O.F16, common.weights_f32(K + N, N, K))
    x = common.activations_f32(K + n, n, K)
    y = dev.mul_mat(O.F16, w, x)
    rows = np.unique(np.concatenate([[0, N - 1], rng.choice(N, 60, replace=False)]))
    toks = np.unique(np.concatenate([[0, n - 1], rng.choice(n, 30, replace=False)]))
    check(y[np.ix_(toks, rows)], orc.mul_mat(O.F16, w[rows], x[toks], nthreads=8, want=("sum_abs",)), "F16 gemm")


# ---- matrices on one activation whose tiles share a launch: the bits of each by itself ----
# (type, K, rows of each, n): one row tile and a ragged one, 64 x 64 tiles; more row tiles than CUs; a first member of one row; two
# super-blocks and one of another type between; a K that is no multiple of a stage; Q6_K and Q3_K in the staging kernel (a launch each) and beside it
@pytest.mark.parametrize("wt,K,rows,n", [(O.Q4_0, 960, (960, 320, 320), 133), (O.Q8_0, 192, (1, 65, 130, 64), 70), (O.Q5_1, 256, (8200, 8190), 130),
                                         (O.Q4_K, 1024, (129, 128, 1), 140), (O.Q5_K, 512, (4100, 4100), 260), (O.Q6_K, 256, (300, 70), 65), (O.Q6_K, 256, (4200, 4106), 520),
                                         (O.Q3_K, 512, (200, 1030), 129), (O.Q3_K, 512, (4200, 4106), 520), (O.Q2_K, 768, (33, 500), 200), (O.IQ4_XS, 768, (256, 65, 130), 41)],
                         ids=lambda v: O.TYPE_NAMES[v] if isinstance(v, int) and v in O.TYPE_NAMES else None)
def test_grouped_gemms_equal_single_calls(dev, orc, wt, K, rows, n):
    rng = np.random.default_rng(K + n)
    other = O.Q4_K if wt in (O.Q5_K, O.Q6_K, O.Q3_K, O.Q2_K) else None
    types = [wt] * len(rows)
    if other is not None and len(rows) == 2:
        types.insert(1, other)
        rows = (rows[0], 64, rows[1])
    ws = [(t, orc.quantize_weights(t, common.weights_f32(K + N + i, N, K))) for i, (t, N) in enumerate(zip(types, rows))]
    x = common.activations_f32(K + n, n, K)
    staged = wt in (O.Q6_K, O.Q3_K) and rows[0] < 4000
    assert group_launches(dev, [(t, W.shape[0]) for t, W in ws], K, n) == 1 + (len(ws) if staged else len(set(types)))
    ys = dev.mul_mat_group(ws, x)
    for i, ((t, W), y) in enumerate(zip(ws, ys)):
        assert y.tobytes() == dev.mul_mat(t, W, x).tobytes(), i
    if len(rows) == 2 or other is not None:
        a, b = ws[0], ws[-1]
        N = min(a[1].shape[0], b[1].shape[0])
        y1, y2 = dev.mul_mat_pair(wt, a[1][:N], b[1][:N], x)
        assert y1.tobytes() == dev.mul_mat(wt, a[1][:N], x).tobytes() and y2.tobytes() == dev.mul_mat(wt, b[1][:N], x).tobytes()
    toks = np.unique(np.concatenate([[0, n - 1], rng.choice(n, 40, replace=False)]))
    W = ws[-1][1]
    pick = np.unique(np.concatenate([[0, W.shape[0] - 1], rng.choice(W.shape[0], min(W.shape[0], 100), replace=False)]))
    ref = orc.mul_mat(ws[-1][0], W[pick], x[toks], nthreads=8, want=("sum_abs",))
    check(ys[-1][np.ix_(toks, pick)], ref, "last member")


# Q4_K and Q5_K above 2048 values, whose members run in one k group and in two alone: one launch in two groups, or in one that adds as two do where that is what
# a member has alone (an odd number of super-blocks, a last tile of four tokens, ragged rows)
@pytest.mark.parametrize("wt,K,rows,n,alone,joined", [(O.Q4_K, 2560, (6912, 6912), 200, (2, 2), "1ELi2ELb0ELb1E"), (O.Q5_K, 2304, (3000, 2900), 260, (2, 2), "2ELi2ELb0ELb0E"),
                                                      (O.Q5_K, 2304, (3000, 5990), 260, (2, 2), "1ELi2ELb0ELb1E"), (O.Q4_K, 2304, (3000, 8001), 260, (2, 1), "1ELi2ELb0ELb1E"),
                                                      (O.Q4_K, 2304, (8001, 2, 3000), 260, (1, 0, 2), None), (O.Q5_K, 2304, (8001, 3000), 260, (1, 2), "1ELi2ELb0ELb1E"),
                                                      (O.Q4_K, 4096, (4096, 4096), 512, (2, 2), "1ELi2ELb0ELb1E"), (O.Q4_K, 2304, (8001, 9000), 260, (1, 1), "1ELi2ELb0ELb0E")],
                         ids=lambda v: O.TYPE_NAMES[v] if isinstance(v, int) and v in O.TYPE_NAMES else None)
def test_joined_k_groups_equal_single_calls(dev, orc, wt, K, rows, n, alone, joined):
    q = orc.quantize_weights(wt, common.weights_f32(K + n, 101, K))
    ws = [np.roll(np.tile(q, (-(-N // 101), 1))[:N], i, axis=0) for i, N in enumerate(rows)]
    x = common.activations_f32(K + n, n, K)
    for w, groups in zip(ws, alone):
        assert groups == 0 or "gemm_kr_kernelILi%dELi2ELi%dELi2ELb0ELb0E" % (wt, groups) in mul_mat_kernels(dev, wt, w, x)[1]
    names = group_kernels(dev, [(wt, N) for N in rows], K, n)
    if joined is not None:
        assert len(names) == 2 and "gemm_kr_kernelILi%dELi2ELi%s" % (wt, joined) in names[1]
    for w, y in zip(ws, dev.mul_mat_group([(wt, w) for w in ws], x)):
        assert y.tobytes() == dev.mul_mat(wt, w, x).tobytes()
    if rows[0] == rows[1]:
        y1, y2 = dev.mul_mat_pair(wt, ws[0], ws[1], x)
        assert y1.tobytes() == dev.mul_mat(wt, ws[0], x).tobytes() and y2.tobytes() == dev.mul_mat(wt, ws[1], x).tobytes()


# ---- expert groups: pairs of each expert around a tile of 64, more experts than a turn of the scan takes, more pairs than are kept in registers ----
@pytest.mark.parametrize("counts,n_used", [((0, 1, 31, 33, 64, 65, 129), 1), ((3, 0) * 160, 1), ((2100, 2101, 0, 2200, 1999), 2)],
                         ids=("tile edges", "320 experts", "8400 pairs"))
@pytest.mark.parametrize("wt", (O.Q4_K, O.Q6_K, O.Q4_0, O.F16), ids=lambda t: O.TYPE_NAMES[t])
def test_expert_groups(dev, orc, wt, counts, n_used):
    K, N = 256, 130
    rng = np.random.default_rng(wt + len(counts))
    ids = rng.permutation(np.repeat(np.arange(len(counts)), counts)).astype(np.int32).reshape(-1, n_used)
    n_tokens = ids.shape[0]
    assert mul_mat_id_launches(dev, wt, K, N, len(counts), n_used, n_tokens) == 3
    experts = np.stack([orc.quantize_weights(wt, common.weights_f32(wt + e, N, K)) for e in range(len(counts))])
    x = common.activations_f32(wt, n_tokens, K).reshape(n_tokens, 1, K)
    check(dev.mul_mat_id(wt, experts, x, ids), orc.mul_mat_id(wt, experts, x, ids, want=("sum_abs",)), "expert groups")


# Ids that name no expert, among the pairs that the grouping keeps in registers (the first 8192) and behind them: their rows are not written
@pytest.mark.parametrize("wt", (O.Q4_K, O.Q4_0, O.F16), ids=lambda t: O.TYPE_NAMES[t])
def test_expert_groups_skip_ids_out_of_range(dev, orc, wt):
    K, N, n_as, n_used, n_tokens = 256, 130, 5, 2, 4300
    rng = np.random.default_rng(wt)
    ids = rng.integers(0, n_as, (n_tokens, n_used)).astype(np.int32)
    at = np.array([0, 63, 1024, 8191, 8192, 8193, 8500, 2 * n_tokens - 1])
    bad = np.zeros(2 * n_tokens, bool)
    bad[at] = True
    ok = ids.copy()
    ids.reshape(-1)[at] = [-1, n_as, 2 ** 31 - 1, -2 ** 31, n_as, -1, 4096, n_as + 5]
    assert mul_mat_id_launches(dev, wt, K, N, n_as, n_used, n_tokens) == 3
    experts = np.stack([orc.quantize_weights(wt, common.weights_f32(wt + e, N, K)) for e in range(n_as)])
    x = common.activations_f32(wt, n_tokens, K).reshape(n_tokens, 1, K)
    y = dev.mul_mat_id(wt, experts, x, ids).reshape(-1, N)
    ref = orc.mul_mat_id(wt, experts, x, ok, want=("sum_abs",))
    assert np.isnan(y[bad]).all() and np.isfinite(y[~bad]).all()
    check(y[~bad], {k: ref[k].reshape(-1, N)[~bad] for k in ("y", "sum_abs")}, "bad ids")


# Few tiles of these types run in the staging kernel (64 rows x 128 pairs), the same rows inside a large matrix in the other one
@pytest.mark.parametrize("wt", (O.Q6_K, O.Q3_K, O.IQ4_XS), ids=lambda t: O.TYPE_NAMES[t])
def test_staged_expert_groups_equal_the_row_kernel(dev, orc, wt):
    K, N, counts = 768, 70, (1, 64, 0, 65, 128, 129, 300)
    rng = np.random.default_rng(wt)
    w = np.stack([orc.quantize_weights(wt, common.weights_f32(wt + e, N, K)) for e in range(len(counts))])
    ids = rng.permutation(np.repeat(np.arange(len(counts)), counts)).astype(np.int32).reshape(-1, 1)
    x = common.activations_f32(wt, ids.shape[0], K)[:, None]
    y = dev.mul_mat_id(wt, w, x, ids)
    check(y, orc.mul_mat_id(wt, w, x, ids, want=("sum_abs",)), "staged groups")
    large = np.concatenate([np.tile(w, (1, 70, 1)), w], axis=1)
    assert np.ascontiguousarray(dev.mul_mat_id(wt, large, x, ids)[:, :, -N:]).tobytes() == y.tobytes()


# An expert larger than an XCD's L2 has its token tiles in columns of 8: one short tile, a column and one tile, two columns and a short one, none
@pytest.mark.parametrize("wt,K,N", [(O.Q4_0, 1024, 8000), (O.Q4_K, 2048, 4100)], ids=lambda v: O.TYPE_NAMES.get(v))
def test_large_experts_with_many_token_tiles(dev, orc, wt, K, N):
    counts = (3, 520, 0, 1060)
    rng = np.random.default_rng(K)
    w = np.stack([np.roll(np.tile(orc.quantize_weights(wt, common.weights_f32(K + e, 100, K)), (-(-N // 100), 1))[:N], e, axis=0) for e in range(4)])
    assert w[0].nbytes > 4 << 20
    ids = rng.permutation(np.repeat(np.arange(4), counts)).astype(np.int32).reshape(-1, 1)
    x = common.activations_f32(K, ids.shape[0], K)
    y = dev.mul_mat_id(wt, w, x[:, None], ids)[:, 0]
    for e in (0, 1, 3):
        of = ids[:, 0] == e
        if counts[e] > 100:
            assert y[of].tobytes() == dev.mul_mat(wt, w[e], x[of], split_k=False).tobytes()
        check(y[of][:50, :150], orc.mul_mat(wt, w[e, :150], x[of][:50], nthreads=8, want=("sum_abs",)), "expert %d" % e)


# ---- rows too short to be split: few tokens and expert pairs as near to the 64-bit sums as the GEMV's 8 tokens are ----
def distance(orc, wt, K, w, x, y):
    """2-norm of y - sum in 64 bits over that of the sum, of the same quantized operands"""
    aq = orc.quantize_activation(O.VEC_DOT_TYPE[wt], x)
    ref = np.array([[orc.vec_dot_exact(wt, K, r, a)[0] for r in w] for a in aq])
    return np.linalg.norm(y - ref) / np.linalg.norm(ref)


# 1600 outputs pin a rounding error's 2-norm to 2 per cent, so a tenth more is a larger error (one chain of additions: 1.3 to 2 times)
@pytest.mark.parametrize("K,n", [(512, 17), (960, 17), (1024, 47), (1920, 32)])
@pytest.mark.parametrize("wt", (O.Q4_0, O.Q8_0, O.Q5_0, O.IQ4_NL, O.Q4_1, O.Q5_1), ids=lambda t: O.TYPE_NAMES[t])
def test_block32_few_tokens_as_near_as_the_gemv(dev, orc, wt, K, n):
    N = 100
    w = orc.quantize_weights(wt, common.weights_f32(K + N, N, K))
    x = common.activations_f32(K + n, n, K)
    gemv = np.concatenate([dev.mul_mat(wt, w, x[i:i + 4]) for i in range(0, n, 4)])
    y = dev.mul_mat(wt, w, x)
    check(y, orc.mul_mat(wt, w, x, nthreads=8, want=("sum_abs",)), "few tokens")
    assert distance(orc, wt, K, w, x, y) <= 1.1 * distance(orc, wt, K, w, x, gemv)


# 60 pairs of 4 experts (grouped, but for the types with a minimum) against the same tokens three at a time (a GEMV per pair)
@pytest.mark.parametrize("K", (512, 4096))
@pytest.mark.parametrize("wt", (O.Q4_0, O.Q8_0, O.Q5_0, O.IQ4_NL, O.Q4_1, O.Q5_1), ids=lambda t: O.TYPE_NAMES[t])
def test_block32_few_expert_pairs_as_near_as_the_gemv(dev, orc, wt, K):
    N, n_as, n_used, n = 5000, 4, 4, 15
    w = np.tile(orc.quantize_weights(wt, common.weights_f32(K, 250, K)), (n_as * N // 250, 1)).reshape(n_as, N, -1)
    x = common.activations_f32(K, n, K).reshape(n, 1, K)
    ids = np.tile(np.arange(4, dtype=np.int32), (n, 1))
    y = dev.mul_mat_id(wt, w, x, ids)[:, :, :100].reshape(n, -1)
    gemv = np.concatenate([dev.mul_mat_id(wt, w, x[i:i + 3], ids[i:i + 3]) for i in range(0, n, 3)])[:, :, :100].reshape(n, -1)
    rows = w[:, :100].reshape(400, -1)
    assert distance(orc, wt, K, rows, x[:, 0], y) <= 1.1 * distance(orc, wt, K, rows, x[:, 0], gemv)


# 60 pairs of 4 experts (grouped up to some length of the rows) against the same tokens three at a time (a GEMV per pair)
@pytest.mark.parametrize("K", (3840, 4096, 8448))
@pytest.mark.parametrize("wt", (O.Q4_K, O.Q5_K, O.Q6_K) + LOW_BIT, ids=lambda t: O.TYPE_NAMES[t])
def test_kquant_few_expert_pairs_as_near_as_the_gemv(dev, orc, wt, K):
    N, n_as, n_used, n = 5000, 4, 4, 15
    w = np.tile(orc.quantize_weights(wt, common.weights_f32(K, 250, K)), (n_as * N // 250, 1)).reshape(n_as, N, -1)
    x = common.activations_f32(K, n, K).reshape(n, 1, K)
    ids = np.tile(np.arange(4, dtype=np.int32), (n, 1))
    y = dev.mul_mat_id(wt, w, x, ids)[:, :, :100].reshape(n, -1)
    gemv = np.concatenate([dev.mul_mat_id(wt, w, x[i:i + 3], ids[i:i + 3]) for i in range(0, n, 3)])[:, :, :100].reshape(n, -1)
    assert (y.tobytes() != gemv.tobytes()) == (K <= {O.Q4_K: 8192, O.Q5_K: 8192, O.Q2_K: 4096}.get(wt, 3840))
    rows = w[0, :100]
    assert distance(orc, wt, K, rows, x[:, 0], y[:, :100]) <= 1.1 * distance(orc, wt, K, rows, x[:, 0], gemv[:, :100])


# K in eight slices of one super-block (Q2_K, IQ4_XS) and in two of four: no further off than rows walked whole (9216 outputs: within 1 per cent).  At 64
# tokens eight waves share it
@pytest.mark.parametrize("n", (64, 72))
@pytest.mark.parametrize("wt", LOW_BIT, ids=lambda t: O.TYPE_NAMES[t])
def test_slices_of_k_as_near_as_whole_rows(dev, orc, wt, n):
    K, N = 2048, 128
    w = orc.quantize_weights(wt, common.weights_f32(K + N, N, K))
    x = common.activations_f32(K + n, n, K)
    names = mul_mat_kernels(dev, wt, w, x)
    assert "gemm_kq_few_kernel" in names[1] if n == 64 else "sum_slices_kernel" in names[2]
    whole, slices = dev.mul_mat(wt, w, x, split_k=False), dev.mul_mat(wt, w, x)
    assert slices.tobytes() != whole.tobytes()
    assert distance(orc, wt, K, w, x, slices) <= 1.03 * distance(orc, wt, K, w, x, whole)


# ---- K-quants of few tokens: tiles of 16 or 32 rows and tokens whose super-blocks are shared by waves ----
# (K, N, n): one row and two super-blocks, a wave each; ragged rows and more waves than a row has left over; 16 and 17 tokens; a second token tile of one
# token; an odd number of super-blocks over eight waves; more row tiles than a turn of workgroups; more waves than 48 KB of local memory serve
@pytest.mark.parametrize("wt", (O.Q4_K, O.Q5_K, O.Q6_K) + LOW_BIT, ids=lambda t: O.TYPE_NAMES[t])
@pytest.mark.parametrize("K,N,n", [(512, 1, 9), (1280, 33, 16), (1280, 47, 17), (1024, 130, 33), (2816, 300, 40), (1024, 20000, 9), (14336, 4000, 9)])
def test_kquant_few_tokens(dev, orc, wt, K, N, n):
    w = np.tile(orc.quantize_weights(wt, common.weights_f32(K + N, min(N, 200), K)), (-(-N // 200), 1))[:N]
    x = common.activations_f32(K + n, n, K)
    x[3] = 0
    assert mul_mat_launches(dev, wt, w, x) == 2
    y = dev.mul_mat(wt, w, x)
    assert y.tobytes() == dev.mul_mat(wt, w, x).tobytes() and np.array_equal(y[:, 200:], y[:, :max(N - 200, 0)] if N < 400 else y[:, :-200])
    rows = np.unique(np.concatenate([np.arange(min(N, 60)), [N - 1]]))
    check(y[:, rows], orc.mul_mat(wt, w[rows], x, nthreads=8, want=("sum_abs",)), "few tokens")
    gemv = np.concatenate([dev.mul_mat(wt, w, x[i:i + 4]) for i in range(0, n, 4)])
    if len(rows) > 40:                        # (2-norms of some hundred outputs: within a tenth)
        assert distance(orc, wt, K, w[rows], x, y[:, rows]) <= 1.1 * distance(orc, wt, K, w[rows], x, gemv[:, rows])


# Every form (row tiles, token tiles) with rows and tokens left over.  Rows of up to three super-blocks, and Q2_K and IQ4_XS, are added in 64 bits: a value is
# its sum rounded once.  The others: no further off than the GEMV.  (Some thousand outputs, some hundred of the smallest: their 2-norm varies by less than a twentieth)
@pytest.mark.parametrize("wt", (O.Q4_K, O.Q5_K, O.Q6_K) + LOW_BIT, ids=lambda t: O.TYPE_NAMES[t])
@pytest.mark.parametrize("K,N,n,form", [(512, 40, 12, (2, 1)), (512, 47, 25, (2, 2)), (1024, 24003, 12, (2, 1)), (1024, 16005, 20, (2, 2)), (2304, 2100, 75, (2, 2)),
                                        (2560, 1100, 140, (2, 2)), (1024, 270, 1111, (1, 2)), (4608, 300, 64, (1, 2)), (8192, 1000, 9, (1, 1))])
def test_kquant_few_tokens_by_form(dev, orc, wt, K, N, n, form):
    if (K, n) in {O.Q3_K: ((512, 25),), O.Q2_K: ((512, 25), (1024, 20))}.get(wt, ()):
        pytest.skip("another kernel is estimated ahead")
    wide = K <= 768 or wt in (O.Q2_K, O.IQ4_XS)
    q = orc.quantize_weights(wt, common.weights_f32(K + N, min(N, 61), K))
    w = np.tile(q, (-(-N // len(q)), 1))[:N]
    x = common.activations_f32(K + n, n, K)
    names = mul_mat_kernels(dev, wt, w, x)
    assert len(names) == 2 and "gemm_kq_few_kernelILi%dELi%dELi%dELb%dE" % ((wt,) + form + (wide,)) in names[1]
    y = dev.mul_mat(wt, w, x)
    assert np.array_equal(y, np.tile(y[:, :len(q)], (1, -(-N // len(q))))[:, :N])
    toks = np.unique(np.linspace(0, n - 1, 40).astype(int))
    aq = orc.quantize_activation(O.VEC_DOT_TYPE[wt], x[toks])
    ref = np.array([[orc.vec_dot_exact(wt, K, r, a)[0] for r in q] for a in aq])
    least = ref.astype(np.float32) if wide else np.concatenate([dev.mul_mat(wt, q, x[toks[i:i + 4]]) for i in range(0, len(toks), 4)])
    assert np.linalg.norm(y[toks, :len(q)] - ref) <= 1.05 * np.linalg.norm(least - ref)


# members of one and of two types, in any order: one launch behind the quantizer, the bits of the single calls
@pytest.mark.parametrize("types", [(O.Q4_K, O.Q4_K, O.Q6_K), (O.Q6_K, O.Q3_K), (O.IQ4_XS, O.Q2_K, O.IQ4_XS), (O.Q5_K, O.Q4_K), (O.Q5_K, O.Q5_K, O.Q5_K), (O.Q2_K, O.Q6_K)],
                         ids=lambda ts: "-".join(O.TYPE_NAMES[t] for t in ts))
@pytest.mark.parametrize("K,n", [(1024, 9), (1024, 20), (512, 12)])
def test_kquant_few_tokens_in_a_group(dev, orc, types, K, n):
    ws = [(t, orc.quantize_weights(t, common.weights_f32(K + i, N, K))) for i, (t, N) in enumerate(zip(types, (200, 33, 129)))]
    x = common.activations_f32(K + n, n, K)
    assert group_launches(dev, [(t, w.shape[0]) for t, w in ws], K, n) == 2
    for (t, w), y in zip(ws, dev.mul_mat_group(ws, x)):
        assert y.tobytes() == dev.mul_mat(t, w, x).tobytes(), O.TYPE_NAMES[t]


# members that take tiles of 16 and of 32 rows alone: of 32 for all of one type, of 16 where there are two types
@pytest.mark.parametrize("types,kernel", [((O.Q4_K,) * 3, "gemm_kq_few_kernelILi12ELi2ELi2E"), ((O.Q3_K,) * 3, "gemm_kq_few_kernelILi11ELi2ELi2E"),
                                          ((O.Q4_K, O.Q6_K, O.Q6_K), "gemm_kq_few_two_kernelILi12ELi14ELi2E")], ids=("one type", "Q3_K", "two types"))
def test_kquant_few_tokens_in_a_group_of_tall_and_short_tiles(dev, orc, types, kernel):
    K, n, rows = 2304, 40, (2001, 2107, 33)
    q = [orc.quantize_weights(t, common.weights_f32(K + i, 50, K)) for i, t in enumerate(types)]
    ws = [(t, np.tile(w, (-(-N // 50), 1))[:N]) for t, w, N in zip(types, q, rows)]
    x = common.activations_f32(K, n, K)
    for (t, w), rt in zip(ws, (1, 2, 1)):
        assert "gemm_kq_few_kernelILi%dELi%dELi2E" % (t, rt) in mul_mat_kernels(dev, t, w, x)[1]
    names = group_kernels(dev, [(t, w.shape[0]) for t, w in ws], K, n)
    assert len(names) == 2 and kernel in names[1]
    for (t, w), y in zip(ws, dev.mul_mat_group(ws, x)):
        assert y.tobytes() == dev.mul_mat(t, w, x).tobytes(), w.shape


# an infinite weight scale gives infinities, not NaN, also where the roundings of the sum are kept
@pytest.mark.parametrize("wt", (O.Q4_0, O.Q8_0, O.Q5_0, O.IQ4_NL), ids=lambda t: O.TYPE_NAMES[t])
def test_block32_few_tokens_with_an_infinite_scale(dev, orc, wt):
    K, N, n = 768, 70, 20
    w = orc.quantize_weights(wt, common.weights_f32(K + N, N, K))
    w[5, :2] = np.array([np.inf], np.float16).view(np.uint8)
    w[7, 10 * (w.shape[1] // 24):][:2] = np.array([-np.inf], np.float16).view(np.uint8)
    x = common.activations_f32(K + n, n, K)
    aq = orc.quantize_activation(O.VEC_DOT_TYPE[wt], x)
    ref = np.array([[orc.vec_dot_exact(wt, K, w[r], a)[0] for r in (5, 7)] for a in aq])
    y = dev.mul_mat(wt, w, x)
    assert np.isinf(ref).sum() > n and np.array_equal(y[:, (5, 7)], ref, equal_nan=True)
    assert np.isfinite(np.delete(y, (5, 7), axis=1)).all()


# ... and so does an infinite activation scale (values above 127 * 65504) or block sum (32 values that add up to more than 65504), whichever wave has the block
@pytest.mark.parametrize("K,n", [(768, 20), (1344, 80)])
@pytest.mark.parametrize("wt", (O.Q4_0, O.Q8_0, O.Q5_0, O.IQ4_NL, O.Q4_1, O.Q5_1), ids=lambda t: O.TYPE_NAMES[t])
def test_block32_few_tokens_with_an_infinite_activation_scale(dev, orc, wt, K, n):
    N = 70
    w = orc.quantize_weights(wt, common.weights_f32(K + N, N, K))
    x = common.activations_f32(K + n, n, K)
    blocks = K // 32
    for t in range(blocks // 2):
        x[t, 64 * t + 5] = 1e7 if t % 2 else -1e7
    x[n - 2, 320:352] = 3000.0
    if n == 80:
        assert "gemm_blk32_few_kernel" in mul_mat_kernels(dev, wt, w, x)[1]
    aq = orc.quantize_activation(O.VEC_DOT_TYPE[wt], x)
    ref = np.array([[orc.vec_dot_exact(wt, K, r, a)[0] for r in w] for a in aq])
    y = dev.mul_mat(wt, w, x)
    assert not np.isfinite(ref[:blocks // 2]).any() and np.isinf(ref).any() and np.isinf(ref[n - 2]).any() == (wt in (O.Q4_1, O.Q5_1))
    assert np.array_equal(np.where(np.isfinite(ref), 0, ref), np.where(np.isfinite(y), 0, y), equal_nan=True)


# ---- the GEMM from 17 tokens on, from 25 with few rows of 1536 values and more; the token in front of each line; a type with a minimum: GEMV passes ----
@pytest.mark.parametrize("K,N,n", [(256, 33, 17), (960, 130, 16), (960, 130, 17), (1472, 70, 31), (1536, 130, 24), (1536, 130, 25), (1920, 2049, 17)])
@pytest.mark.parametrize("wt", (O.Q4_0, O.Q8_0, O.Q5_1, O.IQ4_NL), ids=lambda t: O.TYPE_NAMES[t])
def test_block32_short_rows_of_few_tokens(dev, orc, wt, K, N, n):
    w = orc.quantize_weights(wt, common.weights_f32(K + N, N, K))
    x = common.activations_f32(K + n, n, K)
    check(dev.mul_mat(wt, w, x), orc.mul_mat(wt, w, x, nthreads=8, want=("sum_abs",)), "%d tokens" % n)


# ---- 15 and 16 pairs (a GEMV each), 16 pairs of many short rows (grouped), 130 pairs on many experts with few rows (a GEMV each) ----
@pytest.mark.parametrize("n_tokens,n_used,n_as,K,N,grouped", [(15, 1, 2, 4096, 2000, False), (8, 2, 2, 4096, 2000, False), (15, 1, 4, 256, 4000, False),
                                                              (4, 4, 4, 256, 4000, True), (65, 2, 64, 512, 24, False)])
@pytest.mark.parametrize("wt", (O.Q4_K, O.Q3_K, O.Q4_0), ids=lambda t: O.TYPE_NAMES[t])
def test_expert_matmul_of_few_pairs(dev, orc, wt, n_tokens, n_used, n_as, K, N, grouped):
    assert (mul_mat_id_launches(dev, wt, K, N, n_as, n_used, n_tokens) == 3) == grouped
    rng = np.random.default_rng(n_tokens + wt)
    experts = np.stack([orc.quantize_weights(wt, common.weights_f32(wt + e, N, K)) for e in range(n_as)])
    x = common.activations_f32(wt, n_tokens, K).reshape(n_tokens, 1, K)
    ids = np.stack([rng.permutation(n_as)[:n_used] for _ in range(n_tokens)]).astype(np.int32)
    check(dev.mul_mat_id(wt, experts, x, ids), orc.mul_mat_id(wt, experts, x, ids, want=("sum_abs",)), "few pairs")


# ---- few output tiles of block-32 rows: waves that share the K of a tile.  (K, N, n): one chunk of 256 values; chunks that start early (10, 14 and 30
# blocks); one row, one row more than a tile, 19 tokens and two tiles of tokens; more rows than a turn of workgroups; K over two workgroups too ----
@pytest.mark.parametrize("K,N,n", [(256, 33, 49), (320, 31, 64), (448, 1, 48), (960, 65, 33), (960, 2100, 50), (2112, 97, 19), (4096, 4100, 33), (4096, 40, 66)])
@pytest.mark.parametrize("wt", (O.Q4_0, O.Q8_0, O.Q5_0, O.IQ4_NL, O.Q4_1, O.Q5_1), ids=lambda t: O.TYPE_NAMES[t])
def test_block32_few_tiles(dev, orc, wt, K, N, n):
    rng = np.random.default_rng(K + N + wt)
    w = np.tile(orc.quantize_weights(wt, common.weights_f32(K + N, min(N, 150), K)), (-(-N // 150), 1))[:N]
    x = common.activations_f32(K + n, n, K)
    x[2] *= 2e-3                                  # scales that are subnormal in fp16, and below its smallest
    x[3] *= 1e-9
    x[5] = -np.abs(x[5])
    if K == 2112:
        assert mul_mat_launches(dev, wt, w, x) == 2          # the walk would split K and add the slices
    y = dev.mul_mat(wt, w, x)
    rows = np.unique(np.concatenate([[0, N - 1], rng.choice(N, min(N, 100), replace=False)]))
    check(y[:, rows], orc.mul_mat(wt, w[rows], x, nthreads=8, want=("sum_abs",)), "few tiles")
