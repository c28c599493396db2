"""Which kernels a call takes: the launches of a call are counted as the nodes of a graph that records it."""
import ctypes as C

import numpy as np
import pytest

import common
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    import cactus_amd
    return cactus_amd.Device(0)


class NodeParams(C.Structure):
    _fields_ = [("block", C.c_uint * 3), ("extra", C.c_void_p), ("func", C.c_void_p), ("grid", C.c_uint * 3), ("params", C.c_void_p), ("shared", C.c_uint)]


def kernels(dev, call):
    """Names (mangled) of the kernels of call(stream), which is made once before it is recorded (a kernel's first launch raises its LDS limit)."""
    hip = C.CDLL("libamdhip64.so")
    hip.hipKernelNameRefByPtr.restype = C.c_char_p
    st, graph, count = C.c_void_p(), C.c_void_p(), C.c_size_t()
    dev.check(dev.lib.chip_stream_create(C.byref(st)))
    dev.check(call(st))
    dev.sync(st)
    assert hip.hipStreamBeginCapture(st, 0) == 0
    rc = call(st)
    assert hip.hipStreamEndCapture(st, C.byref(graph)) == 0 and rc == 0
    assert hip.hipGraphGetNodes(graph, None, C.byref(count)) == 0
    nodes, names = (C.c_void_p * count.value)(), []
    assert hip.hipGraphGetNodes(graph, nodes, C.byref(count)) == 0
    for node in nodes:
        p = NodeParams()
        assert hip.hipGraphKernelNodeGetParams(C.c_void_p(node), C.byref(p)) == 0
        names.append(hip.hipKernelNameRefByPtr(C.c_void_p(p.func), st).decode())
    hip.hipGraphDestroy(graph)
    dev.check(dev.lib.chip_stream_destroy(st))
    return names


def launches(dev, call):
    return len(kernels(dev, call))


def mul_mat_id_launches(dev, wt, K, N, n_as, n_used, n_tokens):
    """Of an expert matmul: 3 (quantizer, grouping, GEMM) where its pairs are grouped, fewer where each is a GEMV."""
    L, row = dev.lib, dev.row_size(wt, K)
    rng = np.random.default_rng(K + N)
    dW = dev.alloc(n_as * N * row)
    dev.check(L.chip_memset(dW.ptr, 0, n_as * N * row, None))
    dx = dev.to_device(common.activations_f32(K, n_tokens, K))
    ids = dev.to_device(np.stack([rng.permutation(n_as)[:n_used] for _ in range(n_tokens)]).astype(np.int32))
    dy = dev.alloc(n_tokens * n_used * N * 4)
    wsz = L.chip_mul_mat_id_workspace_size(wt, K, n_as, n_used, n_tokens, 1)
    ws = dev.alloc(wsz)
    return launches(dev, lambda st: L.chip_mul_mat_id(wt, dW.ptr, row, N * row, K, N, n_as, dx.ptr, K, 1, ids.ptr, n_used, n_used, n_tokens,
                                                      dy.ptr, N, ws.ptr, wsz, st))


def group_kernels(dev, members, K, n):
    """Of chip_mul_mat_group over members [(type, rows), ...]."""
    import cactus_amd as ca
    L = dev.lib
    arr, keep, wsz = (ca.Mat * len(members))(), [dev.to_device(common.activations_f32(K, n, K))], 0
    for i, (wt, N) in enumerate(members):
        row = dev.row_size(wt, K)
        dW, dy = dev.alloc(N * row), dev.alloc(n * N * 4)
        dev.check(L.chip_memset(dW.ptr, 0, N * row, None))
        keep += [dW, dy]
        arr[i] = ca.Mat(wt, dW.ptr, row, N, dy.ptr, N, None, 0)
        wsz = max(wsz, L.chip_mul_mat_workspace_size_n(wt, K, N, n))
    ws = dev.alloc(wsz)
    return kernels(dev, lambda st: L.chip_mul_mat_group(arr, len(members), K, keep[0].ptr, K, n, ws.ptr, wsz, st))


def group_launches(dev, members, K, n):
    return len(group_kernels(dev, members, K, n))


def mul_mat_kernels(dev, wt, W, x, split_k=True):
    n, K = x.shape
    N, L = W.shape[0], dev.lib
    dW, dx, dy = dev.to_device(W), dev.to_device(x), dev.alloc(n * N * 4)
    wsz = L.chip_mul_mat_workspace_size_n(wt, K, N, n) if split_k else L.chip_mul_mat_workspace_size(wt, K, n)
    ws = dev.alloc(wsz)
    return kernels(dev, lambda st: L.chip_mul_mat(wt, dW.ptr, W.shape[1], K, N, dx.ptr, K, n, dy.ptr, N, ws.ptr, wsz, st))


def mul_mat_launches(dev, wt, W, x, split_k=True):
    return len(mul_mat_kernels(dev, wt, W, x, split_k))


# quantizer, GEMM over slices of K, slice sum; rows in fours, and one, two and three rows in a token's last group
@pytest.mark.parametrize("N", (300, 301, 302, 303, 3))
@pytest.mark.parametrize("wt", (O.Q3_K, O.Q4_K, O.Q8_0), ids=lambda t: O.TYPE_NAMES[t])
def test_split_k_takes_three_launches_whatever_the_rows(dev, orc, wt, N):
    K, n = 4096, 70
    wq = orc.quantize_weights(wt, common.weights_f32(K + N, N, K))
    x = common.activations_f32(K + n, n, K)
    assert mul_mat_launches(dev, wt, wq, x) == 3
    ref = orc.mul_mat(wt, wq, x, nthreads=8, want=("sum_abs",))
    err = np.abs(dev.mul_mat(wt, wq, x).astype(np.float64) - ref["y"].astype(np.float64))
    assert (err <= 1e-5 * ref["sum_abs"]).all()


# A GEMV per pair is two launches (quantizer, GEMV), the expert groups three (quantizer, grouping, GEMM).  Measured on either side of
# the rule: few pairs an expert, many pairs, and short rows, where the GEMM is ahead with a pair an expert
@pytest.mark.parametrize("wt", (O.Q3_K, O.Q2_K, O.IQ4_XS), ids=lambda t: O.TYPE_NAMES[t])
@pytest.mark.parametrize("K,N,n_as,n_used,n_tokens,gemm", [(2048, 768, 128, 8, 8, False), (1024, 256, 64, 2, 32, False), (2048, 768, 128, 8, 192, True),
                                                           (512, 2048, 32, 4, 100, True), (1024, 256, 8, 8, 40, True), (512, 70, 5, 2, 90, False), (512, 70, 5, 2, 700, True)])
def test_low_bit_expert_matmul_takes_the_gemm_where_it_is_ahead(dev, wt, K, N, n_as, n_used, n_tokens, gemm):
    assert mul_mat_id_launches(dev, wt, K, N, n_as, n_used, n_tokens) == (3 if gemm else 2)


# us, GEMV / GEMM: 69 / 38, 172 / 104, 30 / 45, 71 / 96, 23 / 28, 11 / 13, 17 / 26, 105 / 69, 63 / 70, 29 / 36, 26 / 33; F16 below and from 64 pairs on
@pytest.mark.parametrize("wt,K,N,n_as,n_used,n_tokens,gemm", [
    (O.Q8_0, 3072, 1024, 32, 4, 39, True), (O.Q8_0, 3584, 768, 128, 2, 225, True), (O.Q8_0, 1024, 3676, 28, 8, 4, False),
    (O.Q4_0, 2560, 12214, 12, 8, 4, False), (O.Q5_K, 1536, 3328, 32, 8, 2, False), (O.Q4_K, 512, 2048, 8, 4, 4, False),
    (O.Q4_K, 2048, 768, 128, 8, 8, False), (O.Q4_K, 4096, 14336, 8, 2, 16, True), (O.Q4_K, 4096, 14336, 8, 2, 8, False),
    (O.Q8_0, 2048, 3584, 8, 4, 8, False), (O.IQ4_XS, 3072, 106, 12, 1, 506, False),
    (O.F16, 512, 300, 8, 3, 21, False), (O.F16, 512, 300, 8, 4, 16, True)])
def test_expert_matmul_takes_the_gemm_where_it_is_ahead(dev, wt, K, N, n_as, n_used, n_tokens, gemm):
    assert (mul_mat_id_launches(dev, wt, K, N, n_as, n_used, n_tokens) == 3) == gemm


# long rows with a short last stage, no room to split K: quantizer and six GEMV passes while they are ahead of the GEMM's walk
@pytest.mark.parametrize("wt,n,count", [(O.Q5_0, 48, 7), (O.Q4_1, 48, 7), (O.Q5_1, 48, 7), (O.IQ4_NL, 48, 7), (O.Q5_0, 65, 2), (O.IQ4_NL, 57, 2), (O.Q8_0, 57, 2)])
def test_unsplit_short_last_stage_takes_the_gemm_where_it_is_ahead(dev, orc, wt, n, count):
    wq = orc.quantize_weights(wt, common.weights_f32(5, 64, 8256))
    assert mul_mat_launches(dev, wt, wq, common.activations_f32(6, n, 8256), split_k=False) == count


# 300 to 330 tiles of long rows (us, walk in slices of K / tiles shared by waves: 32.9 / 36.6, 34.7 / 38.0, 19.3 / 21.9), and fewer; 564 tiles of rows
# that are long for two waves (47.5 / 56.5)
@pytest.mark.parametrize("wt,K,N,n,walk", [(O.Q5_0, 9600, 1288, 254, True), (O.IQ4_NL, 9600, 401, 732, True), (O.Q8_0, 4352, 4828, 35, True),
                                           (O.Q8_0, 2176, 4828, 35, False), (O.Q5_0, 1920, 1288, 254, False), (O.Q5_1, 9984, 6009, 89, True),
                                           (O.Q4_0, 4352, 2736, 243, False), (O.IQ4_NL, 4352, 2736, 243, True)])
def test_block32_products_that_half_fill_the_device_stay_in_the_walk(dev, wt, K, N, n, walk):
    names = mul_mat_kernels(dev, wt, np.zeros((N, dev.row_size(wt, K)), np.uint8), common.activations_f32(1, n, K))
    assert len(names) == (3 if walk else 2) and ("gemm_blk32_kernel" if walk else "gemm_blk32_few_kernel") in names[1]


# a tile of 64 tokens reads the rows once, two of 32 twice: Q8_0 by two waves (us, walk / tiles shared by waves: 9.1 / 10.1)
@pytest.mark.parametrize("wt,n,walk", [(O.Q8_0, 46, True), (O.Q8_0, 33, True), (O.Q8_0, 32, False), (O.Q4_0, 46, False)])
def test_block32_products_of_two_token_tiles(dev, wt, n, walk):
    names = mul_mat_kernels(dev, wt, np.zeros((11600, dev.row_size(wt, 768)), np.uint8), common.activations_f32(1, n, 768))
    assert len(names) == 2 and ("gemm_blk32_kernel" if walk else "gemm_blk32_few_kernel") in names[1]


# Q6_K and Q3_K above 32 tokens by the workgroups that the staging kernel has, on either side of the rule and at 32 tokens (us, staging / tiles shared by
# waves: 11.6 / 13.4, 26.8 / 29.2, 11.4 / 13.5)
@pytest.mark.parametrize("wt,K,N,n,staged", [(O.Q6_K, 1024, 11884, 49, True), (O.Q6_K, 3328, 16161, 47, True), (O.Q3_K, 1536, 13500, 33, True), (O.Q6_K, 1024, 10880, 49, False),
                                             (O.Q6_K, 1024, 10881, 49, True), (O.Q3_K, 2048, 12224, 40, False), (O.Q3_K, 2048, 12225, 40, True), (O.Q3_K, 1536, 13500, 32, False)])
def test_kquant_products_that_fill_the_staging_kernel_stay_there(dev, wt, K, N, n, staged):
    names = mul_mat_kernels(dev, wt, np.zeros((N, dev.row_size(wt, K)), np.uint8), common.activations_f32(1, n, K))
    assert len(names) == 2 and ("gemm_kq_kernel" if staged else "gemm_kq_few_kernel") in names[1]


# more 32 x 32 tiles than a device full of two-wave workgroups (us, walk / tiles shared by waves: 274 / 337)
def test_block32_products_of_many_tiles_stay_in_the_walk(dev):
    names = mul_mat_kernels(dev, O.Q8_0, np.zeros((7543, dev.row_size(O.Q8_0, 7168)), np.uint8), common.activations_f32(1, 1042, 7168))
    assert len(names) == 2 and "gemm_blk32_kernel" in names[1]


# kqv of more than 128 columns per KV head: one launch of the GEMM with the 256 bytes it asks for, the same bits whatever lies behind
# them, and nothing written there; one launch of the dot-product kernel without a workspace
@pytest.mark.parametrize("hd,nh,nkv,n,kv", [(128, 8, 2, 70, 264), (64, 6, 3, 133, 1064), (256, 4, 1, 65, 520), (96, 8, 4, 80, 136)])
def test_kqv_of_a_prompt_with_a_small_workspace(dev, orc, hd, nh, nkv, n, kv):
    L, rng = dev.lib, np.random.default_rng(hd + n + kv)
    vt = rng.standard_normal((nkv, hd, kv)).astype(np.float16)
    p = rng.random((nh, n, kv)).astype(np.float32)
    ref = orc.mul_mat_f16_batched(vt, p, want=("sum_abs",))
    dv, dp, dy = dev.to_device(vt), dev.to_device(p), dev.alloc(nh * n * hd * 4)
    outs = []
    for wsz in (0, 256, nh * n * kv * 2 + 4096):
        ws = dev.to_device(np.full(max(wsz, 16), 0x5A, np.uint8))
        assert launches(dev, lambda st: L.chip_mul_mat_f16_batched(dv.ptr, 2 * kv, 2 * kv * hd, kv, hd, nkv, dp.ptr, kv, kv * n, n, nh, dy.ptr,
                                                                   hd, hd * n, ws.ptr if wsz else None, wsz, st)) == 1
        y = dy.download(np.float32, nh * n * hd).reshape(nh, n, hd)
        assert (np.abs(y - ref["y"]) <= 1e-5 * ref["sum_abs"]).all()
        assert (ws.download(np.uint8, max(wsz, 16)) == 0x5A).all()
        outs.append(y)
    assert outs[1].tobytes() == outs[2].tobytes()
    assert outs[0].tobytes() != outs[1].tobytes()
