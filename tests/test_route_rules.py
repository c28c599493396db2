"""CPU-only: which kernels a shape is sent to, as the workspace size queries show it (256 compute units where no device is present)."""
import pytest

import cactus_amd as ca


@pytest.fixture(scope="module")
def lib():
    return ca.load_library()


def splits_k(lib, t, K, N, n):
    return lib.chip_mul_mat_workspace_size_n(t, K, N, n) > lib.chip_mul_mat_workspace_size(t, K, n)


# On either side of the rule (us, GEMV passes / GEMM): the low-bit types take the GEMM, with K split, where it is estimated to be ahead.  The estimate
# is late for Q2_K and IQ4_XS: some of their GEMV cases here are faster through the GEMM by now
@pytest.mark.parametrize("t,K,N,n,gemm", [
    (ca.IQ4_XS, 4096, 1024, 10, False), (ca.IQ4_XS, 8192, 8192, 12, False), (ca.IQ4_XS, 2048, 692, 9, False),        # 12 / 13, 37 / 27, 11 / 11
    (ca.IQ4_XS, 14336, 1024, 12, True), (ca.IQ4_XS, 4096, 4096, 17, True),                                           # 22 / 17, 24 / 15
    (ca.Q3_K, 2816, 300, 10, False), (ca.Q3_K, 3840, 612, 9, False), (ca.Q3_K, 4096, 4096, 9, True), (ca.Q3_K, 14336, 1024, 9, True),    # 11 / 14, 12 / 14, 15 / 14, 19 / 14
    (ca.Q3_K, 14336, 70, 9, True), (ca.Q2_K, 14336, 70, 9, True), (ca.IQ4_XS, 14336, 70, 9, True),                              # 18 / 13, 18 / 12, 18 / 16
    (ca.Q2_K, 2304, 280, 11, False), (ca.Q2_K, 4096, 1024, 10, False), (ca.Q2_K, 4096, 4096, 12, True)])                          # 12 / 11, 12 / 11, 17 / 12
def test_low_bit_types_take_the_gemm_where_it_is_ahead(lib, t, K, N, n, gemm):
    assert splits_k(lib, t, K, N, n) == gemm
    assert splits_k(lib, t, K, N, 70)
    assert not splits_k(lib, t, K, N, 8)


# the third GEMV pass over one or two tokens against the GEMM (us: 14.7 / 17.4, 15.8 / 18.4, 15.2 / 16.2; 20 / 16, 22 / 15, 17 / 16)
@pytest.mark.parametrize("t,K,N,n,gemm", [(ca.Q4_1, 2624, 320, 17, False), (ca.Q5_0, 3648, 960, 17, False), (ca.Q5_1, 3264, 192, 18, False),
                                          (ca.Q5_1, 4160, 320, 17, True), (ca.Q4_0, 2112, 2560, 18, True), (ca.Q4_0, 2624, 960, 17, True),
                                          (ca.Q4_1, 2624, 320, 19, True), (ca.Q4_1, 2560, 320, 17, True)])
def test_short_last_stage_takes_the_gemm_where_it_is_ahead(lib, t, K, N, n, gemm):
    assert splits_k(lib, t, K, N, n) == gemm


def test_rows_too_long_for_the_gemv_stay_accepted(lib):
    """K = 2^18: no token's activations fit a workgroup's local memory, so only the GEMM can run it."""
    for t in (ca.Q3_K, ca.Q2_K, ca.IQ4_XS):
        assert splits_k(lib, t, 1 << 18, 64, 9)


def test_attention_grids_stay_below_the_launch_limit(lib):
    """kq through the GEMM needs room for fp16 activations; a grid of 2^32 threads or more cannot be launched and is not planned."""
    size = lib.chip_mul_mat_f16_batched_workspace_size
    assert size(64, 1 << 20, 8, 8, 100) == 800 * 128
    assert size(64, 1 << 28, 8, 8, 100) == 0                   # 8 x 2 x 2^22 workgroups of 256 threads
    assert size(64, 1 << 24, 8, 8, 1024) == 8192 * 128         # 8 x 8 x 2^17 of the larger tiles


def test_kqv_of_a_prompt_asks_for_no_copy(lib):
    """Its GEMM reads the fp32 probabilities; up to 128 pairs per KV head the split-K kernels still want room for partial outputs."""
    size = lib.chip_mul_mat_f16_batched_workspace_size
    assert size(4096, 128, 8, 32, 512) == 256 and size(4096, 256, 2, 8, 2048) == 256
    assert size(4096, 128, 8, 32, 32) > 256 and size(128, 4096, 8, 32, 512) == 8 * 2048 * 256
