"""Host-side rules of the GEMM entry points: what they refuse and which kernel
they pick.  No GPU: every call here ends before a launch."""
import pytest

from ptcg_amd import native

PTR = 1 << 20   # a 16 B aligned address that nothing dereferences


@pytest.mark.parametrize("epi", [-1, 8, 9, 10])
@pytest.mark.parametrize("out_bf16", [0, 1])
def test_bs_refuses_internal_epilogues(epi, out_bf16):
    """The bf16-operand entry takes the documented epilogues only; 9 (gelu
    alone, a rollout's) would read a bias the entry does not require."""
    with pytest.raises(native.PtcgError, match="epilogue"):
        native.check(native.lib().ptcg_kernel_gemm_bs(64, 64, 64, PTR, 64, PTR, 64, PTR, 64, epi, out_bf16, None, None,
                                                      64, None, 64, None))


REG, F32, SPLIT, SMALL, KSPLIT = range(5)


def path(M, N, K, lda=None, a_t=0, ldb=None, b_t=0, rows_dev=0, ws=1, train=0):
    return native.lib().ptcg_kernel_gemm_path(M, N, K, lda or (M if a_t else K), a_t, ldb or (N if b_t else K), b_t,
                                              rows_dev, ws, train)


@pytest.mark.parametrize("M,N,K", [(4, 4, 1500000), (16, 64, 1200000), (300, 4, 900000)])
@pytest.mark.parametrize("ws", [0, 1])
def test_long_rows_stay_on_the_dma_kernels(M, N, K, ws):
    """k-contiguous operands within the 2^31-byte rules of the DMA kernels
    (tile rows past the end counted) never fall to the register-staged one."""
    assert (max(M, N) + 256) * K + K + 256 < 1 << 29
    assert path(M, N, K, ws=ws) in (SPLIT, SMALL, KSPLIT)
    assert path(M, N, K, ws=ws, train=1) in (F32, SMALL)


def test_rows_past_2_31_bytes_run_the_split():
    assert path(525000, 64, 1024) == SPLIT
    assert path(525000, 64, 1024, train=1) == REG
    assert path(128, 128, 1 << 23) == REG


@pytest.mark.parametrize("a_t,b_t", [(0, 0), (0, 1), (1, 1), (1, 0)])
def test_operands_off_the_128_bit_rules(a_t, b_t):
    M, N, K = (127, 64, 64) if a_t else (64, 64, 127)
    assert path(M, N, K, a_t=a_t, b_t=b_t) == REG
    assert path(64, 64, 64, lda=65, a_t=a_t, b_t=b_t) == REG
    assert path(64, 64, 64, a_t=a_t, b_t=b_t) != REG


@pytest.mark.parametrize("M,N", [(4, 4), (36, 128), (300, 256), (2000, 256)])
@pytest.mark.parametrize("b_t", [0, 1])
def test_long_k_is_split_over_the_chip(M, N, b_t):
    """K over one workgroup's waves ends where the chain of a wave's stages
    (K / 128) costs more than K splits over the chip and their reduce; a
    device row count has no K splits."""
    for K in (256, 1024, 2048):
        assert path(M, N, K, b_t=b_t) == KSPLIT
    for K in (2052, 4096, 16384, 1 << 20):
        assert path(M, N, K, b_t=b_t) in (SMALL, SPLIT)
    assert path(M, N, 4096, b_t=b_t, rows_dev=1) == (KSPLIT if M < 2000 else SMALL)


@pytest.mark.parametrize("M,N", [(65540, 128), (16400, 512), (9000, 1024)])   # 513..568 tiles on 256 CUs
def test_short_k_on_wide_grids_runs_on_fp32_instructions(M, N):
    """A few k stages past the split's two workgroups per CU."""
    for a_t, b_t in ((0, 0), (0, 1), (1, 1), (1, 0)):
        for K in (4, 16, 20, 48):
            assert path(M, N, K, a_t=a_t, b_t=b_t) == F32
        assert path(M, N, 68, a_t=a_t, b_t=b_t) in (SPLIT, SMALL)
    assert path(M, N, 16, rows_dev=1) == F32
    assert path(60000, 128, 16) == SPLIT          # 469 tiles: one round of workgroups
    assert path(200000, 64, 48) == SPLIT          # 1 563 tiles
    assert path(200000, 64, 48, a_t=1, b_t=1) == SPLIT and path(200000, 64, 32, a_t=1, b_t=1) == F32
