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
