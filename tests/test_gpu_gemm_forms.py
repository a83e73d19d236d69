"""The forward's products in the forms the model launches them: a training
step's fp32 matrix instructions (128 x 128 and 64 x 64 tiles, K splits, the
balanced last wave, residual + LayerNorm), the rollout's gelu-only epilogue in
every kernel and reduce that can apply it, and non-finite operands in the
kernels whose rerun is their own.

Tolerance of the fp32 instructions: one rounding of 2^-24 per two k (random
signs) and the final ones, relative L2 <= 2^-24 (2 + sqrt(K / 2)) against
float64; of the split's, the smaller bound of its own tests.
"""
import math

import pytest
import torch

from conftest import rel_l2
from ptcg_amd import native

pytestmark = pytest.mark.gpu
ROLLOUT, TRAIN, BF16, BS = range(4)
REG, F32, SPLIT, SMALL, KSPLIT = range(5)
WS = 32 << 20


def P(t):
    return None if t is None else t.data_ptr()


def path(M, N, K, rows_dev=0, ws=1, train=0):
    return native.lib().ptcg_kernel_gemm_path(M, N, K, K, 0, K, 0, rows_dev, ws, train)


def rand(*shape, seed=0, dtype=torch.float32):
    return torch.randn(*shape, device="cuda", generator=torch.Generator("cuda").manual_seed(seed)).to(dtype)


def fwd(form, A, B, epi=0, bias=None, R=None, ws_floats=WS, rows=None):
    """(C, C2) of the entry; rows: a device row count."""
    M, K = A.shape
    N = B.shape[0]
    ot = torch.bfloat16 if form == BS and epi != 3 else torch.float32
    C, C2 = (torch.full((M, N), 7.0, device="cuda", dtype=ot) for _ in range(2))
    ws = torch.zeros(ws_floats, device="cuda") if ws_floats else None
    nd = None if rows is None else torch.tensor([rows], dtype=torch.int32, device="cuda")
    native.check(native.lib().ptcg_kernel_gemm_fwd(form, M, N, K, P(A), K, P(B), K, P(C), N, epi, P(bias), P(R), N,
                                                   P(C2), N, P(nd), P(ws), ws_floats, None))
    torch.cuda.synchronize()
    return C, C2


# 64-tile kernel (fewer and more stages than its pipeline, K splits), 128-tile
# kernel with a partial last wave, operands off the 128-bit rules
TRAIN_SHAPES = [(1, 4, 4, SMALL), (63, 64, 12, SMALL), (65, 68, 132, SMALL), (100, 132, 1028, SMALL),
                (1200, 256, 256, SMALL), (2000, 256, 1024, SMALL), (5100, 256, 1024, F32), (37391, 132, 4, F32),
                (37391, 128, 20, F32), (33100, 132, 256, F32), (33100, 260, 44, F32), (300, 60, 127, REG)]


@pytest.mark.parametrize("ws_floats", [0, WS])
@pytest.mark.parametrize("M,N,K,kernel", TRAIN_SHAPES)
def test_training_products(M, N, K, kernel, ws_floats, cuda):
    if ws_floats:
        assert path(M, N, K, train=1) == kernel
    A, B, bias, R = rand(M, K, seed=1), rand(N, K, seed=2), rand(N, seed=3), rand(M, N, seed=4)
    acc = A.double() @ B.double().T
    tol = 2.0 ** -24 * (2 + math.sqrt(K / 2))
    for epi, ref in ((0, acc), (1, acc + bias.double()), (3, acc + bias.double() + R.double())):
        C, _ = fwd(TRAIN, A, B, epi, bias, R, ws_floats)
        assert rel_l2(C.cpu(), ref.cpu()) < tol, epi


# device row counts below, at and above whole waves of 128-row tiles: the
# balanced last wave (bounds of one to eight tiles per CU) in both forms
@pytest.mark.parametrize("form", [ROLLOUT, TRAIN])
@pytest.mark.parametrize("M,rows,N,K", [(40000, 1, 256, 256), (40000, 32768, 256, 256), (40000, 37391, 256, 256),
                                        (40000, 40000, 256, 128), (80000, 50001, 256, 1028), (600, 333, 256, 256)])
def test_device_row_counts(form, M, rows, N, K, cuda):
    A, B, bias, R = rand(M, K, seed=1), rand(N, K, seed=2), rand(N, seed=3), rand(M, N, seed=4)
    ref = A[:rows].double() @ B.double().T + bias.double()
    tol = 2.0 ** -24 * (2 + math.sqrt(K / (2 if form == TRAIN else 16)))
    for epi, r in ((1, ref), (3, ref + R[:rows].double())):
        C, _ = fwd(form, A, B, epi, bias, R, rows=rows)
        assert rel_l2(C[:rows].cpu(), r.cpu()) < tol
        assert bool((C[rows:] == 7.0).all())


@pytest.mark.parametrize("rows,K", [(1, 16), (31, 32), (33, 256), (200, 112), (8192, 64), (8193, 64), (20001, 256)])
def test_training_resid_ln_equals_product_then_ln(rows, K, cuda):
    """Two and six stages in flight (above and up to one 32-row tile per CU):
    the training product's and the LayerNorm's bits; rows past a device count
    are left alone."""
    L = native.lib()
    A, W, bias, R = rand(rows, K, seed=1), rand(256, K, seed=2), rand(256, seed=3), rand(rows, 256, seed=4)
    lw, lb = rand(256, seed=5), rand(256, seed=6)
    C2, _ = fwd(TRAIN, A, W, 3, bias, R, ws_floats=0)
    y2, mu2, rs2 = (torch.zeros(s, device="cuda") for s in ((rows, 256), (rows,), (rows,)))
    native.check(L.ptcg_kernel_layernorm_fwd(P(C2), P(lw), P(lb), P(y2), P(mu2), P(rs2), rows, 256, None))
    assert rel_l2(C2.cpu(), (A.double() @ W.double().T + bias.double() + R.double()).cpu()) < \
        2.0 ** -24 * (2 + math.sqrt(K / 2))
    for cut in (None, (rows + 1) // 2):
        C, y = (torch.full((rows, 256), 7.0, device="cuda") for _ in range(2))
        mu, rs = (torch.full((rows,), 7.0, device="cuda") for _ in range(2))
        nd = None if cut is None else torch.tensor([cut], dtype=torch.int32, device="cuda")
        native.check(L.ptcg_kernel_gemm_resid_ln_train(rows, K, P(A), P(W), P(bias), P(R), P(C), P(lw), P(lb), P(y),
                                                       P(mu), P(rs), P(nd), None))
        torch.cuda.synchronize()
        n = cut or rows
        for a, b in ((C, C2), (y, y2), (mu, mu2), (rs, rs2)):
            assert torch.equal(a[:n], b[:n]) and bool((a[n:] == 7.0).all())


# kernel: split at K splits, 64- and 32-row tiles, whole tiles, a balanced last
# wave, the register-staged and scalar-load kernel, odd edges in each
GELU_SHAPES = [(100, 132, 9000), (1000, 132, 2052), (33, 36, 20), (300, 62, 664), (23001, 130, 64), (33100, 132, 256),
               (70000, 128, 20), (300, 61, 127)]


@pytest.mark.parametrize("form", [ROLLOUT, TRAIN, BF16])
@pytest.mark.parametrize("M,N,K", GELU_SHAPES)
def test_gelu_epilogue(form, M, N, K, cuda):
    """gelu alone is the gelu of the pair (gelu', gelu), bit for bit, in every
    kernel and reduce; the pair is checked against float64 elsewhere and here."""
    A, B, bias = rand(M, K, seed=1), rand(N, K, seed=2) / math.sqrt(K), rand(N, seed=3)
    for ws_floats in (0, WS):
        _, pair = fwd(form, A, B, 6, bias, ws_floats=ws_floats)
        C, untouched = fwd(form, A, B, 9, bias, ws_floats=ws_floats)
        assert torch.equal(C, pair) and bool((untouched == 7.0).all())
    # the erf approximation's 1.5e-7 on values of order 1, and the product's own error
    a, b = (A.bfloat16(), B.bfloat16()) if form == BF16 and K % 4 == 0 else (A, B)
    ref = torch.nn.functional.gelu(a.double() @ b.double().T + bias.double())
    assert rel_l2(C.cpu(), ref.cpu()) < 1.5e-7 + 2.0 ** -24 * (4 + math.sqrt(K / 2))


@pytest.mark.parametrize("form", [ROLLOUT, TRAIN])
@pytest.mark.parametrize("M,rows,N,K", [(600, 333, 256, 256), (40000, 37391, 256, 256), (40000, 20001, 132, 256)])
def test_gelu_epilogue_device_rows(form, M, rows, N, K, cuda):
    A, B, bias = rand(M, K, seed=1), rand(N, K, seed=2) / math.sqrt(K), rand(N, seed=3)
    _, pair = fwd(form, A, B, 6, bias, rows=rows)
    C, _ = fwd(form, A, B, 9, bias, rows=rows)
    assert torch.equal(C[:rows], pair[:rows]) and bool((C[rows:] == 7.0).all())


@pytest.mark.parametrize("M,N,K", [(1, 8, 8), (130, 132, 72), (33100, 132, 256)])
def test_gelu_epilogue_bf16_storage(M, N, K, cuda):
    A, B, bias = rand(M, K, seed=1, dtype=torch.bfloat16), rand(N, K, seed=2, dtype=torch.bfloat16), rand(N, seed=3)
    _, pair = fwd(BS, A, B, 6, bias)
    C, _ = fwd(BS, A, B, 9, bias)
    assert torch.equal(C, pair)
    ref = torch.nn.functional.gelu(A.double() @ B.double().T + bias.double())
    assert rel_l2(C.double().cpu(), ref.cpu()) < 2.0 ** -8   # the stored value's rounding


def same_nonfinite(C, ref, tol):
    assert torch.equal(torch.isnan(C), torch.isnan(ref)) and torch.equal(torch.isinf(C), torch.isinf(ref))
    inf, ok = torch.isinf(ref), torch.isfinite(ref)
    assert torch.equal(C[inf], ref[inf]) and rel_l2(C[ok].cpu(), ref[ok].double().cpu()) < tol


# 32-row tiles (split at the fragment reads) and 64-row ones (split while staged)
@pytest.mark.parametrize("rows", [96, 8229])
def test_resid_ln_nonfinite(rows, cuda):
    L, K = native.lib(), 80
    A, W, bias, R = rand(rows, K, seed=1), rand(256, K, seed=2), rand(256, seed=3), rand(rows, 256, seed=4)
    A, W = A + torch.where(A < 0, -0.1, 0.1), W + torch.where(W < 0, -0.1, 0.1)
    A[3, 5], A[50, 9], A[rows - 1, 70], W[200, 11] = math.inf, math.nan, -math.inf, math.inf
    lw, lb = rand(256, seed=5), rand(256, seed=6)
    C, y = (torch.zeros(rows, 256, device="cuda") for _ in range(2))
    mu, rs = (torch.zeros(rows, device="cuda") for _ in range(2))
    native.check(L.ptcg_kernel_gemm_resid_ln(rows, K, P(A), P(W), P(bias), P(R), P(C), P(lw), P(lb), P(y), P(mu), P(rs),
                                             0, None, None))
    torch.cuda.synchronize()
    ref = (A.double() @ W.double().T + bias.double() + R.double()).float()
    same_nonfinite(C, ref, 2.0 ** -24 * (3 + math.sqrt(K / 2)))   # rerun on fp32 instructions


@pytest.mark.parametrize("M,rows,N,K", [(40000, 37391, 256, 256), (600, 333, 256, 256)])
def test_device_rows_nonfinite(M, rows, N, K, cuda):
    """The balanced last wave (whole tiles and tail partials) and the K split
    over waves: an inf in a whole tile, a NaN in the last rows."""
    A, B, bias = rand(M, K, seed=1), rand(N, K, seed=2), rand(N, seed=3)
    A, B = A + torch.where(A < 0, -0.1, 0.1), B + torch.where(B < 0, -0.1, 0.1)
    A[3, 5], A[rows - 1, 250], A[rows - 70, 130], B[201, 100] = math.inf, math.nan, -math.inf, -math.inf
    C, _ = fwd(ROLLOUT, A, B, 1, bias, rows=rows)
    ref = (A[:rows].double() @ B.double().T + bias.double()).float()
    same_nonfinite(C[:rows], ref, 2.0 ** -24 * (3 + math.sqrt(K / 2)))
    assert bool((C[rows:] == 7.0).all())


@pytest.mark.parametrize("args,match", [((4, 64, 64, 64, 1), "form"), ((0, 64, 64, 64, 8), "epilogue"),
                                        ((1, 64, 64, 64, 10), "epilogue"), ((0, 64, 64, 64, 9), "bias")])
def test_refused(args, match):
    form, M, N, K, epi = args
    with pytest.raises(native.PtcgError, match=match):
        native.check(native.lib().ptcg_kernel_gemm_fwd(form, M, N, K, 1 << 20, K, 1 << 20, K, 1 << 20, N, epi, None,
                                                       None, N, None, N, None, None, 0, None))
