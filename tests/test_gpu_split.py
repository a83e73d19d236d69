"""fp32 products on the bf16 matrix pipe (three-way split of the operands):
tile and k edges of the 128 x 128, 64 x 64 and 32 x 32 kernels, non-finite, extreme
and tiny operands, operands past 2^31 bytes, and the residual + LayerNorm forms.

Tolerance, relative L2 against float64: the dropped terms m l and l m are at
most 2^-25 of a product each, with one sign at worst (2^-24); the accumulator of
the large terms is rounded once per 16 k (2^-24 each, random signs), the small
terms' roundings are 2^-8 of those, and the two are added once (2^-24): 2^-24 (2
+ sqrt(K / 16)).  Split-K partials are summed in fp32, one more rounding per
split (at most K / 16 in all, counted above).
"""
import math

import pytest
import torch

from conftest import rel_l2
from ptcg_amd import native

pytestmark = pytest.mark.gpu


def bound(K):
    return 2.0 ** -24 * (2 + math.sqrt(K / 16))


def P(t):
    return None if t is None else t.data_ptr()


def gemm(A, B, M, N, K, a_t, b_t, epi=0, bias=None, R=None, ws_floats=32 << 20):
    """ws_floats 0: no workspace, so no K split of any kind."""
    dA, dB = A.cuda().contiguous(), B.cuda().contiguous()
    C, ws = torch.zeros(M, N, device="cuda"), torch.zeros(ws_floats, device="cuda")
    native.check(native.lib().ptcg_kernel_gemm(M, N, K, P(dA), M if a_t else K, a_t, P(dB), N if b_t else K, b_t, P(C),
                                               N, epi, P(bias), P(R), N, None, N, P(ws) if ws_floats else None, ws_floats,
                                               None))
    torch.cuda.synchronize()
    return C


def operands(M, N, K, a_t, b_t, seed=0):
    g = torch.Generator().manual_seed(seed + M * 7 + N * 3 + K)
    A, B = torch.randn(M, K, generator=g), torch.randn(K, N, generator=g)
    return A, B, (A.T if a_t else A), (B if b_t else B.T)


# 64-tile kernel: tile and k-stage edges, fewer and more stages than its
# pipeline; 128-tile kernel: the same and its balanced tail
SHAPES = [(M, N, K) for M in (4, 60, 64, 68) for N, K in ((64, 4), (68, 12), (4, 132), (132, 1028))] + \
         [(23000, 128, K) for K in (4, 16, 20, 300)] + [(33100, 132, 256), (22656, 64, 44), (128, 132, 9000)]


@pytest.mark.parametrize("a_t,b_t", [(0, 0), (0, 1), (1, 1), (1, 0)])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_edges(M, N, K, a_t, b_t, cuda):
    A, B, a, b = operands(M, N, K, a_t, b_t)
    C = gemm(a, b, M, N, K, a_t, b_t)
    ref = A.cuda().double() @ B.cuda().double()
    assert rel_l2(C.cpu(), ref.cpu()) < bound(K), rel_l2(C.cpu(), ref.cpu())


# a few k stages on wide grids: the fp32 instructions in every layout
@pytest.mark.parametrize("a_t,b_t", [(0, 0), (0, 1), (1, 1), (1, 0)])
@pytest.mark.parametrize("M,N,K", [(33000, 132, 4), (65540, 128, 16), (65540, 128, 20), (16396, 508, 48)])
def test_short_k(M, N, K, a_t, b_t, cuda):
    A, B, a, b = operands(M, N, K, a_t, b_t)
    g = torch.Generator().manual_seed(M)
    bias, R = torch.randn(N, generator=g).cuda(), torch.randn(M, N, generator=g).cuda()
    C = gemm(a, b, M, N, K, a_t, b_t, 3, bias, R)
    ref = A.cuda().double() @ B.cuda().double() + bias.double() + R.double()
    assert rel_l2(C.cpu(), ref.cpu()) < 2.0 ** -24 * (2 + math.sqrt(K / 2))   # an addition per two k


@pytest.mark.parametrize("rows", [4, 20, 64])
def test_short_weight_gradient(rows, cuda):
    """dW and its bias sums over one to four k stages, and the same over a
    device row count."""
    L, n_out, n_in = native.lib(), 33000, 132
    g = torch.Generator("cuda").manual_seed(rows)
    dY, X = (torch.randn(rows, n, device="cuda", generator=g) for n in (n_out, n_in))
    dW, db = torch.zeros(n_out, n_in, device="cuda"), torch.zeros(n_out, device="cuda")
    ws, nd = torch.zeros(32 << 20, device="cuda"), torch.tensor([rows - 3], dtype=torch.int32, device="cuda")
    for n in (rows, rows - 3):
        a = (rows, n_in, n_out, P(dY), n_out, P(X), n_in, P(dW), P(db))
        native.check(L.ptcg_kernel_gemm_dw(*a, P(ws), ws.numel(), None) if n == rows else
                     L.ptcg_kernel_gemm_dw_rows_dev(*a, P(nd), P(ws), ws.numel(), None))
        torch.cuda.synchronize()
        tol = 2.0 ** -24 * (2 + math.sqrt(rows / 2))
        assert rel_l2(dW.cpu(), (dY[:n].double().T @ X[:n].double()).cpu()) < tol
        assert rel_l2(db.cpu(), dY[:n].double().sum(0).cpu()) < 2.0 ** -24 * (2 + math.sqrt(rows))


@pytest.mark.parametrize("M,K", [(4, 4), (96, 4), (96, 16), (23000, 64), (512, 256), (512, 4096)])
@pytest.mark.parametrize("spread", [0.0, 0.5])
def test_one_sign_of_dropped_terms(M, K, spread, cuda):
    """Operands at and just below 1 + 2^-8 - 2^-17, whose dropped terms are the
    largest there are and all of one sign.  All roundings may share a sign too:
    K / 16 of them, on partial sums of half the result on average."""
    N = 128
    g = torch.Generator().manual_seed(K)
    A, B = (1 + 2.0 ** -8 - 2.0 ** -17 * (1 + spread * torch.rand(s, generator=g)) for s in ((M, K), (K, N)))
    C = gemm(A, B.T, M, N, K, 0, 0)
    ref = A.double() @ B.double()
    assert rel_l2(C.cpu(), ref) < 2.0 ** -24 * (2 + K / 32), rel_l2(C.cpu(), ref) * 2 ** 24


# the 64-tile kernel, and K over the waves of 32 x 32 tiles: row, column and k
# edges, waves with no or a partial stage, more stages than are in flight
@pytest.mark.parametrize("ws_floats", [0, 32 << 20])
@pytest.mark.parametrize("b_t", [0, 1])
@pytest.mark.parametrize("M,N,K", [(1, 4, 4), (31, 36, 20), (33, 28, 124), (65, 132, 128), (100, 256, 132),
                                   (300, 64, 664), (16, 32, 1028), (2000, 256, 960)])
def test_small_grids(M, N, K, b_t, ws_floats, cuda):
    A, B, a, b = operands(M, N, K, 0, b_t)
    g = torch.Generator().manual_seed(M)
    bias, R = torch.randn(N, generator=g).cuda(), torch.randn(M, N, generator=g).cuda()
    C = gemm(a, b, M, N, K, 0, b_t, 3, bias, R, ws_floats)
    ref = A.cuda().double() @ B.cuda().double() + bias.double() + R.double()
    assert rel_l2(C.cpu(), ref.cpu()) < bound(K), rel_l2(C.cpu(), ref.cpu())


@pytest.mark.parametrize("M,N,K,a_t,b_t", [(100, 68, 64, 0, 0), (100, 68, 64, 1, 1), (23000, 128, 64, 0, 1),
                                             (100, 68, 160, 0, 1)])
def test_nonfinite(M, N, K, a_t, b_t, cuda):
    """inf, -inf and NaN reach exactly the outputs they reach in float64
    (no other operand element is 0, and no two of them meet)."""
    A, B, _, _ = operands(M, N, K, a_t, b_t, seed=5)
    A = A + torch.where(A < 0, -0.1, 0.1)
    B = B + torch.where(B < 0, -0.1, 0.1)
    A[3, 5], A[50, 9], B[7, 2] = math.inf, math.nan, -math.inf
    C = gemm(A.T if a_t else A, B if b_t else B.T, M, N, K, a_t, b_t).cpu()
    ref = (A.double() @ B.double()).float()
    assert torch.equal(torch.isnan(C), torch.isnan(ref))
    inf = torch.isinf(ref)
    assert torch.equal(C[inf], ref[inf]) and torch.equal(torch.isfinite(C), torch.isfinite(ref))
    ok = torch.isfinite(ref)
    assert rel_l2(C[ok], (A.double() @ B.double())[ok]) < 2.0 ** -24 * (2 + math.sqrt(K / 2))   # fp32 instructions


@pytest.mark.parametrize("scale_a,scale_b", [(2.0 ** 100, 2.0 ** -90), (2.0 ** -100, 1.0), (2.0 ** -110, 2.0 ** 60),
                                             (3.3e38, 2.0 ** -40)])
def test_extremes(scale_a, scale_b, cuda):
    """Operands near the ends of the fp32 range (finite values past the
    largest bf16 among them)."""
    M, N, K = 96, 64, 64
    g = torch.Generator().manual_seed(9)
    A = (0.5 + 0.53 * torch.rand(M, K, generator=g)).clamp(max=1.03) * torch.sign(torch.randn(M, K, generator=g))
    A = (A.double() * scale_a).clamp(-3.4e38, 3.4e38).float()
    B = (torch.randn(K, N, generator=g).double() * scale_b).float()
    C = gemm(A, B.T, M, N, K, 0, 0)
    ref = A.double() @ B.double()
    assert rel_l2(C.cpu(), ref) < 2.0 ** -24 * (2 + math.sqrt(K / 2))


def tiny(M, K, e, seed):
    """Random values of 2^e times [0.5, 1.03), rounded to fp32 (subnormals
    below 2^-126)."""
    g = torch.Generator().manual_seed(seed)
    x = (0.5 + 0.53 * torch.rand(M, K, generator=g, dtype=torch.float64)) * torch.sign(torch.randn(M, K, generator=g))
    return (x * 2.0 ** e).float()


@pytest.mark.parametrize("M", [4, 96, 23000])   # 32 x 32, 64 x 64 (no workspace), 128 x 128 tiles
@pytest.mark.parametrize("e", [-112, -118, -126, -133, -140])
@pytest.mark.parametrize("a_t,b_t", [(0, 0), (1, 1)])
def test_tiny_operands(M, e, a_t, b_t, cuda):
    """Operands down to the fp32 subnormals keep all their bits against a
    large partner, on either side."""
    N, K = 128, 64
    g = torch.Generator().manual_seed(1)
    for swap in (False, True):
        A = torch.randn(M, K, generator=g) * 2.0 ** 60 if swap else tiny(M, K, e, 2)
        B = tiny(K, N, e, 3) if swap else torch.randn(K, N, generator=g) * 2.0 ** 60
        C = gemm(A.T if a_t else A, B if b_t else B.T, M, N, K, a_t, b_t, ws_floats=0 if M == 96 else 32 << 20)
        ref = A.double() @ B.double()
        assert rel_l2(C.cpu(), ref) < bound(K), (swap, rel_l2(C.cpu(), ref))


@pytest.mark.parametrize("rows", [96, 8229])
def test_resid_ln_tiny_operands(rows, cuda):
    """The same in both residual + LayerNorm forms."""
    L, K = native.lib(), 64
    g = torch.Generator().manual_seed(4)
    A, W = tiny(rows, K, -126, 5).cuda(), (torch.randn(256, K, generator=g) * 2.0 ** 100).cuda()
    bias, lw, lb = (torch.zeros(256, device="cuda") for _ in range(3))
    R, C, y = (torch.zeros(rows, 256, device="cuda") for _ in range(3))
    mu, rs = torch.zeros(rows, device="cuda"), torch.zeros(rows, device="cuda")
    native.check(L.ptcg_kernel_gemm_resid_ln(rows, K, P(A), P(W), P(bias), P(R), P(C), P(lw), P(lb), P(y), P(mu),
                                             P(rs), 0, None, None))
    torch.cuda.synchronize()
    ref = A.cpu().double() @ W.cpu().double().T
    assert rel_l2(C.cpu(), ref) < bound(K)


@pytest.mark.parametrize("M", [96, 23000])
def test_sums_past_the_scaled_range(M, cuda):
    """Sums of 2^110 pass the range of the scaled terms and run in fp32."""
    N, K = 64, 64
    A, B, _, _ = operands(M, N, K, 0, 0)
    A, B = A * 2.0 ** 60, B * 2.0 ** 50
    C = gemm(A, B.T, M, N, K, 0, 0)
    assert rel_l2(C.cpu(), A.double() @ B.double()) < 2.0 ** -24 * (2 + math.sqrt(K / 2))   # fp32 instructions


@pytest.mark.parametrize("M,K", [(100, 64), (23000, 64)])
@pytest.mark.parametrize("m,n", [(0, 0), (40, 1), (33, 37), (95, 58)])
def test_one_element_overflow(M, K, m, n, cuda):
    """x y = 2^128 (1 - 2^-11)^2 is finite in fp32, its operands' leading bf16
    terms (both 2^64) multiply to an infinity: one element of a tile, at any
    of its registers (64- and 128-row tiles, both row and column slices)."""
    N = 128
    x = 2.0 ** 63 * (2 - 2.0 ** -10)
    A, B = torch.zeros(M, K), torch.zeros(K, N)
    A[m, 3], B[3, n] = x, x
    C = gemm(A, B.T, M, N, K, 0, 0).cpu()
    ref = (A.double() @ B.double()).float()
    assert torch.isfinite(ref).all() and torch.equal(C, ref)


@pytest.mark.parametrize("rows", [96, 8229])
def test_resid_ln_one_element_overflow(rows, cuda):
    """The same in both residual + LayerNorm forms (32- and 64-row tiles)."""
    L, K = native.lib(), 64
    x = 2.0 ** 63 * (2 - 2.0 ** -10)
    A, W, R = (torch.zeros(s, device="cuda") for s in ((rows, K), (256, K), (rows, 256)))
    A[45, 7], W[41, 7] = x, x
    bias, lw, lb = (torch.zeros(256, device="cuda") for _ in range(3))
    C, y, mu, rs = (torch.zeros(s, device="cuda") for s in ((rows, 256), (rows, 256), (rows,), (rows,)))
    native.check(L.ptcg_kernel_gemm_resid_ln(rows, K, P(A), P(W), P(bias), P(R), P(C), P(lw), P(lb), P(y), P(mu),
                                             P(rs), 0, None, None))
    torch.cuda.synchronize()
    ref = torch.zeros(rows, 256)
    ref[45, 41] = 2.0 ** 127 * (2 - 2.0 ** -9 + 2.0 ** -21)
    assert torch.equal(C.cpu(), ref)


def test_rows_past_2_31_bytes(cuda):
    """A k-contiguous operand past 2^31 bytes: every row of the last tiles."""
    M, N, K = 525000, 64, 1024
    A = torch.randn(M, K, device="cuda", generator=torch.Generator("cuda").manual_seed(1))
    W = torch.randn(N, K, device="cuda", generator=torch.Generator("cuda").manual_seed(2))
    C = torch.zeros(M, N, device="cuda")
    native.check(native.lib().ptcg_kernel_gemm(M, N, K, P(A), K, 0, P(W), K, 0, P(C), N, 0, None, None, N, None, N,
                                               None, 0, None))
    torch.cuda.synchronize()
    for rows in (slice(0, 300), slice(M - 600, M)):
        ref = A[rows].double() @ W.double().T
        assert rel_l2(C[rows].cpu(), ref.cpu()) < bound(K)


@pytest.mark.parametrize("ws_floats", [0, 32 << 20])
@pytest.mark.parametrize("M,N,K", [(4, 4, 1500000), (130, 68, 1000000)])
def test_long_rows(M, N, K, ws_floats, cuda):
    """Rows of 2^20 floats and more: tile rows past the end lie past 2^28
    floats.  K / 16 roundings in one chain without a workspace."""
    A = torch.randn(M, K, device="cuda", generator=torch.Generator("cuda").manual_seed(1))
    W = torch.randn(N, K, device="cuda", generator=torch.Generator("cuda").manual_seed(2))
    C = gemm(A, W, M, N, K, 0, 0, ws_floats=ws_floats)
    assert rel_l2(C.cpu(), (A.double() @ W.double().T).cpu()) < bound(K)


@pytest.mark.parametrize("rows,K", [(1, 16), (31, 32), (33, 256), (8192, 64), (8193, 64), (20001, 256)])
def test_resid_ln_equals_product_then_ln(rows, K, cuda):
    """Both residual + LayerNorm forms (one 32-row tile per CU at most, and
    64-row tiles) give the product's and the LayerNorm's bits."""
    L = native.lib()
    g = torch.Generator("cuda").manual_seed(rows + K)
    f = lambda *s: torch.randn(*s, device="cuda", generator=g)
    A, W, bias, R, lw, lb = f(rows, K), f(256, K), f(256), f(rows, 256), f(256), f(256)
    C, y, C2, y2 = (torch.zeros(rows, 256, device="cuda") for _ in range(4))
    mu, rs, mu2, rs2 = (torch.zeros(rows, device="cuda") for _ in range(4))
    native.check(L.ptcg_kernel_gemm_resid_ln(rows, K, P(A), P(W), P(bias), P(R), P(C), P(lw), P(lb), P(y), P(mu),
                                             P(rs), 0, None, None))
    native.check(L.ptcg_kernel_gemm(rows, 256, K, P(A), K, 0, P(W), K, 0, P(C2), 256, 3, P(bias), P(R), 256, None, 256,
                                    None, 0, None))
    native.check(L.ptcg_kernel_layernorm_fwd(P(C2), P(lw), P(lb), P(y2), P(mu2), P(rs2), rows, 256, None))
    torch.cuda.synchronize()
    for a, b in ((C, C2), (y, y2), (mu, mu2), (rs, rs2)):
        assert torch.equal(a, b)


def test_resid_ln_operand_past_2_32_bytes(cuda):
    """Up to one 32-row tile per CU with an A whose extent does not fit 32
    bits: rows from both ends, C and its LayerNorm (about a dozen fp32
    roundings of 2^-24 after C)."""
    rows, K = 8192, 131088
    L = native.lib()
    g = torch.Generator("cuda").manual_seed(3)
    f = lambda *s: torch.randn(*s, device="cuda", generator=g)
    A, W, bias, R, lw, lb = f(rows, K), f(256, K), f(256), f(rows, 256), f(256), f(256)
    C, y = torch.zeros(rows, 256, device="cuda"), torch.zeros(rows, 256, device="cuda")
    mu, rs = torch.zeros(rows, device="cuda"), torch.zeros(rows, device="cuda")
    native.check(L.ptcg_kernel_gemm_resid_ln(rows, K, P(A), P(W), P(bias), P(R), P(C), P(lw), P(lb), P(y), P(mu),
                                             P(rs), 0, None, None))
    torch.cuda.synchronize()
    Wd = W.double().T.contiguous()
    for sl in (slice(0, 33), slice(4090, 4100), slice(rows - 40, rows)):
        ref = A[sl].double() @ Wd + bias.double() + R[sl].double()
        assert rel_l2(C[sl].cpu(), ref.cpu()) < bound(K), rel_l2(C[sl].cpu(), ref.cpu())
        ln = torch.nn.functional.layer_norm(C[sl].double(), (256,), lw.double(), lb.double(), 1e-5)
        assert rel_l2(y[sl].cpu(), ln.cpu()) < 12 * 2.0 ** -24
