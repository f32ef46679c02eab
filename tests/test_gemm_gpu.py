"""Weight-gradient kernel C = A^T B (csrc/gemm_tn.hip) against float64 on
the same f16/bf16 inputs.  Bound: |C - C64| <= 1e-4 * (|A|^T |B|) elementwise
(the products are exact in fp32; only the fp32 accumulation rounds)."""
import pytest
import torch

from graph_rws_amd.core.ops import gemm_tn, gemm_tn_f32, gemm_tn_f32_tiles, gemm_tn_supported

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("K,M,N", [(0, 8, 16), (1, 8, 8), (31, 128, 136), (1000, 136, 256),
                                   (5000, 256, 8), (100003, 128, 256), (300000, 608, 256)])
def test_gemm_tn_matches_float64(cuda_device, dt, K, M, N):
    print(f"case gemm_tn {dt} K={K} M={M} N={N}", flush=True)
    g = torch.Generator(device=cuda_device).manual_seed(K + M + N)
    A = torch.randn(K, M, generator=g, device=cuda_device).to(dt)
    B = torch.randn(K, N, generator=g, device=cuda_device).to(dt)
    C = gemm_tn(A, B)
    assert C.shape == (M, N) and C.dtype == torch.float32
    ref = A.double().t() @ B.double()
    bound = A.double().abs().t() @ B.double().abs()
    assert bool(((C.double() - ref).abs() <= 1e-4 * bound + 1e-30).all())
    assert torch.equal(C, gemm_tn(A, B))  # deterministic


def test_gemm_tn_strided_and_low_precision_output(cuda_device):
    A0 = torch.randn(20000, 200, device=cuda_device).half()
    A = A0[:, 8:136]  # row stride 200, offset 16 bytes
    B = torch.randn(20000, 64, device=cuda_device).half()
    assert gemm_tn_supported(A, B)
    ref = A.double().t() @ B.double()
    for od in (torch.float16, torch.float32):
        C = gemm_tn(A, B, out_dtype=od)
        assert C.dtype == od
        tol = 2e-3 if od == torch.float16 else 1e-4
        bound = A.double().abs().t() @ B.double().abs()
        assert bool(((C.double() - ref).abs() <= tol * bound).all())
    # a misaligned start and ragged widths go through a widened copy; a
    # ragged width over a wider buffer reuses its row padding (NaN there
    # must not reach the result)
    Am = A0[:, 1:129]
    assert gemm_tn_supported(Am, B)
    Cm = gemm_tn(Am, B)
    bm = Am.double().abs().t() @ B.double().abs()
    assert bool(((Cm.double() - Am.double().t() @ B.double()).abs() <= 1e-4 * bm).all())
    Bp = torch.full((20000, 48), float("nan"), device=cuda_device).half()
    Bp[:, :41] = torch.randn(20000, 41, device=cuda_device).half()
    Br = Bp[:, :41]
    Cr = gemm_tn(A, Br)
    assert Cr.shape == (128, 41) and bool(torch.isfinite(Cr).all())
    br = A.double().abs().t() @ Br.double().abs()
    assert bool(((Cr.double() - A.double().t() @ Br.double()).abs() <= 1e-4 * br).all())
    A41 = torch.randn(20000, 41, device=cuda_device).bfloat16()
    B41 = torch.randn(20000, 41, device=cuda_device).bfloat16()
    C41 = gemm_tn(A41, B41)
    b41 = A41.double().abs().t() @ B41.double().abs()
    assert bool(((C41.double() - A41.double().t() @ B41.double()).abs() <= 1e-4 * b41).all())


def test_graphconv_autocast_backward_uses_split_k(cuda_device):
    """A BCSRGraphConv under f16 autocast: the weight gradients (both paths)
    come out of the split-K kernel and match float64 autograd over the same
    f16-quantised operands within 2e-2 of the largest magnitude."""
    from graph_rws_amd import synth
    from graph_rws_amd.data import BCSRGraph
    from graph_rws_amd.layers import BCSRGraphConv
    torch.manual_seed(0)
    g = synth.chung_lu(6000, 60000, 2.2, seed=5)
    G = BCSRGraph.from_csr(g.row_ptr, g.col_idx, g.values, g.num_nodes, g.num_nodes, tile_cols=16,
                           device=cuda_device, values_dtype=torch.float16)
    conv = BCSRGraphConv(64, 32).to(cuda_device)
    X = torch.randn(g.num_nodes, 64, device=cuda_device).half()
    R = torch.randn(g.num_nodes, 32, device=cuda_device)
    with torch.autocast("cuda", dtype=torch.float16):
        out = conv(G, X, features_target=X)
        loss = (out.float() * R).sum()
    loss.backward()
    import scipy.sparse as sps
    vals16 = torch.from_numpy(g.values.numpy()).half().double().numpy()
    A = torch.from_numpy(sps.csr_matrix((vals16, g.col_idx.numpy(), g.row_ptr.numpy()),
                                        shape=(g.num_nodes, g.num_nodes)).toarray())
    Xd = X.double().cpu()
    Wn = conv.weight_neigh.detach().half().double().cpu().requires_grad_(True)
    Ws = conv.weight_self.detach().half().double().cpu().requires_grad_(True)
    ref = A @ (Xd @ Wn) + Xd @ Ws
    (ref * R.double().cpu()).sum().backward()
    for got, want in ((conv.weight_neigh.grad, Wn.grad), (conv.weight_self.grad, Ws.grad)):
        assert got.dtype == torch.float32
        d = float((got.double().cpu() - want).abs().max())
        assert d <= 2e-2 * float(want.abs().max()), d


@pytest.mark.parametrize("K,M,N", [(0, 8, 16), (1, 4, 4), (31, 32, 36), (255, 33, 64), (257, 65, 7), (4097, 64, 129),
                                   (9000, 1433, 16), (100003, 128, 256), (65536, 200, 41)])
def test_gemm_tn_f32_matches_float64(cuda_device, K, M, N):
    """Edges of the 32/64/128-column tiles, ragged widths and K
    remainders.  Bound: a chunk's rows summed in f32 in order, then the
    chunks' partials: (rows + chunks) * 2^-24 of |A|^T |B|, with the split's
    own chunks (f32_shape in csrc/gemm_tn.hip)."""
    g = torch.Generator(device=cuda_device).manual_seed(K + M + N)
    A = torch.randn(K, M, generator=g, device=cuda_device)
    B = torch.randn(K, N, generator=g, device=cuda_device)
    C = gemm_tn_f32(A, B)
    assert C.shape == (M, N) and C.dtype == torch.float32
    ref = A.double().t() @ B.double()
    bound = A.double().abs().t() @ B.double().abs()
    chunks = max(1, min(max(8, 512 // gemm_tn_f32_tiles(M, N) // 8 * 8), -(-K // 256)))
    rows = -(-(-(-K // chunks)) // 32) * 32
    assert bool(((C.double() - ref).abs() <= (rows + chunks) * 2.0 ** -24 * bound).all())
    assert torch.equal(C, gemm_tn_f32(A, B))  # deterministic
    wide = torch.full((K, N + 9), float("nan"), device=cuda_device)
    wide[:, :N] = B  # a column view of a wider buffer: its padding must not reach the result
    assert torch.equal(C, gemm_tn_f32(A, wide[:, :N]))
    wide[:, 1:N + 1] = B  # a misaligned start
    assert torch.equal(C, gemm_tn_f32(A, wide[:, 1:N + 1]))


@pytest.mark.parametrize("K,M,N", [(1, 4, 4), (31, 32, 36), (33, 64, 65), (255, 33, 64), (257, 65, 7), (4097, 64, 129),
                                   (9001, 1433, 16), (16387, 24, 9), (65537, 200, 41), (100003, 128, 256)])
@pytest.mark.parametrize("wide", ["a", "b"])
def test_gemm_tn_f32_is_exact_on_integers(cuda_device, K, M, N, wide):
    """One operand of odd integers below 4,096 (12 bits: more than an f16 or
    bf16 holds), the other of -1 and 1: every partial sum is a whole number
    below 2^24 (a random walk of 100,003 steps of 2,400 ends under 7.6e5 in
    its root mean square, the limit is 22 times that), so f32 adds exactly
    in any order, and an operand rounded to 16 bits, a row lost from a
    remainder or one taken twice shows in the result."""
    print(f"case gemm_tn_f32 integers K={K} M={M} N={N} {wide}", flush=True)
    g = torch.Generator(device=cuda_device).manual_seed(3 * K + M + N)
    big = [M, N][wide == "b"]
    W = torch.randint(0, 2048, (K, big), generator=g, device=cuda_device) * 2 + 1
    W = (W * (torch.randint(0, 2, (K, big), generator=g, device=cuda_device) * 2 - 1)).float()
    S = (torch.randint(0, 2, (K, M + N - big), generator=g, device=cuda_device) * 2 - 1).float()
    A, B = (W, S) if wide == "a" else (S, W)
    assert torch.equal(gemm_tn_f32(A, B).double(), A.double().t() @ B.double())


def test_tall_f32_weight_grad_of_expanded_and_batched_operands(cuda_device):
    """Operands the f32 kernel does not take (rows that share memory,
    gradients batched by vmap) go to the library's product.  Whole numbers
    up to 8: every sum is below 2^24, so the product is exact."""
    from graph_rws_amd.layers.layer import F32_TN_ROWS, _weight_grad
    n = F32_TN_ROWS + 3
    gen = torch.Generator(device=cuda_device).manual_seed(5)
    x = torch.randint(1, 9, (n, 24), generator=gen, device=cuda_device).float()
    g = torch.randint(1, 9, (n, 9), generator=gen, device=cuda_device).float()
    ones = torch.ones(1, 24, device=cuda_device).expand(n, 24)

    class Product(torch.autograd.Function):
        @staticmethod
        def forward(ctx, x, w):
            ctx.save_for_backward(x)
            return x @ w

        @staticmethod
        def backward(ctx, grad):
            return None, _weight_grad(ctx.saved_tensors[0], grad.contiguous())

    def same(c, a, b):
        assert torch.equal(c.double(), a.double().t() @ b.double())

    with torch.no_grad():
        same(_weight_grad(ones, g), ones, g)
        same(_weight_grad(x, g), x, g)
    w = torch.randn(24, 9, generator=gen, device=cuda_device, requires_grad=True)
    both = torch.stack([g, 2 * g])
    dw, = torch.autograd.grad(Product.apply(x, w), w, both, is_grads_batched=True)
    same(dw[0], x, g)
    same(dw[1], x, 2 * g)
