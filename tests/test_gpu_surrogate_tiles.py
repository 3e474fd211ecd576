"""GPU: the surrogate's products where their tiles, block orders and stores end:
each tile size with rows, columns and contractions short of it, the row and the
split order, masks and bf16 outputs on and off 16-byte rows, the column sums and
the moment-tensor contraction formed beside a product, and Adam on a list.

Sums of K bf16 products in FP32 differ from the exact ones by at most
K 2^-23 times the sum of their magnitudes (each addition rounds once, in any
order); a bf16 result by another 2^-8 of itself."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _bf(rng, r, c, ld=None):
    t = torch.zeros((r, ld or c), dtype=torch.bfloat16, device="cuda:0")
    t[:, :c] = torch.from_numpy(rng.standard_normal((r, c)).astype(np.float32)).to("cuda:0")
    return t


def _exact(a, b):
    a, b = a.double().cpu(), b.double().cpu()
    return a @ b, a.abs() @ b.abs()


# rows, columns, contraction: 64 x 32, 64 x 64 and 128 x 128 tiles, the last with
# 8 row tiles an XCD and more, and remainders of each
SHAPES = [(8, 8, 8), (72, 40, 136), (520, 2056, 72), (1032, 4104, 40), (8200, 264, 200),
          (131080, 136, 72)]


@pytest.mark.parametrize("transB", [0, 1])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_bf16_output_and_mask(M, N, K, transB):
    from cgfd3d_amd import surrogate as sg
    rng = np.random.default_rng(M + N + K)
    a = _bf(rng, M, K)
    b = _bf(rng, N, K) if transB else _bf(rng, K, N)
    bias = torch.from_numpy(rng.standard_normal(N).astype(np.float32)).to("cuda:0")
    want, mag = _exact(a, b.t() if transB else b)
    lim = K * 2.0 ** -23 * mag
    for ld in (N, N + 8, N + 4):                 # the last: rows off 16 bytes
        mask = _bf(rng, M, N, ld)
        out = torch.full((M, ld), 7.0, dtype=torch.bfloat16, device="cuda:0")
        sg.gemm(M, N, K, a, K, 0, b, b.shape[1], transB, epi=sg.EPI_MASK, mask=mask, ldm=ld,
                C16=out, ldc16=ld)
        w = torch.where(mask[:, :N].cpu() > 0, want, torch.zeros(()).double())
        assert ((out[:, :N].double().cpu() - w).abs() <= lim + 2.0 ** -8 * w.abs()).all()
        assert bool((out[:, N:] == 7.0).all())
        sg.gemm(M, N, K, a, K, 0, b, b.shape[1], transB, bias=bias, epi=sg.EPI_RELU, C16=out,
                ldc16=ld)
        w = (want + bias.double().cpu()).clamp(min=0)
        l2 = lim + 2.0 ** -23 * (mag + bias.double().cpu().abs())
        assert ((out[:, :N].double().cpu() - w).abs() <= l2 + 2.0 ** -8 * w.abs()).all()
        assert bool((out[:, N:] == 7.0).all())


@pytest.mark.parametrize("splitk", [1, 5, 8, 19, 128])
@pytest.mark.parametrize("M,N,K", [(8, 8, 64), (136, 72, 4104), (32, 520, 1000), (256, 2056, 264)])
def test_products_with_column_sums(M, N, K, splitk):
    from cgfd3d_amd import surrogate as sg
    rng = np.random.default_rng(M + N + K)
    a, g = _bf(rng, K, M), _bf(rng, K, N)
    c = torch.empty((M, N), device="cuda:0")
    s = torch.empty(N, device="cuda:0")
    work = torch.empty(splitk * (M + 1) * N, device="cuda:0")
    sg.gemm_colsum(M, N, K, a, M, g, N, c, s, splitk, work)
    want, mag = _exact(a.t(), g)
    assert ((c.double().cpu() - want).abs() <= K * 2.0 ** -23 * mag).all()
    g = g.double().cpu()
    assert ((s.double().cpu() - g.sum(0)).abs() <= K * 2.0 ** -23 * g.abs().sum(0)).all()


@pytest.mark.parametrize("nk,nc,times", [(6, 3, 4), (1, 8, 1), (8, 1, 16), (2, 4, 1)])
@pytest.mark.parametrize("nsamp,rps", [(8, 8), (40, 40), (72, 1024)])
def test_contraction_beside_the_product(nsamp, rps, nk, nc, times):
    """Both outputs are those of the product and the contraction apart, bit for bit."""
    from cgfd3d_amd import surrogate as sg
    M, N, K = nsamp * rps, nk * nc * times, 136
    rng = np.random.default_rng(M + N)
    a, b = _bf(rng, M, K), _bf(rng, K, N)
    f = lambda *n: torch.from_numpy(rng.standard_normal(n).astype(np.float32)).to("cuda:0")
    bias, m = f(N), f(nsamp, nk)
    c, c2 = torch.empty((M, N), device="cuda:0"), torch.empty((M, N), device="cuda:0")
    y, y2 = torch.empty(M * N // nk, device="cuda:0"), torch.empty(M * N // nk, device="cuda:0")
    sg.gemm_mt(M, N, K, a, b, bias, c, nk, nc, rps, m, y)
    sg.gemm(M, N, K, a, K, 0, b, N, 0, bias=bias, C32=c2, ldc32=N)
    sg.mt_contract(nsamp, rps * times, nc, nk, m, c2, y2)
    assert torch.equal(c, c2) and torch.equal(y, y2)


def _spread(rng, r, c, ld):
    """r rows of c values ld apart; what lies between them is not touched."""
    t = torch.empty(r * ld, dtype=torch.bfloat16, device="cuda:0").view(r, ld)
    t[:, :c] = torch.from_numpy(rng.standard_normal((r, c)).astype(np.float32)).to("cuda:0")
    return t


# leading dimensions just past the 32-bit byte offsets of 16, 8 and 4 rows
W16, W8, W4 = 143165584, 306783384, 715827888


@pytest.mark.parametrize("M,N,K,transA,transB,lda,ldb", [
    (8, 8, 16, 0, 0, 16, W16), (8, 8, 16, 0, 0, W4, 8), (8, 8, 16, 0, 1, 16, W4),
    (8, 8, 16, 1, 0, W8, 8), (32768, 8, 8, 1, 0, W4, 8)])
def test_rows_past_32_bit_offsets(M, N, K, transA, transB, lda, ldb):
    from cgfd3d_amd import surrogate as sg
    rng = np.random.default_rng(M + lda % 97)
    a = _spread(rng, K, M, lda) if transA else _spread(rng, M, K, lda)
    b = _spread(rng, N, K, ldb) if transB else _spread(rng, K, N, ldb)
    c = torch.empty((M, N), device="cuda:0")
    sg.gemm(M, N, K, a, lda, transA, b, ldb, transB, C32=c, ldc32=N)
    want, mag = _exact(a[:, :M].t() if transA else a[:, :K], b[:, :K].t() if transB else b[:, :N])
    assert ((c.double().cpu() - want).abs() <= K * 2.0 ** -23 * mag).all()
    if transA:
        s, work = torch.empty(N, device="cuda:0"), torch.empty((M + 1) * N, device="cuda:0")
        sg.gemm_colsum(M, N, K, a, lda, b, ldb, c, s, 1, work)
        assert ((c.double().cpu() - want).abs() <= K * 2.0 ** -23 * mag).all()
        g = b[:, :N].double().cpu()
        assert ((s.double().cpu() - g.sum(0)).abs() <= K * 2.0 ** -23 * g.abs().sum(0)).all()


def test_more_blocks_than_a_launch_holds_in_x():
    """2^27 rows in 8 splits: 2^23 blocks of 512 threads.  Rows of ones among zeros,
    so that the result is small whole numbers."""
    from cgfd3d_amd import surrogate as sg
    M, N, K, S = 1 << 27, 8, 256, 8
    a = torch.zeros((M, K), dtype=torch.bfloat16, device="cuda:0")
    at = [0, 127, 128, 1 << 26, M - 129, M - 1]
    a[at] = 1
    b = torch.zeros((K, N), dtype=torch.bfloat16, device="cuda:0")
    b[::3] = 1
    b[1, 5] = 2
    c = torch.empty((M, N), device="cuda:0")
    work = torch.empty(S * M * N, device="cuda:0")
    sg.gemm(M, N, K, a, K, 0, b, N, 0, C32=c, ldc32=N, splitk=S, work=work)
    want = b.float().sum(0)
    assert torch.equal(c[at], want.expand(len(at), N))
    assert int(torch.count_nonzero(c)) == len(at) * N
    del a, c, work
    torch.cuda.empty_cache()


def test_contraction_of_rows_past_32_bit_offsets():
    from cgfd3d_amd import surrogate as sg
    from cgfd3d_amd._lib import check, lib
    M, N, K, nk, nc, ldb = 8, 72, 8, 6, 3, W4
    rng = np.random.default_rng(5)
    a, b = _bf(rng, M, K), _spread(rng, K, N, ldb)
    m = torch.from_numpy(rng.standard_normal((1, nk)).astype(np.float32)).to("cuda:0")
    bias = torch.zeros(N, device="cuda:0")
    c, y = torch.empty((M, N), device="cuda:0"), torch.empty(M * N // nk, device="cuda:0")
    y2 = torch.empty_like(y)
    p = lambda t: t.data_ptr()
    check(lib().cgfds_gemm_bf16_mt(M, N, K, p(a), K, p(b), ldb, p(bias), p(c), N, nk, nc, M, p(m),
                                   p(y), torch.cuda.current_stream().cuda_stream), "gemm_bf16_mt")
    want, mag = _exact(a, b[:, :N])
    assert ((c.double().cpu() - want).abs() <= K * 2.0 ** -23 * mag).all()
    sg.mt_contract(1, M * N // (nk * nc), nc, nk, m, c, y2)
    assert torch.equal(y, y2)


@pytest.mark.parametrize("sizes", [(1,), (1023, 1024, 1025, 7), tuple(range(1, 40))])
def test_adam_on_a_list(sizes):
    from cgfd3d_amd import surrogate as sg
    rng = np.random.default_rng(len(sizes))
    f = lambda n: torch.from_numpy(rng.random(n, dtype=np.float32)).to("cuda:0")
    one = [[f(n), f(n), f(n), f(n),
            torch.empty(n, dtype=torch.bfloat16, device="cuda:0") if i % 2 else None]
           for i, n in enumerate(sizes)]
    many = [[None if t is None else t.clone() for t in q] for q in one]
    for q in one:
        sg.adam(*q, 1e-3, 3)
    sg.adam_multi(many, 1e-3, 3)
    for p, q in zip(one, many):
        assert all(torch.equal(s, t) for s, t in zip(p, q) if s is not None)
