"""Large contractions in two f16 parts (csrc/gemm_f16x2.hip) against binary64: every way the first operand may lie (contiguous in
k with whole and ragged pieces, contiguous in its rows, runs of the outer-product-mean's gradient that are whole stages and
that are not), both tile widths, every kind of output, and what the scales have to follow: rows that differ by 2^80, rows
that grow along k, rows of zeros, and rows that no scale can bring into range.

The bound of the first tests: a product of two parts each is within 2^-21 of |a||b| (two splits of 2^-23, the dropped product of
2^-22), a sum of K terms in binary32 within K / 16 * 2^-24 of sum |a||b|, sixteen products at a time: below (K + 4) * 2^-24
together from K = 72 on, for every output by itself.  It grows with K, where the errors of random operands average out: the tests
after them hold bounds that do not, on operands with ranges within a row (an element below 2^-14 of its row's largest is kept
to 2^-37 of that largest; the outputs to which that matters are computed again) and on parts that are left out."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    assert torch.cuda.is_available(), "GPU tests need a device"
    from proteinpredictmachinelearning_amd import ops as _ops

    return _ops


def _within(got, a, b, scale=1.0, add=None):
    """got against scale * a @ b.T (+ add), all in binary64"""
    K = a.shape[1]
    want = scale * (a @ b.t())
    size = scale * (a.abs() @ b.abs().t())
    if add is not None:
        want, size = want + add, size + add.abs()
    bad = ~((got.double() - want).abs() <= (K + 4) * 2.0 ** -24 * size + 1e-45)
    assert not bool(bad.any()), float(((got.double() - want).abs() / size)[bad].max())


def _operand(g, rows, K, kind):
    x = torch.randn(rows, K, device="cuda", generator=g)
    if kind == "ranges":                                # rows of very different sizes, some of them zero
        x *= torch.exp2(torch.randint(-40, 41, (rows, 1), device="cuda", generator=g).float())
        x[::17] = 0
    elif kind == "growing":                             # every stage's elements larger than the last one's: the scale moves on
        x *= torch.exp2(torch.arange(K, device="cuda").float() * (60.0 / K) - 30)
        x[5::7, :K // 2] = 0                            # (rows whose first half is zero)
    return x


# (M, K, N): ragged in every dimension; K of whole stages, of an odd number of them, of a 16-k step more, not a multiple of
# four; tiles of 256 columns, of 128, and an empty second half of the last one; 6000 x 128 x 1024: rows of whole lines
@pytest.mark.parametrize("kind", ["plain", "ranges", "growing"])
@pytest.mark.parametrize("M,K,N", [(20011, 136, 1004), (26368, 256, 200), (9001, 403, 390), (20600, 128, 1024), (22000, 165, 768), (4100, 320, 1031)])
def test_linear(ops, M, K, N, kind):
    g = torch.Generator(device="cuda").manual_seed(M + K + N)
    a, b = _operand(g, M, K, kind), _operand(g, N, K, "plain" if kind == "growing" else kind) * 0.1
    bias = torch.randn(N, device="cuda", generator=g) if kind == "plain" else None
    got = ops.mul_mat(a, b, bias)
    _within(got, a.double(), b.double(), 1.0, bias.double() if bias is not None else None)
    # the same contraction on operands that are contiguous in their rows: the same parts, the same bits
    if bias is None:
        assert torch.equal(got.view(torch.int32), ops.mul_mat_tn(a.t().contiguous(), b.t().contiguous()).view(torch.int32))


# slices of a long K, the smaller operand first and second
@pytest.mark.parametrize("kind", ["plain", "ranges", "growing"])
@pytest.mark.parametrize("M,K,N", [(768, 26368, 256), (200, 26367, 900), (1024, 4100, 1030), (900, 10609, 321)])
def test_slices(ops, M, K, N, kind):
    g = torch.Generator(device="cuda").manual_seed(M + K + N)
    a, b = _operand(g, M, K, kind), _operand(g, N, K, "plain")
    got = ops.mul_mat_tn(a.t().contiguous(), b.t().contiguous(), 0.5)
    _within(got, a.double(), b.double(), 0.5)
    assert torch.equal(ops.mul_mat_tn(a.t().contiguous(), b.t().contiguous()), ops.mul_mat(a, b))


# residues of whole stages and ragged ones, one and two tiles of features
@pytest.mark.parametrize("D,L,N", [(32, 96, 256), (32, 103, 130), (32, 128, 100), (8, 390, 72)])
def test_outer_product_mean(ops, D, L, N):
    g = torch.Generator(device="cuda").manual_seed(D + L + N)
    left, right = _operand(g, D * L, N, "ranges"), _operand(g, D * L, N, "plain")
    l64, r64 = left.double(), right.double()
    out = ops.outer_product_mean(left.reshape(-1), right.reshape(-1), D, L, N, 1)
    _within(out.reshape(D, D, L, L).permute(0, 2, 1, 3).reshape(D * L, D * L), l64, r64, 1.0 / N)
    grad = _operand(g, D * L, D * L, "ranges")          # rows (d1, i), columns (d2, j)
    g4 = grad.reshape(D, L, D, L).permute(0, 2, 1, 3).contiguous()
    gl, gr = ops.outer_prod_mean_back(g4.reshape(-1), left.reshape(-1), right.reshape(-1), D, L, N, 1)
    _within(gl.reshape(D * L, N), grad.double(), r64.t().contiguous(), 1.0 / N)
    _within(gr.reshape(D * L, N), grad.double().t().contiguous(), l64.t().contiguous(), 1.0 / N)


# Infinities, NaN and rows below 2^-111: those outputs the reference's way, the others what they are without them
@pytest.mark.parametrize("M,K,N", [(20011, 136, 1004), (768, 26368, 256)])
def test_operands_no_scale_brings_into_range(ops, M, K, N):
    g = torch.Generator(device="cuda").manual_seed(M)
    a, b = torch.randn(M, K, device="cuda", generator=g), torch.randn(N, K, device="cuda", generator=g)
    clean = ops.mul_mat(a, b)
    a[7, K - 1] = float("inf")
    a[300, 0] = float("nan")
    a[600] *= 2.0 ** -130
    b[3, 5] = -float("inf")
    b[70] *= 2.0 ** 100
    got = ops.mul_mat(a, b)
    want = a.double() @ b.double().t()
    size = torch.nan_to_num((a.double().abs() @ b.double().abs().t()), nan=0.0, posinf=0.0)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    inf = want.isinf()
    assert torch.equal(got[inf].double(), want[inf])
    fin = want.isfinite()
    assert bool(((got.double() - want).abs()[fin] <= ((K + 4) * 2.0 ** -24 * size + K * 1e-45)[fin]).all())
    far = torch.ones(M, dtype=torch.bool, device="cuda")          # tiles of rows that hold none of the planted elements
    for m in (7, 300, 600):
        far[m // 128 * 128:m // 128 * 128 + 128] = False
    assert torch.equal(got[far][:, 128:], clean[far][:, 128:])


def _narrow(got, a, b, scale=1.0):
    """|got - scale a b^T| within 2^-20 of scale sum |a||b| (the products' 2^-21, as much again for small elements), whatever K is: the
    binary32 sums of these operands, which change sign, stay far below that"""
    want, size = scale * (a @ b.t()), scale * (a.abs() @ b.abs().t())
    bad = ~((got.double() - want).abs() <= 2.0 ** -20 * size + 1e-45)
    assert not bool(bad.any()), (int(bad.sum()), float(((got.double() - want).abs() / size)[bad].max()))


def _spikes(g, a, b, size, where):
    """Columns of k where one operand is enormous and the other zero: one, one in every 32, a tenth of them"""
    K = a.shape[1]
    ks = {"one": [K // 3], "stages": list(range(5, K, 32)), "tenth": list(range(3, K, 10))}[where]
    a, b = a.clone(), b.clone()
    a[:, ks] = size * torch.randn(a.shape[0], len(ks), device="cuda", generator=g)
    b[:, ks] = 0
    return a, b


# Rows whose large elements meet zeros, in either operand, through every way A may lie and every kind of output
@pytest.mark.parametrize("where", ["one", "stages", "tenth"])
@pytest.mark.parametrize("size", [1e5, 1e7, 1e9, 1e12, 1e30])
def test_large_elements_that_meet_zeros(ops, size, where):
    g = torch.Generator(device="cuda").manual_seed(int(np.log10(size)) * 3 + len(where))
    for M, K, N in ((20011, 136, 1004), (26368, 256, 200), (9001, 403, 390), (22000, 165, 768)):      # (the last: streaming stores)
        a, b = (torch.randn(n, K, device="cuda", generator=g) for n in (M, N))
        for first in (True, False):
            x, y = _spikes(g, a, b, size, where) if first else _spikes(g, b, a, size, where)[::-1]
            got = ops.mul_mat(x, y)
            _narrow(got, x.double(), y.double())
            assert torch.equal(got.view(torch.int32), ops.mul_mat_tn(x.t().contiguous(), y.t().contiguous()).view(torch.int32))
    for M, K, N in ((768, 26368, 256), (900, 10609, 321)):      # slices
        a, b = (torch.randn(n, K, device="cuda", generator=g) for n in (M, N))
        for first in (True, False):
            x, y = _spikes(g, a, b, size, where) if first else _spikes(g, b, a, size, where)[::-1]
            _narrow(ops.mul_mat_tn(x.t().contiguous(), y.t().contiguous(), 0.5), x.double(), y.double(), 0.5)
    for D, L, N in ((32, 96, 256), (32, 103, 130), (32, 192, 72)):        # outer-product-mean and its gradients (the last: streaming stores)
        left, right = (torch.randn(D * L, N, device="cuda", generator=g) for _ in range(2))
        x, y = _spikes(g, left, right, size, where)
        out = ops.outer_product_mean(x.reshape(-1), y.reshape(-1), D, L, N, 1)
        _narrow(out.reshape(D, D, L, L).permute(0, 2, 1, 3).reshape(D * L, D * L), x.double(), y.double(), 1.0 / N)
        grad = torch.randn(D * L, D * L, device="cuda", generator=g)
        # enormous gradients of residues whose projection is zero, on the right for one gradient, on the left for the other
        gr_l, right0 = _spikes(g, grad, right.t().contiguous(), size, where)
        gr_r, left0 = _spikes(g, grad.t().contiguous(), left.t().contiguous(), size, where)
        for full, l, r in ((gr_l, left, right0.t().contiguous()), (gr_r.t().contiguous(), left0.t().contiguous(), right)):
            g4 = full.reshape(D, L, D, L).permute(0, 2, 1, 3).contiguous()
            dl, dr = ops.outer_prod_mean_back(g4.reshape(-1), l.reshape(-1), r.reshape(-1), D, L, N, 1)
            if full is gr_l:
                _narrow(dl.reshape(D * L, N), full.double(), r.double().t().contiguous(), 1.0 / N)
            else:
                _narrow(dr.reshape(D * L, N), full.double().t().contiguous(), l.double().t().contiguous(), 1.0 / N)


def test_large_elements_in_a_few_rows_and_rows_that_grow(ops):
    """A spike in single rows, rows whose later elements are larger by 2^100 and meet zeros (what the sums held by then leaves
    binary32's range), rows and columns of zeros between them, a bias, and rows far below the smallest normal number"""
    g = torch.Generator(device="cuda").manual_seed(11)
    M, K, N = 20011, 136, 1004
    a, b = torch.randn(M, K, device="cuda", generator=g), torch.randn(N, K, device="cuda", generator=g)
    b[:, 70:] = 0
    a[5, 100] = 1e20
    a[300:310, 71] = -3e8
    for k, e in ((0, -90), (33, -50), (66, 0), (100, 60), (130, 120)):
        a[700:720, k:] = torch.randn(20, K - k, device="cuda", generator=g) * 2.0 ** e
    a[1000:1003] = 0
    a[2000:2010] *= 2.0 ** -122
    b[17] = 0
    b[40:44, 3] = 1e15
    a[:, 3] *= (torch.arange(M, device="cuda") % 2).float()
    bias = torch.randn(N, device="cuda", generator=g)
    _narrow(ops.mul_mat(a, b), a.double(), b.double())
    got = ops.mul_mat(a, b, bias).double()
    want, size = a.double() @ b.double().t() + bias.double(), a.double().abs() @ b.double().abs().t() + bias.double().abs()
    assert bool(((got - want).abs() <= 2.0 ** -20 * size).all())
    assert not bool(ops.mul_mat(a, b)[1000:1003].any()) and not bool(ops.mul_mat(a, b)[:, 17].any())


# One constant in all elements: the errors of the parts add up instead of averaging out
def test_constants_with_the_largest_rounding(ops):
    x, y = 1 + 2.0 ** -11 - 2.0 ** -23, 1 + 2.0 ** -10 - 2.0 ** -11 + 3 * 2.0 ** -23
    a, b = torch.full((20011, 128), x, device="cuda"), torch.full((1004, 128), y, device="cuda")
    want = 128 * float(np.float32(x)) * float(np.float32(y))
    # the parts' 2^-21, and eight binary32 additions of sixteen products
    assert bool(((ops.mul_mat(a, b).double() - want).abs() <= (2.0 ** -21 + 8 * 2.0 ** -24) * want).all())


# Products that binary32 holds (24 bits together) and that the three kept ones carry: 11 bits against up to 23, either way round
@pytest.mark.parametrize("wide_first", [True, False])
@pytest.mark.parametrize("wide,narrow", [(13, 11), (23, 1)])
def test_exact_products_stay_exact(ops, wide, narrow, wide_first):
    g = torch.Generator(device="cuda").manual_seed(3)

    def whole(bits, *shape):
        x = torch.randint(2 ** (bits - 1), 2 ** bits, shape, device="cuda", generator=g).float()
        return x * (torch.randint(0, 2, shape, device="cuda", generator=g) * 2 - 1) * torch.exp2(torch.randint(0, 4, shape, device="cuda", generator=g).float())

    a = torch.zeros(20011, 136, device="cuda")
    a[torch.arange(20011), torch.randint(0, 136, (20011,), device="cuda", generator=g)] = whole(wide if wide_first else narrow, 20011)   # one a row: no sum to round
    b = whole(narrow if wide_first else wide, 1004, 136)
    assert torch.equal(ops.mul_mat(a, b).double(), a.double() @ b.double().t())


# A bound that does not grow with K, which operands without their low halves (or a product that is left out) fail
@pytest.mark.parametrize("M,K,N", [(20011, 136, 1004), (768, 26368, 256), (900, 10609, 321), (1024, 4100, 1030)])
def test_the_low_halves_are_there(ops, M, K, N):
    g = torch.Generator(device="cuda").manual_seed(M + K + N)
    a, b = (torch.randn(n, K, device="cuda", generator=g) for n in (M, N))
    a64, b64 = a.double(), b.double()
    want = a64 @ b64.t()
    spread = ((a64 * a64) @ (b64 * b64).t()).sqrt()

    def rms(c):
        return float((((c - want) / spread) ** 2).mean().sqrt())

    assert rms(ops.mul_mat(a, b).double()) <= 2.0 ** -19
    assert rms(ops.mul_mat_tn(a.t().contiguous(), b.t().contiguous()).double()) <= 2.0 ** -19
    for part_a, part_b in ((a.half(), b.half()), (a.half(), b), (a, b.half())):      # (each 2^-13 or more)
        assert rms(part_a.double() @ part_b.double().t()) > 2.0 ** -15


@pytest.mark.parametrize("per_thread", [False, True])
def test_recorded_calls_take_no_workspace(ops, per_thread):
    """Contractions that take a workspace, recorded into a graph from a stream of the caller's and from the per-thread default
    stream: an allocation made meanwhile would be gone by the time the graph runs.  Replayed with other work in between, on other
    operands each time; the bits are those of the forms without workspace, the result the eager one's."""
    import ctypes as C

    from proteinpredictmachinelearning_amd import cabi

    lib = cabi.load()                                   # (its handle finds the runtime that it is bound to, too)
    ops._lib()
    own = torch.cuda.Stream()
    stream = C.c_void_p(2 if per_thread else own.cuda_stream)         # 2: hipStreamPerThread
    g = torch.Generator(device="cuda").manual_seed(8)
    cases = [(torch.randn(M, K, device="cuda", generator=g), torch.randn(N, K, device="cuda", generator=g), torch.empty(M, N, device="cuda"))
             for M, K, N in ((26368, 256, 200), (64, 8192, 64))]
    torch.cuda.synchronize()
    graph, exe = C.c_void_p(), C.c_void_p()
    assert lib.hipStreamBeginCapture(stream, 2) == 0
    for a, b, c in cases:
        cabi.check("mul_mat_hip", lib.mul_mat_hip(a.data_ptr(), b.data_ptr(), c.data_ptr(), a.shape[0], a.shape[1], b.shape[0], None, stream))
    assert lib.hipStreamEndCapture(stream, C.byref(graph)) == 0
    assert lib.hipGraphInstantiate(C.byref(exe), graph, None, None, C.c_size_t(0)) == 0
    for _ in range(3):
        for a, b, c in cases:
            a.normal_(generator=g)
            c.fill_(float("nan"))
        torch.cuda.synchronize()
        assert lib.hipGraphLaunch(exe, stream) == 0
        torch.cuda.synchronize()
        for a, b, c in cases:
            _within(c, a.double(), b.double())
            eager = ops.mul_mat(a, b).double()
            assert bool(((c.double() - eager).abs() <= 2.0 ** -19 * (a.double().abs() @ b.double().abs().t())).all())
    assert lib.hipGraphExecDestroy(exe) == 0 and lib.hipGraphDestroy(graph) == 0
