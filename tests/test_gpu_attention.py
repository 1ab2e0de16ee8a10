"""GPU parity of the fused attention forward (flash_attn_forward_hip) against the CPU oracle, which is
itself checked bit for bit against the reference's compiled src/ops/FlashAttn.cpp.

Bar: 1e-4 relative on O (normwise per case, the f32 bar of this backend) and 1e-5 + 1e-5 * |LSE| on
LSE.  The GPU sums in another order (exact bf16 split products on the matrix pipe, binary32 sums, keys 32 at a
time, hardware exp/log), so equality is not expected; special rows (fully masked, masked first block) must match exactly: O = 0, LSE = -inf.
"""
import json
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

RTOL = 1e-4


@pytest.fixture(scope="module")
def ops():
    assert torch.cuda.is_available(), "GPU tests need a device"
    from proteinpredictmachinelearning_amd import ops as _ops

    return _ops


def _dev(a):
    return None if a is None else torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _run(ops, q, k, v, bias=None, **kw):
    o, lse = ops.flash_attn_forward(_dev(q), _dev(k), _dev(v), _dev(bias), **kw)
    ops.synchronize()
    return o.cpu().numpy(), lse.cpu().numpy()


def _check(got_o, got_lse, want_o, want_lse):
    dead = np.isneginf(want_lse)
    assert (np.isneginf(got_lse) == dead).all(), "rows written as masked differ"
    assert (got_o[dead] == 0).all()
    scale = max(np.abs(want_o).max(), 1e-30)
    err = np.abs(got_o.astype(np.float64) - want_o).max() / scale
    assert err <= RTOL, f"O normwise {err:.3e}"
    live = ~dead
    lerr = np.abs(got_lse[live].astype(np.float64) - want_lse[live])
    assert (lerr <= 1e-5 + 1e-5 * np.abs(want_lse[live])).all(), f"LSE {lerr.max():.3e}"


CASES = [
    # B, h, L, d, causal, bias
    (1, 1, 1, 4, False, False),          # a single key
    (2, 3, 37, 8, False, True),          # ragged tile, small head
    (1, 4, 103, 32, False, True),        # pair-track plane of the configured model (L = 103, d = 32)
    (1, 4, 103, 32, False, False),
    (1, 2, 128, 32, True, False),        # four full tiles, causal
    (1, 2, 129, 32, False, True),        # first shape of the eight-wave instance, ragged
    (2, 2, 256, 32, False, True),        # MSA-track plane (L = 256): bias rows read 16 bytes at a time
    (1, 2, 300, 32, True, True),         # more keys than one LDS stage holds (256)
    (1, 2, 70, 64, False, True),         # d = 64 instance
    (1, 1, 200, 64, True, False),        # d = 64, two LDS stages (128 keys each), causal
    (1, 2, 45, 20, False, True),         # d not a multiple of 32: padded columns
    (1, 1, 64, 48, False, False),
]


@pytest.mark.parametrize("B,h,L,d,causal,use_bias", CASES)
def test_flash_attn_forward_matches_oracle(ops, oracle, B, h, L, d, causal, use_bias):
    rng = np.random.default_rng(1000 * L + d + int(causal))
    q, k, v = [rng.standard_normal((B, h, L, d)).astype(np.float32) for _ in range(3)]
    bias = (2 * rng.standard_normal((B, h, L, L))).astype(np.float32) if use_bias else None
    want_o, want_lse = oracle.flash_attn_forward(q, k, v, bias, causal=causal)
    got_o, got_lse = _run(ops, q, k, v, bias, causal=causal)
    _check(got_o, got_lse, want_o, want_lse)


# planes of 129 to 256: waves without queries, tiles past the last key
@pytest.mark.parametrize("L,d,causal", [(130, 24, False), (161, 32, True), (193, 8, False), (224, 32, False), (255, 32, True), (257, 32, False)])
def test_flash_attn_forward_whole_planes(ops, oracle, L, d, causal):
    rng = np.random.default_rng(L)
    q, k, v = [rng.standard_normal((1, 3, L, d)).astype(np.float32) for _ in range(3)]
    bias = (2 * rng.standard_normal((1, 3, L, L))).astype(np.float32)
    _check(*_run(ops, q, k, v, bias, causal=causal), *oracle.flash_attn_forward(q, k, v, bias, causal=causal))


# four-wave and eight-wave work-groups on either side of the numbers of planes between which the choice changes: same bits
@pytest.mark.parametrize("planes", [129, 300, 400])
@pytest.mark.parametrize("L,d,causal,use_bias", [(129, 32, False, True), (161, 24, True, True), (176, 32, False, False), (224, 8, True, False),
                                                 (255, 32, False, True), (256, 32, True, True)])
def test_flash_attn_forward_has_the_bits_of_fewer_planes(ops, planes, L, d, causal, use_bias):
    g = torch.Generator(device="cuda")
    g.manual_seed(planes + L)
    q, k, v = (torch.randn(1, planes, L, d, device="cuda", generator=g) for _ in range(3))
    bias = torch.randn(1, planes, L, L, device="cuda", generator=g) if use_bias else None
    o, lse = ops.flash_attn_forward(q, k, v, bias, causal=causal)
    for p0 in range(0, planes, 100):
        part = [None if t is None else t[:, p0:p0 + 100].contiguous() for t in (q, k, v, bias)]
        o1, lse1 = ops.flash_attn_forward(*part, causal=causal)
        assert torch.equal(o[:, p0:p0 + 100], o1) and torch.equal(lse[:, p0:p0 + 100], lse1)


def test_reference_golden_vectors(ops):
    path = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "flash_attn_forward.json")
    with open(path) as f:
        cases = json.load(f)["cases"]
    for c in cases:
        shape = (c["B"], c["h"], c["L"], c["d"])
        f32 = lambda bits, shp: np.array(bits, dtype=np.uint32).view(np.float32).reshape(shp)  # noqa: E731
        bias = f32(c["bias"], (c["B"], c["h"], c["L"], c["L"])) if c["bias"] is not None else None
        got_o, got_lse = _run(ops, f32(c["q"], shape), f32(c["k"], shape), f32(c["v"], shape), bias,
                              causal=c["causal"], scale=c["scale"], eps=c["eps"], Bc=c["Bc"])
        _check(got_o, got_lse, f32(c["o"], shape), f32(c["lse"], shape[:3]))


def test_scale_eps_and_missing_lse(ops, oracle):
    rng = np.random.default_rng(3)
    q, k, v = [rng.standard_normal((1, 2, 50, 16)).astype(np.float32) for _ in range(3)]
    want_o, want_lse = oracle.flash_attn_forward(q, k, v, None, scale=0.3, eps=0.5)
    got_o, got_lse = _run(ops, q, k, v, scale=0.3, eps=0.5)
    _check(got_o, got_lse, want_o, want_lse)
    o, lse = ops.flash_attn_forward(_dev(q), _dev(k), _dev(v), scale=0.3, eps=0.5, want_lse=False)
    ops.synchronize()
    assert lse is None and np.array_equal(o.cpu().numpy(), got_o)


def test_masked_rows_and_the_masked_first_block(ops, oracle):
    rng = np.random.default_rng(4)
    B, h, L, d = 1, 2, 160, 32
    q, k, v = [rng.standard_normal((B, h, L, d)).astype(np.float32) for _ in range(3)]
    bias = rng.standard_normal((B, h, L, L)).astype(np.float32)
    bias[0, 0, 5, :] = -np.inf            # masked entirely
    bias[0, 0, 6, :64] = -np.inf          # the reference's first block (Bc = 64) masked: row poisoned
    bias[0, 0, 7, :63] = -np.inf          # one key of a 64-key first block survives; a 32-key first block does not
    bias[0, 1, 8, 64:] = -np.inf          # only the first block survives: ordinary row
    bias[0, 1, 9, :32] = -np.inf          # with Bc = 32 this row is poisoned, with 64 it is not
    for Bc in (64, 32):
        want_o, want_lse = oracle.flash_attn_forward(q, k, v, bias, Bc=Bc)
        assert np.isneginf(want_lse[0, 0, 5]) and np.isneginf(want_lse[0, 0, 6]) and np.isfinite(want_lse[0, 1, 8])
        assert np.isfinite(want_lse[0, 0, 7]) == (Bc == 64)
        assert np.isneginf(want_lse[0, 1, 9]) == (Bc == 32)
        got_o, got_lse = _run(ops, q, k, v, bias, Bc=Bc)
        _check(got_o, got_lse, want_o, want_lse)


def test_closed_forms_at_the_configured_sizes(ops):
    """Size-independent properties at the MSA-track shape (planes 824, L 256, d 32), where the oracle
    would take minutes: equal scores give the mean of V; V = 1 gives rows of 1; a per-row shift of the
    bias moves LSE by the shift and leaves O alone."""
    g = torch.Generator(device="cuda").manual_seed(5)
    B, h, L, d = 103, 8, 256, 32
    k = torch.randn(B, h, L, d, device="cuda", generator=g)
    v = torch.randn(B, h, L, d, device="cuda", generator=g)
    o, lse = ops.flash_attn_forward(torch.zeros_like(k), k, v, eps=0.0)
    mean = v.mean(dim=2, keepdim=True)
    assert float((o - mean).abs().max()) <= 1e-5
    assert float((lse - float(np.log(L))).abs().max()) <= 1e-5
    q = torch.randn(B, h, L, d, device="cuda", generator=g)
    o1, lse1 = ops.flash_attn_forward(q, k, torch.ones_like(v), eps=0.0)
    assert float((o1 - 1).abs().max()) <= 1e-5
    Bs, hs = 8, 8
    bias = torch.randn(Bs, hs, L, L, device="cuda", generator=g)
    shift = torch.randn(Bs, hs, L, 1, device="cuda", generator=g)
    qa, ka, va = q[:Bs].contiguous(), k[:Bs].contiguous(), v[:Bs].contiguous()
    oa, la = ops.flash_attn_forward(qa, ka, va, bias)
    ob, lb = ops.flash_attn_forward(qa, ka, va, bias + shift)
    assert float((oa - ob).abs().max()) <= 2e-5
    assert float((lb - la - shift[..., 0]).abs().max()) <= 2e-5
    # against torch's own softmax attention in float64 on a few planes
    s = torch.einsum("bhid,bhjd->bhij", qa.double(), ka.double()) / np.sqrt(d) + bias.double()
    want = torch.einsum("bhij,bhjd->bhid", torch.softmax(s, dim=-1), va.double())
    assert float((oa.double() - want).abs().max()) <= RTOL * float(want.abs().max())


def test_refused_arguments(ops):
    from proteinpredictmachinelearning_amd import cabi

    lib = cabi.load()
    x = torch.zeros(4 * 72, device="cuda")
    p = x.data_ptr()
    args = lambda d, ptr=p: (1, 1, 4, d, 0, 0.0, 1e-9, 64, ptr, p, p, None, p, None, None)  # noqa: E731
    assert lib.flash_attn_forward_hip(*args(72)) == 1          # d > 64 (src/backend/CUDABackend.cpp:457-463)
    assert lib.flash_attn_forward_hip(*args(6)) == 1           # d % 4 != 0
    assert lib.flash_attn_forward_hip(*args(8, p + 4)) == 1    # misaligned
    assert lib.flash_attn_forward_hip(1, 1, 0, 8, 0, 0.0, 1e-9, 64, p, p, p, None, p, None, None) == 1
    assert lib.flash_attn_forward_hip(1, 1, 4, 8, 0, 0.0, 1e-9, 64, None, p, p, None, p, None, None) == 1
    assert b"flash_attn_forward_hip" in lib.ppml_hip_last_error()


@pytest.mark.parametrize("B,h,L,d,causal,use_bias", [(1, 3, 103, 32, False, True), (2, 2, 256, 32, False, True),
                                                     (1, 2, 77, 20, True, False), (1, 1, 150, 64, False, True)])
@pytest.mark.parametrize("in_ld,out_ld", [(True, True), (True, False), (False, True)])
def test_layouts_without_the_bridges(ops, oracle, B, h, L, d, causal, use_bias, in_ld, out_ld):
    """Q, K, V handed over as (B,h,d,L) and / or O wanted as (B,h,d,L): the graph tensors on either side of the
    permutation copies the reference wraps around the node (ComputeGraphHelper.cpp:456-458, 483)."""
    rng = np.random.default_rng(L + 7 * d)
    q, k, v = [rng.standard_normal((B, h, L, d)).astype(np.float32) for _ in range(3)]
    bias = rng.standard_normal((B, h, L, L)).astype(np.float32) if use_bias else None
    want_o, want_lse = oracle.flash_attn_forward(q, k, v, bias, causal=causal)
    t = (lambda x: np.ascontiguousarray(x.transpose(0, 1, 3, 2))) if in_ld else (lambda x: x)
    o, lse = ops.flash_attn_forward(_dev(t(q)), _dev(t(k)), _dev(t(v)), _dev(bias), causal=causal, in_ld=in_ld, out_ld=out_ld)
    ops.synchronize()
    got_o = o.cpu().numpy()
    if out_ld:
        got_o = got_o.transpose(0, 1, 3, 2)
    _check(got_o, lse.cpu().numpy(), want_o, want_lse)


# ----------------------------------------------------------------------------- backward
def _check_grad(got, want, name):
    # inputs are O(1); a gradient that is exactly zero in exact arithmetic (a single key: dS = dP - D = 0) comes
    # out as rounding noise of size 1e-8, hence the floor of the scale
    scale = max(np.abs(want).max(), 1e-3)
    err = np.abs(got.astype(np.float64) - want).max() / scale
    assert err <= RTOL, f"{name} normwise {err:.3e}"


@pytest.mark.parametrize("B,h,L,d,causal,use_bias", [
    (1, 1, 1, 4, False, False), (2, 2, 37, 8, False, True), (1, 4, 103, 32, False, True), (1, 2, 128, 32, True, False),
    (1, 2, 160, 32, True, True),       # more rows than one LDS stage (128), causal: skipped chunks and tiles
    (2, 2, 256, 32, False, True), (1, 2, 70, 64, False, True), (1, 1, 150, 64, True, True), (1, 2, 45, 20, False, True),
])
def test_flash_attn_backward_matches_oracle(ops, oracle, B, h, L, d, causal, use_bias):
    rng = np.random.default_rng(7000 + 10 * L + d)
    q, k, v, do = [rng.standard_normal((B, h, L, d)).astype(np.float32) for _ in range(4)]
    bias = rng.standard_normal((B, h, L, L)).astype(np.float32) if use_bias else None
    if bias is not None and not causal and L > 4:
        bias[0, 0, 3, :] = -np.inf                  # a masked row: no gradient from it, zeros in its dbias row
    o, lse = oracle.flash_attn_forward(q, k, v, bias, causal=causal)
    want = oracle.flash_attn_backward(q, k, v, bias, o, do, lse, causal=causal)
    got = ops.flash_attn_backward(_dev(q), _dev(k), _dev(v), _dev(bias), _dev(o), _dev(do), _dev(lse), causal=causal)
    ops.synchronize()
    for g, w, name in zip(got, want, ("dQ", "dK", "dV", "dbias")):
        _check_grad(g.cpu().numpy(), w, name)
    db = got[3].cpu().numpy()
    assert (db[np.isneginf(lse)] == 0).all()        # rows without a visible key: exact zeros
    if bias is not None:
        assert (db[np.isneginf(bias) & ~np.isneginf(lse)[..., None]] == 0).all()    # masked keys of live rows
    if causal:
        assert (np.triu(db[0, 0], 1) == 0).all()


@pytest.mark.parametrize("planes,L,d,causal,use_bias", [
    (2, 31, 32, False, True), (2, 32, 8, False, False), (3, 33, 32, True, True),      # one key tile, whole and ragged
    (2, 129, 32, False, True), (2, 255, 24, False, True), (1, 256, 32, True, False),  # four waves' keys and one more, eight waves'
    (100, 257, 4, False, True), (97, 288, 32, True, True),                            # a second round of keys (dQ added to), ragged and whole
    (520, 40, 32, False, True),                                                       # more planes than work-groups: loads run on into the next plane
])
def test_flash_attn_backward_in_one_pass(ops, planes, L, d, causal, use_bias):
    """The one-pass kernel at the edges of its key tiles, rounds and plane lists, against the same gradients in binary64."""
    g = torch.Generator(device="cuda")
    g.manual_seed(L * 7 + d)
    q, k, v, do = (torch.randn(1, planes, L, d, device="cuda", generator=g) for _ in range(4))
    bias = torch.randn(1, planes, L, L, device="cuda", generator=g) if use_bias else None
    if use_bias:
        bias[0, :, 1, :] -= 200.0                   # a row whose LSE lies far below zero: a key past the matrix must not see exp(0 - LSE)
    o, lse = ops.flash_attn_forward(q, k, v, bias, causal=causal)
    got = ops.flash_attn_backward(q, k, v, bias, o, do, lse, causal=causal)
    Q, K, V, DO = (t[0].double() for t in (q, k, v, do))
    s = torch.matmul(Q, K.transpose(1, 2).contiguous()) / np.sqrt(d)
    if use_bias:
        s = s + bias[0].double()
    if causal:
        s = s.masked_fill(torch.ones(L, L, dtype=torch.bool, device="cuda").triu(1), float("-inf"))
    p = torch.softmax(s, -1)
    ds = p * (torch.matmul(DO, V.transpose(1, 2).contiguous()) - (DO * torch.matmul(p, V)).sum(-1, keepdim=True))
    want = (torch.matmul(ds, K) / np.sqrt(d), torch.matmul(ds.transpose(1, 2).contiguous(), Q) / np.sqrt(d),
            torch.matmul(p.transpose(1, 2).contiguous(), DO), ds)
    for x, w, name in zip(got, want, ("dQ", "dK", "dV", "dbias")):
        x, w = x[0].cpu().numpy(), w.cpu().numpy()
        _check_grad(x, w, name)        # (logits near -200 carry 2^-16 of rounding, exp(LSE - ...) as much: 3e-5)


# beyond 256 rows in few planes: two kernels; either side of the numbers of planes from which one pass takes over (3/8 and
# 1/2 of 256 CUs with a bias, 3/5 of them without)
@pytest.mark.parametrize("planes,L,d,causal,use_bias", [
    (2, 257, 32, False, True), (2, 300, 20, True, True), (3, 300, 32, False, False), (1, 520, 32, True, False),
    (95, 257, 32, False, True), (96, 257, 32, False, True), (95, 260, 8, True, False), (96, 260, 8, True, False),
    (153, 257, 16, False, False), (154, 257, 16, False, False), (127, 513, 8, False, True), (128, 513, 8, False, True),
])
def test_flash_attn_backward_of_long_planes(ops, planes, L, d, causal, use_bias):
    test_flash_attn_backward_in_one_pass(ops, planes, L, d, causal, use_bias)


# one pass for the whole set, two kernels for most of the others: rounds of 256 keys, ragged tiles, the features' remainder,
# and enough planes for the exceptions (256 x 150, 200 x 260 causal, 200 x 400)
@pytest.mark.parametrize("planes,L,d,causal,use_bias", [
    (2, 31, 32, False, True), (3, 103, 20, True, True), (2, 128, 4, False, False), (2, 160, 32, False, True), (2, 255, 24, True, False),
    (256, 150, 32, False, True), (200, 260, 32, True, True), (200, 400, 12, False, True), (160, 300, 32, False, False),
    (300, 256, 32, False, True), (130, 520, 32, False, True), (2, 300, 32, False, True),
])
def test_flash_attn_backward_subsets_have_the_bits_of_the_whole(ops, planes, L, d, causal, use_bias):
    g = torch.Generator(device="cuda")
    g.manual_seed(3 * L + d)
    q, k, v, do = (torch.randn(1, planes, L, d, device="cuda", generator=g) for _ in range(4))
    bias = torch.randn(1, planes, L, L, device="cuda", generator=g) if use_bias else None
    o, lse = ops.flash_attn_forward(q, k, v, bias, causal=causal)
    names = ("dq", "dk", "dv", "dbias")
    whole = ops.flash_attn_backward(q, k, v, bias, o, do, lse, causal=causal, want=names)
    for mask in range(1, 15):
        want = tuple(n for i, n in enumerate(names) if mask >> i & 1)
        got = ops.flash_attn_backward(q, k, v, bias, o, do, lse, causal=causal, want=want)
        for n, x, w in zip(names, got, whole):
            assert (x is not None) == (n in want)
            assert x is None or torch.equal(x, w), (want, n)


# dQ and dbias on the memory of Q (dO, O) and the bias: a query's row and a pair's bias are read before they are written, in
# one round of keys (256 x 150), in rounds (causal 200 x 260, 200 x 400) and where the rows kernel is the rule (3 x 300)
@pytest.mark.parametrize("planes,L,d,causal", [(256, 150, 32, False), (200, 260, 32, True), (200, 400, 16, False), (3, 300, 32, True)])
def test_flash_attn_backward_rows_in_place(ops, planes, L, d, causal):
    from proteinpredictmachinelearning_amd import cabi

    g = torch.Generator(device="cuda")
    g.manual_seed(L)
    q, k, v, do = (torch.randn(1, planes, L, d, device="cuda", generator=g) for _ in range(4))
    bias = torch.randn(1, planes, L, L, device="cuda", generator=g)
    o, lse = ops.flash_attn_forward(q, k, v, bias, causal=causal)
    dq, _, _, db = ops.flash_attn_backward(q, k, v, bias, o, do, lse, causal=causal, want=("dq", "dbias"))
    for name in ("q", "o", "do"):
        x = dict(q=q.clone(), o=o.clone(), do=do.clone())
        out_b = bias.clone()
        rc = cabi.load().flash_attn_backward_hip(1, planes, L, d, int(causal), 0.0, x["q"].data_ptr(), k.data_ptr(), v.data_ptr(),
                                                 out_b.data_ptr(), x["o"].data_ptr(), x["do"].data_ptr(), lse.data_ptr(),
                                                 x[name].data_ptr(), None, None, out_b.data_ptr(), torch.cuda.current_stream().cuda_stream)
        assert rc == 0
        assert torch.equal(x[name], dq) and torch.equal(out_b, db), name


# one pass and two kernels (few long planes, 64 features), one round of keys and two, whole and ragged tiles
@pytest.mark.parametrize("planes,L,d,use_bias", [(2, 70, 32, True), (3, 160, 24, False), (2, 256, 32, True), (97, 300, 32, True), (97, 288, 8, False),
                                                 (2, 300, 32, True), (2, 150, 64, True)])
def test_causal_backward_keeps_what_a_query_does_not_see_out_of_its_gradients(ops, planes, L, d, use_bias):
    """A position whose operands are not finite: the tiles of 32 rows before it (K, V: queries that do not see it) and
    behind it (Q, dO: keys it does not see) keep the bits of the clean call."""
    g = torch.Generator(device="cuda")
    g.manual_seed(L + d)
    q, k, v, do = (torch.randn(1, planes, L, d, device="cuda", generator=g) for _ in range(4))
    bias = torch.randn(1, planes, L, L, device="cuda", generator=g) if use_bias else None
    o, lse = ops.flash_attn_forward(q, k, v, bias, causal=True)
    clean = ops.flash_attn_backward(q, k, v, bias, o, do, lse, causal=True)
    masked = torch.ones(L, L, dtype=torch.bool, device="cuda").triu(1)
    for at in (L - 2, 40):
        first, behind = at // 32 * 32, at // 32 * 32 + 32
        for name in ("q", "k", "v", "do"):
            for value in (float("nan"), float("inf")):
                x = dict(q=q, k=k, v=v, do=do)
                x[name] = x[name].clone()
                x[name][:, :, at] = value
                o2, lse2 = ops.flash_attn_forward(x["q"], x["k"], x["v"], bias, causal=True)
                dq, dk, dv, db = ops.flash_attn_backward(x["q"], x["k"], x["v"], bias, o2, x["do"], lse2, causal=True)
                what = f"{name} = {value} at {at}"
                if name in ("k", "v"):
                    assert torch.equal(dq[:, :, :first], clean[0][:, :, :first]), what
                else:
                    assert torch.equal(dk[:, :, behind:], clean[1][:, :, behind:]) and torch.equal(dv[:, :, behind:], clean[2][:, :, behind:]), what
                if use_bias:
                    assert torch.equal(db[:, :, :first], clean[3][:, :, :first]) and not db[:, :, masked].any(), what


def test_flash_attn_backward_subsets_and_determinism(ops, oracle):
    rng = np.random.default_rng(77)
    B, h, L, d = 1, 3, 90, 32
    q, k, v, do = [rng.standard_normal((B, h, L, d)).astype(np.float32) for _ in range(4)]
    bias = rng.standard_normal((B, h, L, L)).astype(np.float32)
    o, lse = oracle.flash_attn_forward(q, k, v, bias)
    args = [_dev(x) for x in (q, k, v, bias, o, do, lse)]
    full = [t.cpu().numpy() for t in ops.flash_attn_backward(*args)]
    again = [t.cpu().numpy() for t in ops.flash_attn_backward(*args)]
    for a, b in zip(full, again):
        assert np.array_equal(a, b)                 # one owner per output element: no atomics, bit-stable
    dq, dk, dv, db = ops.flash_attn_backward(*args, want=("dk",))
    assert dq is None and dv is None and db is None and np.array_equal(dk.cpu().numpy(), full[1])
    dq, dk, dv, db = ops.flash_attn_backward(*args, want=("dq", "dv"))
    assert dk is None and db is None and np.array_equal(dq.cpu().numpy(), full[0]) and np.array_equal(dv.cpu().numpy(), full[2])
    dq, dk, dv, db = ops.flash_attn_backward(*args, want=("dbias",))
    assert np.array_equal(db.cpu().numpy(), full[3])
    # the scale argument: caller's head dimension instead of d
    o2, lse2 = oracle.flash_attn_forward(q, k, v, bias, scale=0.5)
    want = oracle.flash_attn_backward(q, k, v, bias, o2, do, lse2, scale=0.5)
    got = ops.flash_attn_backward(*args[:4], _dev(o2), args[5], _dev(lse2), scale=0.5)
    for g, w, name in zip(got, want, ("dQ", "dK", "dV", "dbias")):
        _check_grad(g.cpu().numpy(), w, name)


def test_backward_reference_golden_vectors(ops):
    path = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "flash_attn_forward.json")
    with open(path) as f:
        cases = json.load(f)["backward_cases"]
    for c in cases:
        shape = (c["B"], c["h"], c["L"], c["d"])
        sq = (c["B"], c["h"], c["L"], c["L"])
        f32 = lambda bits, shp: np.array(bits, dtype=np.uint32).view(np.float32).reshape(shp)  # noqa: E731
        bias = f32(c["bias"], sq) if c["bias"] is not None else None
        got = ops.flash_attn_backward(_dev(f32(c["q"], shape)), _dev(f32(c["k"], shape)), _dev(f32(c["v"], shape)), _dev(bias),
                                      _dev(f32(c["o"], shape)), _dev(f32(c["do"], shape)), _dev(f32(c["lse"], shape[:3])), causal=c["causal"])
        ops.synchronize()
        for g, key, shp in zip(got, ("dq", "dk", "dv", "dbias"), (shape, shape, shape, sq)):
            _check_grad(g.cpu().numpy(), f32(c[key], shp), key)


# rows that end inside a tile of 32 keys, on one, and one past it; one work-group per plane and several, four waves and eight; every instance
@pytest.mark.parametrize("L", [3, 33, 50, 64, 103, 131, 161, 257])
@pytest.mark.parametrize("d", [4, 32, 48])
@pytest.mark.parametrize("causal", [False, True])
def test_forward_keeps_to_its_own_rows(ops, L, d, causal):
    """Bias is read in pieces of sixteen bytes without a test of the row's end: what the next row, or the next plane, begins with must
    not reach a row's result.  A row of NaN, and a plane of infinities, leave every other row the bits it has without them."""
    torch.manual_seed(L * d)
    planes = 3
    for in_ld in (False, True):
        shape = (1, planes, d, L) if in_ld else (1, planes, L, d)
        q, k, v = (torch.randn(shape, device="cuda") for _ in range(3))
        bias = torch.randn(1, planes, L, L, device="cuda")
        clean, lse = ops.flash_attn_forward(q, k, v, bias, causal=causal, in_ld=in_ld)
        bad = bias.clone()
        r = L // 2
        bad[0, 0, r] = float("nan")
        bad[0, 2] = float("-inf")
        out, lse2 = ops.flash_attn_forward(q, k, v, bad, causal=causal, in_ld=in_ld)
        keep = torch.ones(planes, L, dtype=torch.bool, device="cuda")
        keep[0, r] = False
        keep[2] = False
        assert torch.equal(out[0][keep].view(torch.int32), clean[0][keep].view(torch.int32))
        assert torch.equal(lse2[0][keep].view(torch.int32), lse[0][keep].view(torch.int32))


@pytest.mark.parametrize("L", [3, 33, 50, 103, 131])
@pytest.mark.parametrize("d", [4, 32, 48])
@pytest.mark.parametrize("causal", [False, True])
def test_backward_keeps_to_its_own_rows(ops, L, d, causal):
    """The rows kernel reads the bias like the forward: a row of NaN leaves dQ and dbias of every other row the bits they have without it."""
    torch.manual_seed(L + d)
    planes = 3
    q, k, v, do = (torch.randn(1, planes, L, d, device="cuda") for _ in range(4))
    bias = torch.randn(1, planes, L, L, device="cuda")
    o, lse = ops.flash_attn_forward(q, k, v, bias, causal=causal)
    bad = bias.clone()
    r = L // 2
    bad[0, 0, r] = float("nan")
    want = ("dq", "dbias")
    dq, _, _, db = ops.flash_attn_backward(q, k, v, bias, o, do, lse, causal=causal, want=want)
    dq2, _, _, db2 = ops.flash_attn_backward(q, k, v, bad, o, do, lse, causal=causal, want=want)
    keep = torch.ones(planes, L, dtype=torch.bool, device="cuda")
    keep[0, r] = False
    assert torch.equal(dq[0][keep].view(torch.int32), dq2[0][keep].view(torch.int32))
    assert torch.equal(db[0][keep].view(torch.int32), db2[0][keep].view(torch.int32))
