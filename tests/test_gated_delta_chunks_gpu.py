"""The gated delta rule in chunks of 64 tokens against the recurrence in 64 bits and against blocks of 16 tokens: lengths around whole
chunks and tiles, head sizes with and without whole 16-byte pieces, shared heads, states that go on, decays that vanish, prompts
longer than the workspace holds, and the shapes that stay with the blocks."""
import pytest
import torch

from conftest import rel_l2

pytestmark = pytest.mark.gpu
# fp32 sums over 64 tokens and 128 channels, errors of random signs that the recurrence contracts: below 32 roundings of 2^-24
TOL = 2e-6


def make(seed, B, L, H, G, d, dv, dtype, strong=False, pad=0):
    g = torch.Generator().manual_seed(seed)
    n = 2 * G * d + H * dv + pad
    x = torch.nn.functional.silu(torch.randn(B, L, n, generator=g)).to(dtype)
    ab = (torch.randn(B, L, 2 * H, generator=g) * (4 if strong else 1)).to(dtype)
    return x, ab, (torch.randn(H, generator=g) + (3 if strong else -2)).to(dtype), torch.randn(H, generator=g).to(dtype)


def reference(x, ab, a_log, dt_bias, H, G, d, dv, S=None):
    B, L = x.shape[:2]
    x, ab = x.double(), ab.double()
    unit = lambda t: t / (t.square().sum(-1, keepdim=True) + 1e-6).sqrt()
    share = lambda t: t.repeat_interleave(H // G, 2)
    q = share(unit(x[..., :G * d].view(B, L, G, d)) * d ** -0.5)
    k = share(unit(x[..., G * d:2 * G * d].view(B, L, G, d)))
    v = x[..., 2 * G * d:2 * G * d + H * dv].view(B, L, H, dv)
    decay = torch.exp(-torch.exp(a_log.double()) * torch.nn.functional.softplus(ab[..., :H] + dt_bias.double()))
    beta = torch.sigmoid(ab[..., H:])
    S = torch.zeros(B, H, d, dv, dtype=torch.float64, device=x.device) if S is None else S.double()
    out = torch.empty(B, L, H, dv, dtype=torch.float64, device=x.device)
    for t in range(L):
        S = S * decay[:, t, :, None, None]
        u = beta[:, t, :, None] * (v[:, t] - (k[:, t, :, None] @ S)[:, :, 0])
        S = S + k[:, t, :, :, None] * u[:, :, None]
        out[:, t] = (q[:, t, :, None] @ S)[:, :, 0]
    return out, S


def run(case, H, G, d, dv, state, fresh=True):
    from based_amd import ops

    x, ab, a_log, dt_bias = case
    o = ops.gated_delta_scan(x[..., :G * d], x[..., G * d:2 * G * d], x[..., 2 * G * d:2 * G * d + H * dv], ab[..., :H], ab[..., H:], a_log,
                             dt_bias, state, H, G, fresh)
    return o, state[..., :dv]


def in_chunks(B, L, H, d, dv):
    from based_amd import _lib

    return _lib.lib().based_gated_delta_scan_work(B, L, H, d, dv) > 0


def empty_state(B, H, d, dv, dev):
    return torch.full((B, H, d, (dv + 3) // 4 * 4), float("nan"), device=dev)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("L", [256, 257, 271, 272, 319, 320, 321, 500])
def test_lengths(dev, dtype, L):
    case = [t.to(dev) for t in make(L, 2, L, 3, 3, 64, 48, dtype)]
    assert in_chunks(2, L, 3, 64, 48)
    o, S = run(case, 3, 3, 64, 48, empty_state(2, 3, 64, 48, dev))
    ref, S_ref = reference(*case, 3, 3, 64, 48)
    assert rel_l2(o, ref) < TOL and rel_l2(S, S_ref) < TOL


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("strong", [False, True])
@pytest.mark.parametrize("H,G,d,dv,pad", [(4, 2, 16, 16, 0), (2, 1, 18, 10, 3), (3, 3, 20, 70, 1), (1, 1, 64, 256, 0), (6, 2, 72, 36, 0), (4, 4, 128, 128, 8)])
def test_heads(dev, dtype, strong, H, G, d, dv, pad):
    L = 300
    case = [t.to(dev) for t in make(d, 1, L, H, G, d, dv, dtype, strong, pad)]
    assert in_chunks(1, L, H, d, dv)
    state = empty_state(1, H, d, dv, dev)
    o, S = run(case, H, G, d, dv, state)
    ref, S_ref = reference(*case, H, G, d, dv)
    assert rel_l2(o, ref) < TOL and rel_l2(S, S_ref) < TOL
    # the same tokens again behind that state
    o, S = run(case, H, G, d, dv, state, fresh=False)
    ref, S_ref = reference(*case, H, G, d, dv, S_ref)
    assert rel_l2(o, ref) < TOL and rel_l2(S, S_ref) < TOL


def test_spans_of_a_long_prompt(dev):
    """More chunks than the workspace holds at once."""
    from based_amd import _lib

    B, L, H, d, dv = 4, 1990, 16, 128, 128
    chunks = (L + 63) // 64
    floats = _lib.lib().based_gated_delta_scan_work(B, L, H, d, dv)
    assert 0 < floats <= 64 << 20 and floats < _lib.lib().based_gated_delta_scan_work(B, 64 * 8, H, d, dv) // 8 * chunks
    case = [t.to(dev) for t in make(3, B, L, H, H, d, dv, torch.bfloat16)]
    o, S = run(case, H, H, d, dv, empty_state(B, H, d, dv, dev))
    ref, S_ref = reference(*case, H, H, d, dv)
    assert rel_l2(o, ref) < TOL and rel_l2(S, S_ref) < TOL


@pytest.mark.parametrize("B,L,H,d,dv", [(1, 255, 4, 64, 64), (1, 300, 2, 129, 64), (5, 256, 13, 64, 64), (1, 256, 64, 64, 132)])
def test_shapes_that_stay_with_blocks(dev, B, L, H, d, dv):
    assert not in_chunks(B, L, H, d, dv)
    case = [t.to(dev) for t in make(4, B, L, H, H, d, dv, torch.float32)]
    o, S = run(case, H, H, d, dv, empty_state(B, H, d, dv, dev))
    ref, S_ref = reference(*case, H, H, d, dv)
    assert rel_l2(o, ref) < 3e-6 and rel_l2(S, S_ref) < 3e-6


def test_rows_of_no_whole_pieces(dev):
    """Heads of more than 64 channels whose rows start anywhere: blocks."""
    H, d, dv, L = 2, 96, 32, 300
    x, ab, a_log, dt_bias = (t.to(dev) for t in make(6, 1, L, H, H, d, dv, torch.float32, pad=1))
    state = empty_state(1, H, d, dv, dev)
    wide = torch.zeros(1, L, x.shape[-1] + 2, device=dev)
    wide[..., 1:-1] = x
    o, S = run((wide[..., 1:], ab, a_log, dt_bias), H, H, d, dv, state)
    ref, S_ref = reference(x, ab, a_log, dt_bias, H, H, d, dv)
    assert rel_l2(o, ref) < 3e-6 and rel_l2(S, S_ref) < 3e-6


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("scale", [1e-12, 1e17, 1e18])
def test_long_and_short_queries(dev, dtype, scale):
    """Queries and keys whose squares' sum fits 32 bits and, times the head size, does not; and those that the constant beside it hides."""
    L, H, d, dv = 257, 2, 128, 32
    case = [t.to(dev) for t in make(8, 1, L, H, H, d, dv, dtype)]
    case[0][..., :2 * H * d] *= scale
    assert in_chunks(1, L, H, d, dv)
    o, S = run(case, H, H, d, dv, empty_state(1, H, d, dv, dev))
    ref, S_ref = reference(*case, H, H, d, dv)
    assert rel_l2(o, ref) < TOL and rel_l2(S, S_ref) < TOL


@pytest.mark.parametrize("B,H,d,dv,first", [(1, 4, 16, 16, 4), (4, 8, 16, 64, 8), (4, 8, 64, 128, 4), (8, 8, 64, 128, 6), (2, 8, 64, 512, 7),
                                            (4, 8, 96, 256, 10), (8, 8, 96, 128, None), (1, 8, 128, 128, 4), (2, 8, 128, 128, 5),
                                            (8, 8, 128, 128, 4), (2, 8, 128, 256, 7)])
def test_where_chunks_begin(dev, B, H, d, dv, first):
    """The first whole number of chunks that goes in chunks, and a token less: the same numbers on both sides of the line."""
    edge = 64 * (first or 12)
    for L in (edge - 1, edge):
        assert in_chunks(B, L, H, d, dv) == (first is not None and L == edge)
        case = [t.to(dev) for t in make(L, B, L, H, H, d, dv, torch.float32)]
        o, S = run(case, H, H, d, dv, empty_state(B, H, d, dv, dev))
        ref, S_ref = reference(*case, H, H, d, dv)
        assert rel_l2(o, ref) < 3e-6 and rel_l2(S, S_ref) < 3e-6  # (the tolerance of the blocks)


def test_batch_stride_of_one_sequence(dev):
    """The stride of a batch of one is any number."""
    H, d, dv, L = 2, 96, 32, 400
    x, *gates = (t.to(dev) for t in make(6, 1, L, H, H, d, dv, torch.bfloat16))
    x = x.as_strided(x.shape, (x.stride(0) + 1, x.stride(1), 1))
    o, S = run((x, *gates), H, H, d, dv, empty_state(1, H, d, dv, dev))
    ref, S_ref = reference(x, *gates, H, H, d, dv)
    assert rel_l2(o, ref) < TOL and rel_l2(S, S_ref) < TOL


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("d,dv", [(64, 64), (128, 40)])
@pytest.mark.parametrize("scale", [1e-24, 1e24])
def test_parts_of_small_and_large_values(dev, dtype, d, dv, scale):
    """32 bits of a state and of values whose smallest parts (2^-16 of them) are near the ends of the format, an element of 64 in 1,000 times
    the others; states that go on."""
    L, H = 330, 3
    x, *gates = make(9, 2, L, H, H, d, dv, dtype)
    x[..., 2 * H * d:] *= scale
    x[..., 2 * H * d::64] *= 1000
    case = [t.to(dev) for t in (x, *gates)]
    assert in_chunks(2, L, H, d, dv)
    state = empty_state(2, H, d, dv, dev)
    S_ref = None
    for fresh in (True, False):
        o, S = run(case, H, H, d, dv, state, fresh=fresh)
        ref, S_ref = reference(*case, H, H, d, dv, S_ref)
        # (norms of 1e-24 have no squares in 32 bits)
        assert rel_l2(o.double() / scale, ref / scale) < TOL and rel_l2(S.double() / scale, S_ref / scale) < TOL


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("scale", [1e-32, 3e37])
def test_ends_of_the_range_of_the_parts(dev, dtype, scale):
    """The smallest and the largest values that keep all of their 24 bits."""
    L, H, d, dv = 330, 3, 64, 64
    x, *gates = make(9, 2, L, H, H, d, dv, torch.float32)
    x[..., 2 * H * d:] *= scale
    case = [t.to(dtype).to(dev) for t in (x, *gates)]
    assert in_chunks(2, L, H, d, dv)
    o, S = run(case, H, H, d, dv, empty_state(2, H, d, dv, dev))
    ref, S_ref = reference(*case, H, H, d, dv)
    assert rel_l2(o.double() / scale, ref / scale) < TOL and rel_l2(S.double() / scale, S_ref / scale) < TOL


@pytest.mark.parametrize("B,L,H,d,dv,chunks", [(5, 256, 13, 64, 64, True), (13, 257, 5, 128, 128, True), (8, 512, 16, 64, 128, True),
                                               (8, 513, 16, 64, 128, False), (7, 300, 13, 80, 64, False), (43, 256, 3, 64, 64, False),
                                               (4, 256, 16, 128, 256, True), (4, 257, 12, 18, 52, True), (4, 511, 16, 16, 128, False),
                                               (4, 512, 16, 16, 128, True), (4, 256, 16, 32, 252, False), (3, 320, 16, 32, 256, True)])
def test_many_heads(dev, B, L, H, d, dv, chunks):
    """Many heads, and few channels: chunks in bf16 where they are the faster form, blocks in fp32 and in front of and behind it."""
    from based_amd import _lib

    x, ab, a_log, dt_bias = (t.to(dev) for t in make(B + L, B, L, H, H, d, dv, torch.bfloat16))
    at = lambda dtype: _lib.lib().based_gated_delta_scan_work_as(x.data_ptr(), x.data_ptr(), B, L, H, d, dv, *x.stride()[:2], dtype) > 0
    assert at(_lib.BASED_BF16) == chunks and not at(_lib.BASED_F32) and not in_chunks(B, L, H, d, dv)
    got, S = run((x, ab, a_log, dt_bias), H, H, d, dv, empty_state(B, H, d, dv, dev))
    want, T = reference(x, ab, a_log, dt_bias, H, H, d, dv)
    tol = TOL if chunks else 3e-6  # (blocks: as above)
    assert rel_l2(got, want) < tol and rel_l2(S, T) < tol


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("d,dv", [(64, 64), (128, 40)])
@pytest.mark.parametrize("what", ["value", "key", "gate"])
@pytest.mark.parametrize("at", [16, 20, 31, 40, 63, 64 + 50, 299])
def test_a_number_that_is_none(dev, dtype, d, dv, what, at):
    """A value, a key or a gate that is not finite stays out of the tokens in front of its tile of 16, of the other value channels and of the other
    heads, to the last bit: products take 32 tokens at a time, and zero times infinity is no zero."""
    B, L, H = 2, 300, 3
    clean = [t.to(dev) for t in make(5, B, L, H, H, d, dv, dtype)]
    assert in_chunks(B, L, H, d, dv)
    want, S_want = run(clean, H, H, d, dv, empty_state(B, H, d, dv, dev))
    for bad in (float("nan"), float("inf")):
        x, ab = clean[0].clone(), clean[1].clone()
        if what == "gate":
            if bad == float("inf"):
                continue  # (a gate of one)
            ab[1, at, H + 1] = bad
        else:
            x[1, at, (H * d + d + 5) if what == "key" else (2 * H * d + dv + 5)] = bad
        o, S = run((x, ab, *clean[2:]), H, H, d, dv, empty_state(B, H, d, dv, dev))
        assert not o[1, at, 1, 5].isfinite() and not S[1, 1, :, 5].isfinite().any()
        free = torch.ones(B, L, H, dv, dtype=torch.bool, device=dev)
        free[1, at // 16 * 16:, 1, slice(5, 6) if what == "value" else slice(None)] = False
        assert torch.equal(o[free], want[free])
        kept = torch.ones_like(S, dtype=torch.bool)
        kept[1, 1, :, slice(5, 6) if what == "value" else slice(None)] = False
        assert torch.equal(S[kept], S_want[kept])


@pytest.mark.parametrize("B,L,H,d,dv,chunks", [(8, 1025, 16, 116, 32, True), (8, 1024, 16, 112, 32, True), (8, 1025, 16, 112, 32, False), (7, 1025, 16, 104, 48, True),
                                               (5, 300, 16, 96, 64, True), (27, 300, 3, 96, 64, False), (27, 300, 3, 72, 16, True), (8, 513, 15, 64, 128, True),
                                               (5, 300, 16, 48, 128, True), (27, 300, 3, 48, 128, False), (4, 1024, 16, 48, 256, True),
                                               (4, 1025, 16, 48, 256, False), (4, 1025, 16, 16, 128, False), (6, 1025, 8, 16, 160, True)])
def test_both_sides_of_the_lines_for_bf16(dev, B, L, H, d, dv, chunks):
    """Every line of the rule for bf16: channels, heads, workgroups, and prompts that are long for them."""
    test_many_heads(dev, B, L, H, d, dv, chunks)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,L,H,d,dv", [(4, 2500, 16, 64, 64), (4, 1600, 16, 128, 128)])
def test_work_space_of_a_long_prompt(dev, dtype, B, L, H, d, dv):
    """In a work space of exactly what was asked for, whatever lies behind it stays as it is; several launch pairs."""
    from based_amd import _lib, ops

    x, ab, a_log, dt_bias = (t.to(dev) for t in make(11, B, L, H, H, d, dv, dtype))
    lib, s = _lib.lib(), ops._stream_ptr(x)
    q, k, v, a, b = (x[..., :H * d], x[..., H * d:2 * H * d], x[..., 2 * H * d:], ab[..., :H], ab[..., H:])
    code = _lib.BASED_BF16 if dtype == torch.bfloat16 else _lib.BASED_F32
    floats = lib.based_gated_delta_scan_work_as(q.data_ptr(), k.data_ptr(), B, L, H, d, dv, *x.stride()[:2], code)
    assert 0 < floats <= 48 << 20
    room = torch.full((floats + 4096,), 7.0, device=dev)
    o, S = torch.empty(B, L, H, dv, device=dev), torch.empty(B, H, d, dv, device=dev)
    _lib.check(lib.based_gated_delta_scan_chunks(q.data_ptr(), k.data_ptr(), v.data_ptr(), a.data_ptr(), b.data_ptr(), a_log.data_ptr(), dt_bias.data_ptr(),
                                                 S.data_ptr(), room.data_ptr(), o.data_ptr(), B, L, H, H, d, dv, dv, *x.stride()[:2], *ab.stride()[:2], 1, code, s))
    want, T = run((x, ab, a_log, dt_bias), H, H, d, dv, empty_state(B, H, d, dv, dev))
    assert torch.equal(o, want) and torch.equal(S, T) and (room[floats:] == 7).all()
