"""The gated recurrence over portions whose length, block width and rows put its 16-token, 64-token and 64-channel edges everywhere."""
import pytest
import torch

from oracle import sozilix_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("L,W,blocks,rows,carry", [
    (1, 64, 1, "own", True), (15, 8, 2, "own", True), (16, 68, 1, "own", False), (17, 60, 1, "shifted", True), (63, 192, 3, "sliced", True),
    (64, 33, 1, "own", True), (65, 260, 2, "sliced", False), (577, 72, 1, "own", True), (2049, 16, 2, "shifted", True),
    (130, 136, 1, "over u", True), (200, 66, 2, "over y", True), (1000, 8, 1, "beside u", False), (6000, 1024, 16, "own", True)])
def test_rglru_segments(dev, dtype, L, W, blocks, rows, carry):
    """`rows`: tensors of their own; rows that start off an aligned address; slices of wider rows; an output in the place of an input
    or in the same rows."""
    from based_amd import ops

    B, n = 3, W // blocks
    g = torch.Generator().manual_seed(L * 131 + W)
    u, y = (torch.randn(B, L, W, generator=g).to(dtype) for _ in range(2))
    ra, ri = ((torch.randn(blocks, n, n, generator=g) * n ** -0.5).to(dtype) for _ in range(2))
    rb, ib = (torch.randn(W, generator=g).to(dtype) for _ in range(2))
    lam = (2 * torch.randn(W, generator=g) - 3).to(dtype)
    start = torch.randn(B, W, generator=g)

    def placed(t):
        if rows == "shifted":
            return torch.empty(B, L, W + 5, dtype=dtype, device=dev)[..., 3:3 + W].copy_(t)
        if rows == "sliced":
            return torch.empty(B, L, 2 * W + 8, dtype=dtype, device=dev)[..., W:2 * W].copy_(t)
        return t.to(dev)

    ud, yd, out = placed(u), placed(y), placed(torch.full((B, L, W), float("nan"), dtype=dtype))
    if rows == "beside u":
        both = torch.full((B, L, 2 * W), float("nan"), dtype=dtype, device=dev)
        ud, out = both[..., :W].copy_(u), both[..., W:]
    out = {"over u": ud, "over y": yd}.get(rows, out)
    state = start.to(dev) if carry else torch.full((B, W), float("nan"), device=dev)
    ops.rglru_prefill(ud, yd, *(t.to(dev) for t in (ra, rb, ri, ib, lam)), state, 8.0, fresh=not carry, out=out)
    # in 64 bits; a start state decays as a zero-input sequence does: the recurrence is linear in (u i sqrt, S)
    zr = torch.einsum("blkn,kmn->blkm", u.double().view(B, L, blocks, n), ra.double()).reshape(B, L, W) + rb.double()
    zi = torch.einsum("blkn,kmn->blkm", u.double().view(B, L, blocks, n), ri.double()).reshape(B, L, W) + ib.double()
    log_a = -8.0 * torch.sigmoid(zr) * torch.nn.functional.softplus(lam.double())
    x = torch.sqrt(-torch.expm1(2 * log_a)) * torch.sigmoid(zi) * u.double()
    S, ref = start.double() if carry else torch.zeros(B, W, dtype=torch.float64), []
    for t in range(L):
        S = log_a[:, t].exp() * S + x[:, t]
        ref.append(S * O.gelu_tanh(y[:, t].double()))
    ref = torch.stack(ref, 1)
    # fp32: a dozen roundings of 2^-24 each through gates, decays and the scan; bf16 outputs add half of 2^-8 each
    rel = lambda a, b: ((a.double().cpu() - b).norm() / b.norm()).item()  # noqa: E731
    assert rel(state, S) < 2e-6, rel(state, S)
    assert rel(out, ref) < (2e-6 if dtype == torch.float32 else 2.5e-3), rel(out, ref)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("W,shift", [(72, 0), (72, 8), (72, -3), (33, 0), (33, 1), (128, -128), (128, 128), (120, 128)])
def test_outputs_in_the_rows_of_the_input(dev, dtype, W, shift):
    """An output `shift` columns from the input in the same rows (over it, partly over it, beside it) is what it is on its own."""
    from based_amd import ops

    B, L = 2, 70
    g = torch.Generator().manual_seed(W + shift)
    rnd = lambda *s: torch.randn(*s, generator=g).to(dtype).to(dev)  # noqa: E731
    both = rnd(B, L, 3 * 128)
    u, y, gates = both[..., 128:128 + W], rnd(B, L, W), (rnd(1, W, W) * W ** -0.5, rnd(W), rnd(1, W, W) * W ** -0.5, rnd(W), rnd(W) - 3)
    want, s0, s1 = torch.empty(B, L, W, dtype=dtype, device=dev), torch.zeros(B, W, device=dev), torch.zeros(B, W, device=dev)
    ops.rglru_prefill(u.clone(), y, *gates, s0, 8.0, True, out=want)
    outside = both.clone()
    out = both[..., 128 + shift:128 + shift + W]
    ops.rglru_prefill(u, y, *gates, s1, 8.0, True, out=out)
    assert torch.equal(out, want) and torch.equal(s0, s1)
    outside[..., 128 + shift:128 + shift + W] = want
    assert torch.equal(both, outside)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("L,W,blocks", [(70, 40, 40), (66, 14, 7), (130, 15, 5), (65, 96, 24), (64, 48, 4), (100, 100, 1), (129, 65, 1)])
def test_narrow_blocks(dev, dtype, L, W, blocks):
    """Tiles with few live channels, of whole pieces and element by element."""
    test_rglru_segments(dev, dtype, L, W, blocks, "own", True)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("L", [1, 3, 15, 16, 17, 20, 31, 32, 33])
@pytest.mark.parametrize("W,blocks,rows,carry", [(64, 1, "own", True), (512, 2, "sliced", False), (144, 2, "shifted", True), (33, 1, "own", True)])
def test_short_prompts(dev, dtype, L, W, blocks, rows, carry):
    """Segments of one and of two 16-token tiles: rows in whole pieces and not, one round of the contraction and several."""
    test_rglru_segments(dev, dtype, L, W, blocks, rows, carry)


@pytest.mark.parametrize("L", [4095, 4096, 4097, 4160, 4161, 8192, 8193, 12500])
def test_groups_of_segments(dev, L):
    """Lengths around one, two and three groups of 64 segments."""
    test_rglru_segments(dev, torch.float32, L, 20, 1, "own", True)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("over", [False, True])
@torch.inference_mode()  # (torch keeps its generator's graph state in the mode of the process's first recording)
def test_replays(dev, dtype, over):
    """A recorded portion of two groups of segments: every replay starts its tickets and words anew, with eager portions in between."""
    from based_amd import ops

    B, L, W, n = 2, 4200, 128, 64
    g = torch.Generator().manual_seed(77)
    rnd = lambda *s: torch.randn(*s, generator=g).to(dtype).to(dev)  # noqa: E731
    gates = (rnd(2, n, n) * n ** -0.5, rnd(W), rnd(2, n, n) * n ** -0.5, rnd(W), rnd(W) - 3)
    inputs = [(rnd(B, L, W), rnd(B, L, W), torch.randn(B, W, generator=g).to(dev)) for _ in range(3)]

    def run(u, y, state, out):
        return ops.rglru_prefill(u, y, *gates, state, 8.0, False, out=u if over else out)

    want = []
    for u, y, state in inputs:
        u, state = u.clone(), state.clone()
        want.append((run(u, y, state, torch.empty_like(u)).clone(), state))
    u, y, state, out = torch.empty_like(inputs[0][0]), torch.empty_like(inputs[0][1]), torch.empty(B, W, device=dev), torch.empty_like(inputs[0][0])
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        run(u.zero_(), y.zero_(), state.zero_(), out)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        res = run(u, y, state, out)
    for i in (0, 1, 2, 0, 2):
        for t, x in zip((u, y, state), inputs[i]):
            t.copy_(x)
        if not over:
            out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(res, want[i][0]) and torch.equal(state, want[i][1]), i
        eager = run(inputs[1][0].clone(), inputs[1][1], inputs[1][2].clone(), torch.empty_like(out))
        assert torch.equal(eager, want[1][0])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("L", [1, 17, 40, 64, 130, 4200, 8300])
def test_infinite_states_outlive_segments(dev, L, dtype):
    """An infinity times decays that are small, none of them zero, stays one, however small their product."""
    from based_amd import ops

    B, W = 2, 24
    g = torch.Generator().manual_seed(L)
    rnd = lambda *s: torch.randn(*s, generator=g).to(dtype).to(dev)  # noqa: E731
    u, gates = rnd(B, L, W), (rnd(1, W, W) * W ** -0.5, rnd(W), rnd(1, W, W) * W ** -0.5, rnd(W), rnd(W) + 1)  # decays of 2^-8 and less
    y = rnd(B, L, W).abs() + 0.1
    state = torch.zeros(B, W, device=dev)
    state[0, 3], state[1, 7] = float("inf"), float("-inf")
    out = ops.rglru_prefill(u, y, *gates, state, 8.0, False, out=torch.empty_like(u))
    assert (out[0, :, 3] == float("inf")).all() and (out[1, :, 7] == float("-inf")).all()
    assert state[0, 3] == float("inf") and state[1, 7] == float("-inf")
    out[0, :, 3], out[1, :, 7], state[0, 3], state[1, 7] = 0, 0, 0, 0
    assert out.isfinite().all() and state.isfinite().all()
