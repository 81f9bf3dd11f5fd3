"""Window attention over fp32 prompts: the matrix form and, for rows off a 16-byte address, the general one, both against 64 bits."""
import pytest
import torch

from oracle import sozilix_oracle as O

pytestmark = pytest.mark.gpu


def _run(dev, q, k, v, window, scale, start, rope, shift):
    """The portion from `start` on, the rows before it already in the cache; rows of q, k, v and the output `shift` elements off."""
    from based_amd import ops

    B, L, H, d = q.shape
    G, dv = v.shape[2:]
    cache = torch.full((B, L, G, d + dv), float("nan"), device=dev)

    def placed(t, rows):
        return torch.empty(B, rows, t + shift, device=dev)[..., shift:]

    kw = dict(rope=rope, out_scale=0.5)
    qd, kd, vd = (t.to(dev).flatten(2) for t in (q, k, v))
    if start:
        ops.window_attn_prefill(qd[:, :start], kd[:, :start], vd[:, :start], cache, H, G, window, scale, 0,
                                out=torch.empty(B, start, H * dv, device=dev), **kw)
    qs, out = placed(H * d, L - start).copy_(qd[:, start:]), placed(H * dv, L - start)
    ks, vs = placed(G * d, L - start).copy_(kd[:, start:]), placed(G * dv, L - start).copy_(vd[:, start:])
    ops.window_attn_prefill(qs, ks, vs, cache, H, G, window, scale, start, out=out, **kw)
    return 2 * out.double().cpu().view(B, L - start, H, dv)


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("H,G,d,dv,L,start,window,rot,half,scale", [
    (4, 1, 64, 64, 1, 0, 1, 0, False, 0.2), (16, 4, 64, 64, 131, 0, 33, 32, False, 0.125), (3, 1, 60, 36, 97, 31, 16, 4, False, 0.2),
    (6, 2, 68, 64, 65, 0, 100, 8, True, -0.1), (2, 2, 4, 128, 200, 7, 31, 0, False, 0.5), (5, 1, 128, 100, 160, 96, 64, 128, True, 0.1),
    (1, 1, 32, 4, 300, 290, 500, 24, True, 0.0)])
def test_window_prefill_f32(dev, H, G, d, dv, L, start, window, rot, half, scale, shift):
    from based_amd.mixers.window_attention import _ExactRotary

    B = 2
    g = torch.Generator().manual_seed(H * L + window)
    q, k, v = (torch.randn(B, L, n, m, generator=g) for n, m in ((H, d), (G, d), (G, dv)))
    rope = _ExactRotary(rot, base=100.0, interleaved=not half).tables(L, dev) if rot else None
    out = _run(dev, q, k, v, window, scale, start, rope, shift)
    qq, kk = q.double(), k.double()
    if rot:
        perm = torch.arange(d)
        if half:
            perm[:rot] = torch.tensor([c // 2 + (c % 2) * (rot // 2) for c in range(rot)])
        qq, kk = (torch.stack([O.rotate(x[b][..., perm], 100.0, rot) for b in range(B)]) for x in (qq, kk))
    ref = torch.stack([O.window_softmax(qq[b], kk[b], v[b].double(), scale, window) for b in range(B)])[:, start:]
    err = (out - ref).norm(dim=-1) / ref.norm(dim=-1)
    # scores of up to 20 and sums of 128 products: 20 * 2^-24 on every weight, and as much again from the rotation
    assert float(err.max()) < 3e-6, float(err.max())


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_rows_that_do_not_see_a_key_do_not_take_its_value(dev, bad):
    B, L, H, G, d, window, at = 1, 150, 4, 2, 64, 40, 70
    g = torch.Generator().manual_seed(9)
    q, k, v = (torch.randn(B, L, n, d, generator=g) for n in (H, G, G))
    clean = _run(dev, q, k, v, window, 0.1, 0, None, 0)
    k[:, at, 0], v[:, at, 0, 5] = bad, bad
    out = _run(dev, q, k, v, window, 0.1, 0, None, 0)
    sees = torch.zeros(L, dtype=torch.bool)
    sees[at:at + window] = True
    assert not out[:, sees][:, :, :2].isfinite().all(-1).any()
    assert torch.allclose(out[:, ~sees], clean[:, ~sees], rtol=1e-5, atol=1e-6) and torch.equal(out[:, :, 2:], clean[:, :, 2:])


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("bad", [float("nan"), float("inf"), float("-inf")])
def test_scale_of_zero(dev, bad, shift):
    """Zero times an infinite score is no number, whatever its sign, in every row that sees the key and in no other."""
    B, L, H, G, d, window, at = 1, 150, 4, 2, 64, 40, 70
    g = torch.Generator().manual_seed(10)
    q, k, v = (torch.randn(B, L, n, d, generator=g) for n in (H, G, G))
    k[:, at, 0, 5] = bad
    out = _run(dev, q, k, v, window, 0.0, 0, None, shift)
    sees = torch.zeros(L, dtype=torch.bool)
    sees[at:at + window] = True
    assert out[:, sees][:, :, :2].isnan().all()
    mean = torch.stack([v[0, max(0, t - window + 1):t + 1].double().mean(0) for t in range(L)])[None].repeat_interleave(H // G, 2)
    assert torch.allclose(out[:, ~sees], mean[:, ~sees], rtol=0, atol=1e-6) and torch.allclose(out[:, :, 2:], mean[:, :, 2:], rtol=0, atol=1e-6)


@pytest.mark.parametrize("d,dv,H,G,L,start,window", [
    (4, 4, 16, 4, 100, 0, 200), (8, 64, 16, 1, 90, 30, 64), (16, 16, 16, 16, 90, 20, 300), (24, 24, 16, 4, 70, 0, 33), (32, 32, 8, 2, 70, 10, 129),
    (48, 20, 6, 2, 65, 0, 40), (64, 64, 4, 4, 60, 40, 70), (64, 32, 16, 4, 16, 100, 90), (12, 128, 4, 1, 70, 0, 50), (32, 100, 2, 2, 70, 5, 64),
    (64, 128, 1, 1, 17, 0, 9), (80, 80, 4, 2, 70, 20, 100), (96, 32, 8, 8, 50, 0, 90), (96, 96, 2, 2, 70, 0, 128), (128, 64, 4, 1, 50, 7, 66),
    (128, 128, 4, 4, 70, 0, 33), (100, 40, 16, 16, 20, 40, 16)])
def test_both_sides_of_the_rule_for_few_rows(dev, d, dv, H, G, L, start, window):
    """Batches on either side of the number of rows from which on the matrix form runs: two of them, and eight times as many."""
    for B in (1, 2, 16):
        g = torch.Generator().manual_seed(d + dv)
        q, k, v = (torch.randn(B, start + L, n, m, generator=g) for n, m in ((H, d), (G, d), (G, dv)))
        out = _run(dev, q, k, v, window, d ** -0.5, start, None, 0)
        rows = slice(0, B, max(1, B - 1))  # the first and the last sequence
        ref = torch.stack([O.window_softmax(qq.double(), kk.double(), vv.double(), d ** -0.5, window) for qq, kk, vv in
                           zip(q[rows], k[rows], v[rows])])[:, start:]
        err = (out[rows] - ref).norm(dim=-1) / ref.norm(dim=-1)
        assert float(err.max()) < 3e-6, (B, float(err.max()))  # (scores of up to 5 and sums of 128 products)


@pytest.mark.parametrize("d,dv,H,G,B,L,window", [
    (64, 64, 16, 16, 1, 1024, 300), (64, 64, 16, 16, 1, 1025, 300), (32, 64, 16, 4, 1, 3200, 290), (32, 64, 16, 4, 1, 3201, 290), (64, 48, 16, 4, 1, 2048, 240),
    (64, 48, 16, 4, 1, 2048, 241), (64, 128, 15, 3, 4, 320, 200), (64, 128, 15, 3, 4, 321, 200), (128, 64, 16, 4, 1, 300, 129), (96, 32, 4, 4, 1, 1500, 513)])
def test_both_sides_of_the_rule_for_two_wavefronts(dev, d, dv, H, G, B, L, window):
    """512 workgroups and more, 800 and more, 256 keys and more, 300 workgroups and more with wide values; wide keys."""
    g = torch.Generator().manual_seed(L)
    q, k, v = (torch.randn(B, L, n, m, generator=g) for n, m in ((H, d), (G, d), (G, dv)))
    out = _run(dev, q, k, v, window, d ** -0.5, 0, None, 0)[-1]
    ref = O.window_softmax(q[-1].double(), k[-1].double(), v[-1].double(), d ** -0.5, window)
    err = (out - ref).norm(dim=-1) / ref.norm(dim=-1)
    assert float(err.max()) < 3e-6, float(err.max())  # (scores of up to 5 and sums of 128 products)


@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("H,G,d,dv,B,L,start,window,rot,half", [
    (16, 4, 64, 64, 1, 777, 0, 129, 32, False), (16, 4, 64, 64, 1, 300, 77, 129, 32, True), (6, 2, 60, 36, 3, 190, 0, 20, 8, False),
    (16, 16, 64, 64, 1, 130, 1, 64, 64, False), (12, 4, 64, 100, 1, 200, 40, 200, 16, True), (8, 1, 100, 64, 2, 128, 0, 65, 4, False),
    (16, 2, 64, 64, 2, 500, 0, 513, 32, False)])
def test_cache_that_the_attention_fills(dev, H, G, d, dv, B, L, start, window, rot, half, norm):
    """Rows of the cache behind a portion, and what a second portion makes of them: written by the attention itself, or in front of it where the
    portion's own keys lie in the output's rows."""
    from based_amd import ops
    from based_amd.mixers.window_attention import _ExactRotary

    g = torch.Generator().manual_seed(L)
    n = L + start
    rope = _ExactRotary(rot, base=100.0, interleaved=not half).tables(n, dev)
    x = torch.randn(B, n, H * d + G * (d + dv), generator=g).to(dev)
    q, k, v = x[..., :H * d], x[..., H * d:(H + G) * d], x[..., (H + G) * d:]
    kw = dict(rope=rope, value_norm_eps=1e-5 if norm else None)

    def run(inside):
        cache = torch.full((B, n + 2, G, d + dv), float("nan"), device=dev)
        room = x.clone() if inside else torch.full((B, n, H * dv), float("nan"), device=dev)
        kk, vv = (room[..., H * d:(H + G) * d], room[..., (H + G) * d:]) if inside else (k, v)
        out = room[..., :H * dv] if inside and dv <= d else torch.empty(B, n, H * dv, device=dev) if inside else room
        qq = q
        for lo, hi in ((0, start), (start, n)):
            if hi > lo:
                s = slice(lo, hi)
                ops.window_attn_prefill(qq[:, s], kk[:, s], vv[:, s], cache, H, G, window, d ** -0.5, lo, out=out[:, s], **kw)
        return out.clone(), cache

    out, cache = run(False)
    ref, rows = run(True)
    # (a rotation's two products are added in one order or the other: 2^-24 of the larger)
    assert float((cache[:, :n] - rows[:, :n]).abs().max()) <= 2 ** -23 * float(rows[:, :n].abs().max()) and cache[:, n:].isnan().all()
    # (two forms of the same sums of up to 513 weights: a few roundings of 2^-24)
    assert float((out - ref).norm() / ref.norm()) < 1e-6
    want = v.view(B, n, G, dv).double()
    if norm:
        want = want / (want.square().mean(-1, keepdim=True) + 1e-5).sqrt()
    assert float((cache[:, :n, :, d:].double() - want).norm() / want.norm()) < 2e-7
