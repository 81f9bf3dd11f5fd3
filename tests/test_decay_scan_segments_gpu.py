"""Decaying states over long portions that the matrix form does not take (fp32, odd sizes): cut into segments or in one chain."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("channel", [True, False])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,L,H,d,dv,start", [(1, 255, 1, 64, 16, 0), (1, 256, 2, 20, 17, 0), (2, 257, 1, 33, 64, 5), (1, 1031, 1, 130, 9, 40),
                                              (1, 400, 3, 68, 31, 63)])
def test_decay_scan_segments(dev, B, L, H, d, dv, start, dtype, channel):
    from based_amd import ops

    g = torch.Generator().manual_seed(L * 7 + d)
    rnd = lambda *s: torch.randn(*s, generator=g).to(dtype)  # noqa: E731
    q, k, v, u = rnd(B, L, H, d), rnd(B, L, H, d), rnd(B, L, H, dv), rnd(H, d)
    lw = -torch.exp(0.5 * torch.randn(B, L, H, d, generator=g) + torch.linspace(-7, 1, d)) / math.log(2)
    decay = [0.999, 0.0, 0.9][:H]
    kw = dict(head_decay=ops.head_decays(decay, dev)) if not channel else dict(bonus=u.to(dev))
    qd, kd, vd = (torch.empty(B, L, t.shape[2] * t.shape[3] + 1, dtype=dtype, device=dev)[..., 1:].copy_(t.flatten(2)) for t in (q, k, v))
    state = torch.full((B, H, dv, (d + 3) // 4 * 4), float("nan"), device=dev)
    out = []
    for s in ([slice(0, start), slice(start, L)] if start else [slice(0, L)]):
        if channel:
            kw["channel_log2"] = lw[:, s].flatten(2).contiguous().to(dev)
        out.append(ops.decay_scan(qd[:, s], kd[:, s], vd[:, s], state, H, fresh=s.start == 0, **kw))
    out = torch.cat(out, 1).double().cpu().view(B, L, H, dv)
    S, ref = torch.zeros(B, H, d, dv, dtype=torch.float64), []
    for t in range(L):
        qt, kt, vt = (x[:, t].double() for x in (q, k, v))
        kv = kt[..., None] * vt[:, :, None]
        if channel:
            ref.append(((S + u.double()[..., None] * kv) * qt[..., None]).sum(2))
            S = 2.0 ** lw[:, t].double()[..., None] * S + kv
        else:
            S = torch.tensor(decay, dtype=torch.float32).double().view(1, H, 1, 1) * S + kv  # (decays as fp32 holds them)
            ref.append((S * qt[..., None]).sum(2))
    ref = torch.stack(ref, 1)
    rel = lambda a, b: ((a - b).norm() / b.norm()).item()  # noqa: E731
    # The slowest decays keep a thousand tokens.  Each rounds the decay and the sum by up to 2^-24, independently: 2 * 2^-24 * 1000^0.5 =
    # 3.8e-6; bf16 outputs add half of 2^-8.
    tol = 4e-6 if dtype == torch.float32 else 3e-3
    assert rel(out, ref) < tol and rel(out[:, -8:], ref[:, -8:]) < tol, (rel(out, ref), rel(out[:, -8:], ref[:, -8:]))
    assert rel(state[..., :d].double().cpu(), S.transpose(2, 3)) < 4e-6


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("L", [255, 300, 513])
def test_head_decays_below_zero(dev, L, dtype):
    """A decay that changes its sign from token to token has no logarithm, but powers: in segments as in one chain."""
    from based_amd import ops

    H, d, dv, decay = 3, 20, 17, [-0.9, -0.9995, -1.0]
    g = torch.Generator().manual_seed(L)
    q, k, v = (torch.randn(1, L, H * n, generator=g).to(dtype) for n in (d, d, dv))
    state = torch.randn(1, H, dv, 20, generator=g)
    S, ref = state.double().transpose(2, 3), []
    w = torch.tensor(decay, dtype=torch.float32).double().view(1, H, 1, 1)
    for t in range(L):
        qt, kt, vt = (x[:, t].double().view(1, H, -1) for x in (q, k, v))
        S = w * S + kt[..., None] * vt[:, :, None]
        ref.append((S * qt[..., None]).sum(2).flatten(1))
    state = state.to(dev)
    out = ops.decay_scan(q.to(dev), k.to(dev), v.to(dev), state, H, head_decay=ops.head_decays(decay, dev), fresh=False)
    rel = lambda a, b: ((a.double().cpu() - b).norm() / b.norm()).item()  # noqa: E731
    # as above: up to five hundred roundings of 2^-24 that lie independently, and half of 2^-8 of bf16 outputs
    assert rel(out, torch.stack(ref, 1)) < (4e-6 if dtype == torch.float32 else 3e-3)
    assert rel(state, S.transpose(2, 3)) < 4e-6


@pytest.mark.parametrize("B,L,d", [(3, 45, 130), (65, 45, 130), (50, 33, 250)])
def test_long_keys_in_many_workgroups(dev, B, L, d):
    """Keys of more than 128 channels: 16 tokens at a time, or 8 where the workgroups are many; whole tiles and a rest."""
    from based_amd import ops

    H, dv = 2, 128
    g = torch.Generator().manual_seed(B + L)
    q, k, v, u = (torch.randn(*s, generator=g) for s in ((B, L, H * d), (B, L, H * d), (B, L, H * dv), (H, d)))
    lw = -torch.exp(torch.randn(B, L, H * d, generator=g) - 2)
    decay = [0.9, 0.99]
    dp = (d + 3) // 4 * 4
    S0 = torch.randn(B, H, dv, dp, generator=g)
    for channel in (True, False):
        kw = dict(channel_log2=lw.to(dev), bonus=u.to(dev)) if channel else dict(head_decay=ops.head_decays(decay, dev))
        state = S0.to(dev)
        out = ops.decay_scan(q.to(dev), k.to(dev), v.to(dev), state, H, fresh=False, **kw)
        S, ref = S0[..., :d].double().transpose(2, 3), []
        w = torch.tensor(decay, dtype=torch.float32).double().view(1, H, 1, 1)
        for t in range(L):
            qt, kt, vt = (x[:, t].double().view(B, H, -1) for x in (q, k, v))
            kv = kt[..., None] * vt[:, :, None]
            if channel:
                ref.append(((S + u.double()[..., None] * kv) * qt[..., None]).sum(2).flatten(1))
                S = 2.0 ** lw[:, t].double().view(B, H, d, 1) * S + kv
            else:
                S = w * S + kv
                ref.append((S * qt[..., None]).sum(2).flatten(1))
        rel = lambda a, b: ((a.double().cpu() - b).norm() / b.norm()).item()  # noqa: E731
        assert rel(out, torch.stack(ref, 1)) < 1e-6 and rel(state[..., :d], S.transpose(2, 3)) < 1e-6  # (some dozens of roundings of 2^-24)


@pytest.mark.parametrize("channel", [True, False])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,L,H,d,dv", [(4, 1023, 16, 64, 64), (4, 1025, 16, 64, 64),            # eight or nine segments of two pieces
                                        (1, 64 * 64 + 70, 1, 20, 17), (2, 64 * 130 + 1, 1, 8, 4),  # 33 of two, 44 of three
                                        (8, 257, 16, 64, 64), (8, 320, 16, 20, 64),                # one chain, and three of two, the last of a piece
                                        (8, 271, 16, 68, 60), (8, 272, 16, 68, 60)])               # one chain, and three
def test_segments_of_several_pieces(dev, B, L, H, d, dv, dtype, channel):
    """Segments longer than a 64-token piece, the last one shorter than the others: fresh, and from a state that goes on."""
    from based_amd import ops

    g = torch.Generator().manual_seed(L + d)
    dp = (d + 3) // 4 * 4
    mk = lambda *s: torch.randn(*s, generator=g).to(dtype).to(dev)  # noqa: E731
    q, k, v, u = mk(B, L, H * d), mk(B, L, H * d), mk(B, L, H * dv), mk(H, d)
    if dtype == torch.bfloat16:  # rows off an 8-byte address, which the matrix form would take
        q, k, v = (torch.empty(B, L, t.shape[2] + 1, dtype=dtype, device=dev)[..., 1:].copy_(t) for t in (q, k, v))
    lw = -torch.exp(0.5 * torch.randn(B, L, H * d, generator=g) - 4).to(dev)
    decay = torch.linspace(0.9, 0.9995, H).tolist()
    kw = dict(channel_log2=lw, bonus=u) if channel else dict(head_decay=ops.head_decays(decay, dev))
    S0 = torch.zeros(B, H, dv, dp)
    S0[..., :d] = torch.randn(B, H, dv, d, generator=g)
    rel = lambda a, b: ((a.double() - b).norm() / b.norm()).item()  # noqa: E731
    for fresh in (True, False):
        state = torch.full((B, H, dv, dp), float("nan"), device=dev) if fresh else S0.to(dev)
        out = ops.decay_scan(q, k, v, state, H, fresh=fresh, **kw)
        S = torch.zeros(B, H, d, dv, dtype=torch.float64, device=dev) if fresh else S0[..., :d].double().transpose(2, 3).to(dev)
        w = torch.tensor(decay, dtype=torch.float32).double().view(1, H, 1, 1).to(dev)
        ref = torch.empty(B, L, H * dv, dtype=torch.float64, device=dev)
        for t in range(L):
            qt, kt, vt = (x[:, t].double().view(B, H, -1) for x in (q, k, v))
            kv = kt[..., None] * vt[:, :, None]
            if channel:
                ref[:, t] = ((S + u.double()[..., None] * kv) * qt[..., None]).sum(2).flatten(1)
                S = 2.0 ** lw[:, t].double().view(B, H, d, 1) * S + kv
            else:
                S = w * S + kv
                ref[:, t] = (S * qt[..., None]).sum(2).flatten(1)
        # decays of 0.99 and 0.9995 keep a hundred to two thousand tokens: 2 * 2^-24 * 2000^0.5 = 5e-6; bf16 outputs add half of 2^-8
        assert rel(out, ref) < (5e-6 if dtype == torch.float32 else 3e-3) and rel(state[..., :d], S.transpose(2, 3)) < 5e-6


@pytest.mark.parametrize("channel", [True, False])
def test_infinite_states_outlive_segments(dev, channel):
    """An infinity times decays that are small, none of them zero, stays one, however small their product; times zero it is no number."""
    from based_amd import ops

    H, d, dv, L = 2, 20, 17, 300
    g = torch.Generator().manual_seed(3)
    q, k, v, u = (torch.randn(*s, generator=g).to(dev) for s in ((1, L, H * d), (1, L, H * d), (1, L, H * dv), (H, d)))
    lw = torch.full((1, L, H, d), -9.0)
    lw[:, 100, 1] = float("-inf")
    kw = dict(channel_log2=lw.flatten(2).to(dev), bonus=u) if channel else dict(head_decay=ops.head_decays([2.0 ** -9, 0.0], dev))
    state = torch.zeros(1, H, dv, d, device=dev)
    state[:, :, 3, 5] = float("inf")
    state[:, :, 4, 5] = float("-inf")
    out = ops.decay_scan(q, k, v, state, H, fresh=False, **kw).view(1, L, H, dv)
    assert state[0, 0, 3, 5] == float("inf") and state[0, 0, 4, 5] == float("-inf")
    assert state[0, 1, 3, 5].isnan() and state[0, 1, 4, 5].isnan()
    assert out[:, :, 0, 3].isinf().all() and out[:, :, 0, 4].isinf().all() and out[:, 101:, 1, 3].isnan().all()
    state[:, :, 3:5, 5], out[..., 3:5] = 0, 0
    assert state.isfinite().all() and out.isfinite().all()


@pytest.mark.parametrize("channel", [True, False])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("L,d", [(1, 3), (1, 17), (8, 64), (9, 66), (8, 101), (9, 128), (1, 130), (8, 255), (9, 256)])
def test_few_tokens(dev, L, d, dtype, channel):
    """Portions of one piece of tokens and one more; states in rows of 16-byte pieces whose rest stays as it is, bonuses of any alignment."""
    from based_amd import ops

    B, H, dv = 2, 3, 21
    g = torch.Generator().manual_seed(L + d)
    dp = (d + 3) // 4 * 4
    q, k, v = (torch.randn(B, L, H * n + 1, generator=g).to(dtype).to(dev)[..., 1:] for n in (d, d, dv))
    u = torch.randn(H, d, generator=g).to(dtype).to(dev)
    lw = -torch.exp(torch.randn(B, L, H * d, generator=g) - 2).to(dev)
    decay = [0.9, 0.99, 0.5]
    kw = dict(channel_log2=lw, bonus=u) if channel else dict(head_decay=ops.head_decays(decay, dev))
    S0 = torch.full((B, H, dv, dp), float("nan"))
    S0[..., :d] = torch.randn(B, H, dv, d, generator=g)
    rel = lambda a, b: ((a.double() - b).norm() / b.norm()).item()  # noqa: E731
    for fresh in (True, False):
        state = S0.to(dev)
        out = ops.decay_scan(q, k, v, state, H, fresh=fresh, **kw)
        S = torch.zeros(B, H, d, dv, dtype=torch.float64, device=dev) if fresh else S0[..., :d].double().transpose(2, 3).to(dev)
        w = torch.tensor(decay, dtype=torch.float32).double().view(1, H, 1, 1).to(dev)
        ref = torch.empty(B, L, H * dv, dtype=torch.float64, device=dev)
        for t in range(L):
            qt, kt, vt = (x[:, t].double().view(B, H, -1) for x in (q, k, v))
            kv = kt[..., None] * vt[:, :, None]
            if channel:
                ref[:, t] = ((S + u.double()[..., None] * kv) * qt[..., None]).sum(2).flatten(1)
                S = 2.0 ** lw[:, t].double().view(B, H, d, 1) * S + kv
            else:
                S = w * S + kv
                ref[:, t] = (S * qt[..., None]).sum(2).flatten(1)
        # sums of up to 256 products of 2^-24 each, independent: 16 * 2^-24 = 1e-6; bf16 outputs add half of 2^-8
        assert rel(out, ref) < (1e-6 if dtype == torch.float32 else 3e-3) and rel(state[..., :d], S.transpose(2, 3)) < 1e-6
        assert state[..., d:].isnan().all()


@pytest.mark.parametrize("channel", [True, False])
@pytest.mark.parametrize("fresh", [True, False])
@pytest.mark.parametrize("L,d,dv", [(512, 64, 64), (577, 20, 36), (1100, 64, 100), (2048, 60, 64), (2304, 64, 64), (2500, 36, 16), (700, 72, 64),
                                    (2817, 20, 16), (4100, 36, 16), (4353, 64, 16)])
def test_segments_of_the_matrix_form(dev, L, d, dv, fresh, channel):
    """Two segments to seventeen of bf16 portions, put together by those behind them (up to ten with channel decays, sixteen with head decays) or by
    a launch of its own, against 64-bit sums token by token and against one chain of portions that are too short for segments."""
    from based_amd import ops

    B, H, decay = 1, 2, [0.9995, 0.9]
    g = torch.Generator().manual_seed(L + d)
    q, k, v = (torch.randn(B, L, H * n, generator=g).bfloat16().to(dev) for n in (d, d, dv))
    dp = (d + 3) // 4 * 4
    start = torch.zeros(B, H, dv, dp) if fresh else torch.randn(B, H, dv, dp, generator=g)
    state = torch.full((B, H, dv, dp), float("nan"), device=dev) if fresh else start.to(dev)
    lw = (-torch.exp(0.5 * torch.randn(B, L, H, d, generator=g) + torch.linspace(-7, 1, d)) / math.log(2)).flatten(2).to(dev)
    u = torch.randn(H, d, generator=g).bfloat16().to(dev)
    kw = dict(head_decay=ops.head_decays(decay, dev)) if not channel else dict(bonus=u)
    part = lambda s: dict(channel_log2=lw[:, s].contiguous()) if channel else {}  # noqa: E731
    whole = ops.decay_scan(q, k, v, state, H, fresh=fresh, **kw, **part(slice(0, L)))
    chain, pieces = start.to(dev), []
    for at in range(0, L, 192):
        s = slice(at, min(at + 192, L))
        pieces.append(ops.decay_scan(q[:, s], k[:, s], v[:, s], chain, H, fresh=False, **kw, **part(s)))
    rel = lambda a, b: ((a.double() - b.double()).norm() / b.double().norm()).item()  # noqa: E731
    # outputs: one rounding to bf16 that falls another way, 2^-8 of few values; states: 32-bit sums in another order over up to 4400 tokens
    assert rel(whole, torch.cat(pieces, 1)) < 1e-3
    assert rel(state[..., :d], chain[..., :d]) < 1e-5
    S, ref = start[..., :d].double().transpose(2, 3).to(dev), torch.empty(B, L, H, dv, dtype=torch.float64, device=dev)
    w = 2.0 ** lw.double().view(B, L, H, d, 1) if channel else torch.tensor(decay, device=dev).double().view(1, 1, H, 1, 1).expand(B, L, H, 1, 1)
    qd, kd, vd = (x.double().view(B, L, H, -1) for x in (q, k, v))
    for t in range(L):
        kv = kd[:, t, :, :, None] * vd[:, t, :, None]
        if channel:
            ref[:, t] = ((S + u.double()[..., None] * kv) * qd[:, t, ..., None]).sum(2)
        S = w[:, t] * S + kv
        if not channel:
            ref[:, t] = (S * qd[:, t, ..., None]).sum(2)
    # bf16 outputs: half of 2^-8 at most, 2^-9 / 3^0.5 = 1.1e-3 evenly spread; a state's terms keep 16 bits each, 2^-17 / 3^0.5 = 4.4e-6
    assert rel(whole.view(B, L, H, dv), ref) < 3e-3 and rel(state[..., :d], S.transpose(2, 3)) < 2e-5


def _head_decays_in_64_bits(q, k, v, w, state):
    """o (B, L, H, dv) and the state (B, H, dv, d) behind a portion, token by token."""
    B, L, H, d = q.shape
    S, o = state.double().transpose(2, 3), []
    for t in range(L):
        S = w.double().view(1, H, 1, 1) * S + k[:, t].double()[..., None] * v[:, t].double()[:, :, None]
        o.append((S * q[:, t].double()[..., None]).sum(2))
    return torch.stack(o, 1), S.transpose(2, 3)


@pytest.mark.parametrize("L,d,dv", [(100, 64, 64), (301, 20, 36), (513, 64, 64), (577, 32, 16), (1100, 64, 100), (2048, 60, 64), (2500, 36, 16),
                                    (200, 72, 64), (1030, 128, 64)])
def test_signs_of_head_decays_in_the_matrix_form(dev, L, d, dv):
    """Decays below zero, zero and above, bf16: one chain, two segments to eight that put the ones in front together themselves, ten, and heads of
    more than 64 channels."""
    from based_amd import ops

    B, decay = 2, [-0.9, -0.9995, -1.0, 0.0, 0.999, -2.0 ** -9]
    H, g = len(decay), torch.Generator().manual_seed(L + d)
    q, k, v = (torch.randn(B, L, H, n, generator=g).bfloat16() for n in (d, d, dv))
    S0 = torch.randn(B, H, dv, d, generator=g)
    state = S0.to(dev)
    got = ops.decay_scan(*(x.flatten(2).to(dev) for x in (q, k, v)), state, H, head_decay=ops.head_decays(decay, dev), fresh=False)
    want, S = _head_decays_in_64_bits(q, k, v, torch.tensor(decay), S0)
    got, state = got.double().cpu().view(B, L, H, dv), state.double().cpu()
    for h in range(H):  # each head by itself: they differ in size by up to fifty times
        rel = lambda a, b: ((a[..., h, :] - b[..., h, :]).norm() / b[..., h, :].norm()).item()  # noqa: E731
        # bf16 outputs: half of 2^-8 at most, 2^-9 / 3^0.5 = 1.1e-3 evenly spread; weights keep 16 bits
        assert rel(got, want) < 3e-3 and rel(got[:, -8:], want[:, -8:]) < 3e-3, (decay[h], rel(got, want))
        rel = lambda a, b: ((a[:, h] - b[:, h]).norm() / b[:, h].norm()).item()  # noqa: E731
        # a sum's terms keep 16 bits each, 2^-17 / 3^0.5 = 4.4e-6 evenly spread, signs independent
        assert rel(state, S) < 2e-5, (decay[h], rel(state, S))


@pytest.mark.parametrize("L", [60, 150, 513, 1100, 2500])
def test_infinite_states_in_the_matrix_form(dev, L):
    """An infinite part of the state that enters, head decays, bf16, one chain to ten segments: infinite and no numbers where they are token by token."""
    from based_amd import ops

    decay, d, dv = [-0.9, 2.0 ** -9, 0.0, 0.999, -2.0 ** -9], 64, 64
    H, g = len(decay), torch.Generator().manual_seed(L)
    q, k, v = (torch.randn(1, L, H, n, generator=g).bfloat16() for n in (d, d, dv))
    S0 = torch.randn(1, H, dv, d, generator=g)
    S0[:, :, 3, 5], S0[:, :, 40, 63] = float("inf"), float("-inf")
    state = S0.to(dev)
    got = ops.decay_scan(*(x.flatten(2).to(dev) for x in (q, k, v)), state, H, head_decay=ops.head_decays(decay, dev), fresh=False)
    want, S = _head_decays_in_64_bits(q, k, v, torch.tensor(decay), S0)
    for a, b in ((got.cpu().view(1, L, H, dv), want), (state.cpu(), S)):
        assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.isinf(), b.isinf()) and torch.equal(a[a.isinf()] > 0, b[b.isinf()] > 0)


@pytest.mark.parametrize("L", [60, 513, 1100, 2500])
def test_infinite_states_and_channel_decays_in_the_matrix_form(dev, L):
    """The same with channel decays: the state's part stays infinite, and what does not meet it stays a number."""
    from based_amd import ops

    H, d, dv, g = 2, 64, 64, torch.Generator().manual_seed(L)
    q, k, v, u = (torch.randn(*s, generator=g).bfloat16().to(dev) for s in ((1, L, H * d), (1, L, H * d), (1, L, H * dv), (H, d)))
    lw = torch.full((1, L, H * d), -2.0 ** -5, device=dev)  # (2^-2 over 64 tokens, 2^-79 over all)
    state = torch.randn(1, H, dv, d, generator=g).to(dev)
    state[:, :, 3, 5], state[:, :, 40, 63] = float("inf"), float("-inf")
    out = ops.decay_scan(q, k, v, state, H, channel_log2=lw, bonus=u, fresh=False).view(1, L, H, dv)
    assert (state[:, :, 3, 5] == float("inf")).all() and (state[:, :, 40, 63] == float("-inf")).all()
    assert not out[..., [3, 40]].isfinite().any()
    state[:, :, 3, 5], state[:, :, 40, 63], out[..., [3, 40]] = 0, 0, 0
    assert state.isfinite().all() and out.isfinite().all()
