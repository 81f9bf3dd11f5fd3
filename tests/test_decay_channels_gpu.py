"""Channel decays over prompts in bf16, against the recurrence in 64 bits: every split of heads and channels over wavefronts, at the edges of pieces of
64 tokens, of segments, and of rows in whole 16-byte pieces or not."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [(2, 70, 3, 20, 12),        # up to 32 channels
         (1, 1, 1, 64, 64), (2, 16, 2, 64, 64), (1, 17, 3, 64, 64), (3, 128, 2, 64, 64),  # one piece and two, two wavefronts to the same tokens
         (2, 130, 5, 44, 36),       # rows of 8-byte pieces
         (2, 65, 3, 64, 72),        # value channels of two workgroups
         (30, 129, 14, 64, 64), (30, 66, 14, 60, 44),  # many heads: one wavefront
         (1, 193, 2, 64, 64), (3, 704, 2, 64, 64), (1, 705, 1, 52, 20), (65, 260, 6, 64, 64),  # segments: four of a piece, ten and more, none
         (2, 133, 2, 128, 128), (1, 64, 3, 96, 68), (2, 700, 2, 128, 64), (1, 1100, 1, 72, 128),  # workgroups of 64 value channels
         (33, 66, 4, 128, 128), (34, 130, 4, 100, 132),  # of 128
         # segments of seven pieces and of six; one of 15 in all and three of 16; workgroups of 128 and 64
         (2, 1700, 16, 128, 128), (4, 768, 8, 72, 128), (6, 833, 8, 128, 72), (5, 960, 16, 96, 128), (5, 961, 16, 96, 128), (2, 1700, 16, 128, 64)]


@pytest.mark.parametrize("silu", [False, True])
@pytest.mark.parametrize("fresh", [True, False])
@pytest.mark.parametrize("B,L,H,d,dv", CASES)
def test_channel_decays(dev, B, L, H, d, dv, fresh, silu):
    from based_amd import ops

    g = torch.Generator(device=dev).manual_seed(L * 7 + d + B)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)  # noqa: E731
    x = rnd(B, L, H * (2 * d + dv)).bfloat16()
    q, k, v = x[..., :H * d], x[..., H * d:2 * H * d], x[..., 2 * H * d:]
    u = rnd(H, d).bfloat16()
    lw = -torch.exp(rnd(B, L, H * d) + 2 * rnd(H * d) - 3) / math.log(2)
    dp = (d + 3) // 4 * 4
    state = rnd(B, H, dv, dp)
    S = torch.zeros(B, H, d, dv, dtype=torch.float64, device=dev) if fresh else state[..., :d].double().transpose(2, 3)
    act = ops.ACT_SILU if silu else ops.ACT_NONE
    out = ops.decay_scan(q, k, v, state, H, channel_log2=lw, bonus=u, activation=act, fresh=fresh)
    f = lambda t, n: (torch.nn.functional.silu(t.double()).bfloat16() if silu else t).double().view(B, L, H, n)  # noqa: E731
    qd, kd, vd, w, ref = f(q, d), f(k, d), f(v, dv), 2.0 ** lw.double().view(B, L, H, d), []
    for t in range(L):
        kv = kd[:, t, :, :, None] * vd[:, t, :, None]
        ref.append(((S + u.double()[..., None] * kv) * qd[:, t, :, :, None]).sum(2).flatten(1))
        S = w[:, t, :, :, None] * S + kv
    ref = torch.stack(ref, 1)
    rel = lambda a, b: ((a.double() - b).norm() / b.norm()).item()  # noqa: E731
    # outputs: half of the 2^-8 of bf16 at most.  Keys enter the state as pairs of bf16 (within 2^-18 of themselves), decayed by products of up to a
    # few hundred factors of 2^-24 each: 2^-17 together; a silu that falls the other way in bf16 moves one key or value in some thousands by 2^-8.
    assert rel(out, ref) < 3.9e-3 and rel(out[:, -1:], ref[:, -1:]) < 3.9e-3
    assert rel(state[..., :d], S.transpose(2, 3)) < (1e-4 if silu else 7.7e-6)


@pytest.mark.parametrize("B,H,d,dv", [(2, 3, 32, 32), (4, 16, 64, 64), (40, 16, 64, 64), (2, 8, 128, 128), (40, 8, 128, 128)])
def test_weights_inside_16_tokens_are_of_32_bits(dev, B, H, d, dv):
    """Keys that nearly cancel, in two channels of opposite sign whose decays differ by 2^-12: what is left of a weight is 2^-12 of its two parts."""
    from based_amd import ops

    g = torch.Generator(device=dev).manual_seed(d + B)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)  # noqa: E731
    L = 80
    q, k, lw = rnd(B, L, H, d // 2).bfloat16(), rnd(B, L, H, d // 2).bfloat16(), -0.1 * torch.rand(B, L, H, d // 2, generator=g, device=dev)
    q, k, lw = (torch.stack(x, -1).reshape(B, L, H * d) for x in ((q, q), (k, -k), (lw, lw - 2.0 ** -12)))
    v, u = rnd(B, L, H * dv).bfloat16(), torch.zeros(H, d, device=dev).bfloat16()
    out = ops.decay_scan(q, k, v, torch.zeros(B, H, dv, d, device=dev), H, channel_log2=lw, bonus=u, fresh=True)[:, 2:16].double()
    qd, kd, vd = (x[:, :16].double().view(B, 16, H, -1) for x in (q, k, v))
    lc = torch.cumsum(lw[:, :16].double().view(B, 16, H, d), 1)
    want = torch.zeros(B, 16, H, dv, dtype=torch.float64, device=dev)
    for t in range(2, 16):  # (neighbours have no decay between them: their two parts are nothing together)
        for s in range(t - 1):
            want[:, t] += (qd[:, t] * kd[:, s] * 2.0 ** (lc[:, t - 1] - lc[:, s])).sum(-1, keepdim=True) * vd[:, s]
    want = want[:, 2:].flatten(2)
    # 2^-9 of an output for its rounding to bf16, and 2^-23 of its parts for their decays: n of them, of parts that differ by n 2^-12.5
    assert ((out - want).norm() / want.norm()).item() < 2 ** -9 + 2 ** -10.5


@pytest.mark.parametrize("B,L,H,channels", [(1, 40, 2, True), (3, 130, 4, True), (2, 700, 2, True), (2, 130, 3, False)])
def test_outputs_in_the_place_of_queries(dev, B, L, H, channels):
    """By the entry points themselves: heads of 128 whose outputs are written where their queries lie, as from a copy of these."""
    from based_amd import _lib

    d, lib = 128, _lib.lib()
    g = torch.Generator(device=dev).manual_seed(L)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)  # noqa: E731
    q, k, v, u, row = rnd(B, L, H * d).bfloat16(), rnd(B, L, H * d).bfloat16(), rnd(B, L, H * d).bfloat16(), rnd(H, d).bfloat16(), H * d
    lw = -torch.exp(rnd(B, L, H * d) - 3)
    heads, got = torch.stack([torch.full((H,), -0.1, device=dev), torch.full((H,), 2 ** -0.1, device=dev)]), []
    for own in (False, True):
        state, room = torch.zeros(B, H, d, d, device=dev), q.clone()
        src = room if own else q
        sizes, tail = (B, L, H, d, d, d), (L * row, row) * 4 + (0, 1, 0, torch.cuda.current_stream().cuda_stream)
        work = torch.empty(max(1, lib.based_decay_scan_channels_work(0, *sizes, 0), lib.based_decay_scan_work_of(0, *sizes, 0)), device=dev)
        if channels:
            code = lib.based_decay_scan_channels(src.data_ptr(), k.data_ptr(), v.data_ptr(), lw.data_ptr(), u.data_ptr(), state.data_ptr(), work.data_ptr(),
                                                 room.data_ptr(), *sizes, *tail)
        else:
            code = lib.based_decay_scan(src.data_ptr(), k.data_ptr(), v.data_ptr(), None, heads.data_ptr(), None, state.data_ptr(), work.data_ptr(),
                                        room.data_ptr(), *sizes, *tail)
        assert code == 0
        got.append((room.double(), state))
    rel = lambda a, b: ((a.double() - b.double()).norm() / b.double().norm()).item()  # noqa: E731
    # (sums in another order may round to the other of two neighbours in bf16; keys enter the state as pairs of bf16, within 2^-17 of themselves)
    assert rel(got[1][0], got[0][0]) < 2 ** -10 and rel(got[1][1], got[0][1]) < 2 ** -16


def test_work_space_of_channel_decays():
    """Segments by the rule of channel decays for aligned bf16, those of the general form for everything else; none for short prompts."""
    from based_amd import _lib

    lib = _lib.lib()
    floats = lambda segs, B, H, D, DV: B * H * segs * (DV + 1) * D  # noqa: E731
    for B, L, H, D, segs in [(1, 192, 16, 64, 0), (1, 193, 16, 64, 4), (5, 320, 16, 64, 5), (4, 2048, 16, 64, 10), (1, 4096, 16, 64, 16), (30, 513, 16, 64, 0),
                             (2, 500, 8, 128, 8), (4, 2048, 8, 128, 8), (4, 1536, 8, 128, 4), (10, 961, 8, 128, 3), (10, 960, 8, 128, 0), (16, 1024, 8, 128, 0),
                             (30, 500, 8, 128, 0)]:
        sizes = (B, L, H, D, D, D)
        assert lib.based_decay_scan_channels_work(0, *sizes, 0) == floats(segs, B, H, D, D), (B, L, H, D)
        assert lib.based_decay_scan_channels_work(4, *sizes, 0) == lib.based_decay_scan_work_of(4, *sizes, 0)  # (off 8 bytes)
        assert lib.based_decay_scan_channels_work(0, *sizes, 1) == lib.based_decay_scan_work_of(0, *sizes, 1)
