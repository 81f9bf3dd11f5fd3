"""The C-ABI library loads and exports every symbol include/based_hip.h declares, the ctypes
binding covers exactly that set, and argument validation works without a GPU (validation
happens before any HIP call)."""
import ctypes
import os
import re

import pytest

from based_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared():
    text = open(os.path.join(ROOT, "include", "based_hip.h")).read()
    return set(re.findall(r"BASED_API\s+[\w\s\*]+?\b(based_\w+)\s*\(", text))


def test_header_symbols_are_exported_and_bound():
    declared = _declared()
    assert {"based_linear_attn_step", "based_linear_attn_prefill", "based_swa_prefill", "based_swa_step",
            "based_hip_version", "based_hip_last_error"} <= declared
    assert os.path.exists(_lib.LIB_PATH), "build the library first: python -m based_amd.build"
    handle = ctypes.CDLL(_lib.LIB_PATH)
    for name in declared:
        assert hasattr(handle, name), f"{name} declared in the header but not exported"
    assert set(_lib.SIGNATURES) == declared


def test_header_constants_match_binding():
    text = open(os.path.join(ROOT, "include", "based_hip.h")).read()
    m = re.search(r"#define\s+BASED_PREFILL_SEGMENT_STATE_BYTES\s+(\d+)", text)
    assert m and int(m.group(1)) == _lib.PREFILL_SEGMENT_STATE_BYTES


def test_version_and_error_string():
    lib = _lib.lib()
    assert lib.based_hip_version() >= 1
    assert isinstance(lib.based_hip_last_error(), bytes)


def test_argument_validation_without_gpu():
    lib = _lib.lib()
    # null pointers -> BASED_ERR_ARG (4), nothing launched
    rc = lib.based_linear_attn_step(None, None, None, None, None, None, 1, 1, 64, 0, 0, 0, 0, 0, 0, 0, 0, 1e-12, 0, None)
    assert rc == 4 and b"null" in lib.based_hip_last_error()
    with pytest.raises(ValueError):
        _lib.check(rc)
    buf = (ctypes.c_float * 64)()
    p = ctypes.cast(buf, ctypes.c_void_p)
    # unsupported head dim -> BASED_ERR_SHAPE (1)
    rc = lib.based_linear_attn_step(p, p, p, p, p, p, 1, 1, 40, 0, 0, 0, 0, 0, 0, 0, 0, 1e-12, 0, None)
    assert rc == 1
    # window too wide -> BASED_ERR_SHAPE
    rc = lib.based_swa_prefill(p, p, p, p, 1, 1, 8, 0, 64, 64, 0, 64, 64, 0, 64, 64, 0, 64, 64, 129, 0.125, None, None, 0, None, None, 0, 0, 0, 0, 0, None)
    assert rc == 1
    # fp32 is not a sliding-window element type -> BASED_ERR_DTYPE (2)
    rc = lib.based_swa_prefill(p, p, p, p, 1, 1, 8, 0, 64, 64, 0, 64, 64, 0, 64, 64, 0, 64, 64, 64, 0.125, None, None, 0, None, None, 0, 0, 0, 0, 1, None)
    assert rc == 2
    # misaligned stride -> BASED_ERR_ALIGN (3)
    rc = lib.based_linear_attn_prefill(p, p, p, p, None, None, 1, 1, 8, 64, 0, 0, 20, 0, 0, 16, 0, 0, 64, 0, 0, 64, 1e-12, 0, None)
    assert rc == 3
    # one state pointer without the other -> BASED_ERR_ARG
    rc = lib.based_linear_attn_prefill(p, p, p, p, p, None, 1, 1, 8, 64, 0, 0, 16, 0, 0, 16, 0, 0, 64, 0, 0, 64, 1e-12, 0, None)
    assert rc == 4
    # empty batch is a no-op success
    rc = lib.based_swa_prefill(p, p, p, p, 0, 1, 8, 0, 64, 64, 0, 64, 64, 0, 64, 64, 0, 64, 64, 64, 0.125, None, None, 0, None, None, 0, 0, 0, 0, 0, None)
    assert rc == 0
    # one rotary table without the other -> BASED_ERR_ARG
    rc = lib.based_swa_prefill(p, p, p, p, 1, 1, 8, 0, 64, 64, 0, 64, 64, 0, 64, 64, 0, 64, 64, 64, 0.125, p, None, 8, None, None, 0, 0, 0, 0, 0, None)
    assert rc == 4
    # gated convolution: kernel size outside 2..4 -> BASED_ERR_SHAPE
    rc = lib.based_gated_conv_prefill(p, p, None, p, None, 1, 4, 8, 5, 64, 16, 32, 8, 0, 0, None)
    assert rc == 1
    # allocation-free segmented prefill: more scratch than the static array holds -> BASED_ERR_SHAPE,
    # refused before any HIP call
    rc = lib.based_linear_attn_prefill_split_static(p, p, p, p, None, None, 256, 16, 4096, 64, 0, 0, 16, 0, 0, 16,
                                                    0, 0, 64, 0, 0, 64, 1e-12, 0, 4, None)
    assert rc == 1 and b"scratch" in lib.based_hip_last_error()


def test_parts_hold_what_they_are_for():
    """The partial build for streamed models names existing sources, and these define every entry point
    the streamed operations call."""
    from based_amd import build

    text = ""
    for name in build.PARTS["streaming"]:
        text += open(os.path.join(build.CSRC, f"{name}.hip")).read()
    for entry in ("based_add_norm", "based_stream_conv", "based_window_attn_prefill", "based_window_attn_step",
                  "based_gated_delta_scan", "based_gated_rms_norm", "based_gated_delta_step", "based_rglru_prefill",
                  "based_rglru_step", "based_decode_linear_stream", "based_decode_linear", "based_swiglu", "based_greedy_step",
                  "based_hip_last_error"):
        assert re.search(rf"BASED_API [\w\*]+\s*\**{entry}\(|BASED_API const char\* {entry}\(", text), entry


def test_header_matches_argument_lists():
    """Every ctypes argument list has the number and kinds of arguments the header declares."""
    text = re.sub(r"/\*.*?\*/", "", open(os.path.join(ROOT, "include", "based_hip.h")).read(), flags=re.S)
    names = {"c_void_p": "p", "c_char_p": "p", "c_long": "l", "c_longlong": "l", "c_float": "f", "c_int": "i"}
    for m in re.finditer(r"BASED_API\s+[\w\s\*]+?\b(based_\w+)\s*\(([^;]*?)\);", text, re.S):
        args = [x for x in m.group(2).split(",") if x.strip() != "void"]
        kinds = ["p" if "*" in x else "l" if "int64" in x else "f" if "float" in x else "i" for x in args]
        assert kinds == [names.get(t.__name__, "p") for t in _lib.SIGNATURES[m.group(1)][1]], m.group(1)


def test_streamed_argument_validation_without_gpu():
    lib = _lib.lib()
    buf = (ctypes.c_float * 64)()
    p = ctypes.cast(buf, ctypes.c_void_p)
    assert lib.based_add_norm(None, None, None, None, None, 1, 8, 8, 8, 8, 8, 1e-5, 1, 1.0, 0, None) == 4
    # nine taps -> BASED_ERR_SHAPE; in place -> BASED_ERR_ARG
    q = ctypes.c_void_p(p.value + 64)
    assert lib.based_stream_conv(p, p, None, q, None, None, 0, 1, 1, 8, 9, 8, 8, 8, 8, 0, 0, 0, 0, None) == 1
    assert lib.based_stream_conv(p, p, None, p, None, None, 0, 1, 1, 8, 4, 8, 8, 8, 8, 0, 0, 0, 0, None) == 4
    # three query heads over two key/value heads; a portion that runs past the cache
    tail = (0.1, 0, 0.0, 1.0, None, None, 0, 0, 0, 0, None)
    assert lib.based_window_attn_prefill(p, p, p, p, p, 0, 1, 2, 3, 2, 8, 8, 4, *([8] * 10), 4, *tail) == 1
    assert lib.based_window_attn_prefill(p, p, p, p, p, 3, 1, 2, 2, 2, 8, 8, 4, *([8] * 10), 4, *tail) == 1
    # query/key size above 256
    assert lib.based_gated_delta_scan(*([p] * 10), 1, 1, 1, 1, 264, 8, 8, 8, 8, 8, 8, 1, 0, None) == 1
    # channels that do not divide into blocks
    assert lib.based_rglru_prefill(*([p] * 12), 1, 1, 10, 3, *([8] * 6), 8.0, 1, 0, None) == 1
    assert b"blocks" in lib.based_hip_last_error()


def test_rglru_scratch_wherever_elements_are_shared():
    """An output that shares an element with the input gets a scratch, columns beside the input's in the same rows get none."""
    import itertools

    lib = _lib.lib()
    none = 0
    for B, L, W, sl, sb, size, code in itertools.product((1, 2), (1, 3), (2, 3), (3, 6, 7), (3, 6, 14, 21, 25), (2, 4), (0, 1)):
        if size != (2 if code == _lib.BASED_BF16 else 4):
            continue
        u = {b * sb + t * sl + w for b in range(B) for t in range(L) for w in range(W)}
        for at in range(-60, 61):
            floats = lib.based_rglru_prefill_work(4096, 4096 + at * size, B, L, W, sb, sl, sb, sl, code)
            meet = any(x + at in u for x in u)
            assert floats in (0, (B * L * W * size + 3) // 4) and (floats or not meet), (B, L, W, sl, sb, at)
            none += not floats and min(u) < max(u) + at and max(u) > min(u) + at
    assert none > 100  # (side by side, stretches of memory overlapping)
    # other strides: whatever overlaps
    assert lib.based_rglru_prefill_work(4096, 4096 + 8, 1, 3, 2, 8, 4, 8, 8, 1) > 0
    assert lib.based_rglru_prefill_work(4096, 4096 + 4 * 64, 1, 3, 2, 8, 4, 8, 8, 1) == 0


def test_decay_work_is_for_the_form_that_runs():
    """Aligned bf16 (the matrix form) asks for its own segments, everything else for those of the general form; one number covers both."""
    lib = _lib.lib()

    def of(B, L, H, D, DV, code, q=4096, log2=4096, pad=0):
        bits = q | 8192 | log2 // 2  # the addresses of the tensors, twice their strides
        for stride in (L * (H * D + pad), H * D + pad, L * H * DV, H * DV):
            bits |= 2 * stride
        return lib.based_decay_scan_work_of(bits, B, L, H, D, DV, (D + 3) // 4 * 4, code)

    floats = lambda segs, B, H, D, DV: B * H * segs * (DV + 1) * ((D + 3) // 4 * 4)  # noqa: E731
    for B, L, H, D, DV, mfma, general in [(1, 256, 16, 64, 64, 0, 4), (1, 2048, 16, 64, 64, 8, 32), (4, 2048, 16, 64, 64, 8, 8),
                                          (1, 100, 16, 64, 64, 0, 0), (8, 257, 16, 64, 64, 0, 0), (8, 320, 16, 64, 64, 0, 3), (64, 2048, 16, 64, 64, 0, 0)]:
        assert of(B, L, H, D, DV, 0) == floats(mfma, B, H, D, DV), (B, L)
        for other in (dict(code=1), dict(code=0, q=4098), dict(code=0, q=4100), dict(code=0, log2=4104), dict(code=0, pad=1), dict(code=0, pad=2)):
            assert of(B, L, H, D, DV, **other) == floats(general, B, H, D, DV), (B, L, other)
        assert lib.based_decay_scan_work(B, L, H, D, DV, 64) == floats(max(mfma, general), B, H, D, DV)
    from based_amd import ops

    header = open(os.path.join(ROOT, "include", "based_hip.h")).read()
    least = int(re.search(r"#define BASED_DECAY_SEGMENTS_MIN (\d+)", header).group(1))
    assert least == ops.DECAY_SEGMENTS_MIN
    for D in (4, 64, 128, 256):  # what is not asked about would take none, and the least that takes some is asked about
        assert lib.based_decay_scan_work(1, least - 1, 1, D, 4, D) == 0 and lib.based_decay_scan_work(1, least, 1, 64, 4, 64) > 0


def test_delta_chunks_take_the_rows_they_can():
    """What the library says about tensors is what the chunks' entry takes: no rows off 16 bytes above 64 channels, none too long, and a
    batch stride counts only where there is a batch."""
    from based_amd import ops

    lib = _lib.lib()

    def of(B=1, L=640, H=4, D=128, DV=64, q=4096, k=8192, sb=640 * 1280, sl=1280):
        return lib.based_gated_delta_scan_work_of(q, k, B, L, H, D, DV, sb, sl)

    full = lib.based_gated_delta_scan_work(1, 640, 4, 128, 64)
    assert of() == full > 0 and of(sb=640 * 1280 + 1) == full and of(B=2) > 0
    for refused in (dict(B=2, sb=640 * 1280 + 1), dict(sl=1281), dict(q=4100), dict(k=8200), dict(sl=1 << 24), dict(L=100), dict(D=130)):
        assert of(**refused) == 0, refused
    assert of(D=64, sl=1281, q=4100) == lib.based_gated_delta_scan_work(1, 640, 4, 64, 64) > 0
    header = open(os.path.join(ROOT, "include", "based_hip.h")).read()
    assert int(re.search(r"#define BASED_DELTA_CHUNKS_MIN (\d+)", header).group(1)) == ops.DELTA_CHUNKS_MIN
    for D in (8, 16, 32, 48, 64, 96, 128):  # what is not asked about would not be taken
        assert lib.based_gated_delta_scan_work(1, ops.DELTA_CHUNKS_MIN - 1, 1, D, 16) == 0
    p = ctypes.c_void_p(4096)
    chunks = lambda L, D, sl: lib.based_gated_delta_scan_chunks(*([p] * 10), 1, L, 4, 4, D, 64, 64, L * sl, sl, 4, 4, 1, 0, None)  # noqa: E731
    assert chunks(640, 132, 1280) == 1 and chunks(100, 128, 1280) == 1 and chunks(640, 128, 1 << 24) == 1  # BASED_ERR_SHAPE
    assert chunks(640, 128, 1281) == 3  # BASED_ERR_ALIGN


def test_delta_work_of_no_type_serves_either_type():
    """A shape that the queries without a type send through chunks of 64 tokens goes through them in either type, in no more work space: few
    and many heads, channels and values on both sides of every tile count, lengths on both sides of the first chunks."""
    lib = _lib.lib()
    taken = 0
    for B, H in [(1, 1), (1, 2), (1, 3), (2, 4), (1, 16), (3, 8), (4, 8), (6, 8), (4, 16), (5, 16), (8, 16), (9, 16)]:
        for D in (8, 16, 17, 32, 33, 48, 49, 64, 65, 96, 97, 112, 128, 129):
            for DV in (16, 17, 64, 128, 129, 256, 257, 272, 368, 369, 400, 512, 1024):
                for L in (255, 256, 319, 320, 383, 384, 447, 448, 512, 640, 1024, 1025, 2048, 4096):
                    floats = lib.based_gated_delta_scan_work(B, L, H, D, DV)
                    of = lib.based_gated_delta_scan_work_of(None, None, B, L, H, D, DV, 0, 8 * 128)
                    assert of == (floats if D <= 64 or D % 4 == 0 else 0)  # (rows of whole pieces above 64)
                    if of > 0:
                        taken += 1
                        for dtype in (_lib.BASED_BF16, _lib.BASED_F32):
                            own = lib.based_gated_delta_scan_work_as(None, None, B, L, H, D, DV, 0, 8 * 128, dtype)
                            assert 0 < own <= floats, (B, H, D, DV, L, dtype)
    assert taken > 2000


def test_delta_work_is_what_a_type_takes():
    """Queries and keys of bf16 are one part of three of fp32's, in the work space too."""
    lib = _lib.lib()
    for B, L, H, D, DV in [(4, 2048, 8, 64, 128), (1, 300, 8, 128, 128), (1, 512, 2, 64, 16)]:
        narrow, wide = (lib.based_gated_delta_scan_work_as(None, None, B, L, H, D, DV, 0, 4096, t) for t in (_lib.BASED_BF16, _lib.BASED_F32))
        chunks, tiles, values = B * H * ((L + 63) // 64), 4 if D <= 64 else 8, (DV + 15) // 16
        # operands of 1 KB: W (6 a tile of channels), queries, keys and outputs' weights in their parts, values in 32 bits; a row of factors
        assert narrow == chunks * (((6 + 2 + 2) * tiles + 18 + 4 * values) * 256 + 132)
        assert wide == chunks * (((6 + 4 + 6) * tiles + 18 + 4 * values) * 256 + 132)
