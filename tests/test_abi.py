"""CPU-side checks of the C-ABI library: it loads and exports what include/xsmi355.h declares."""
import ctypes
import itertools
import math
import os
import random
import re

import pytest

from xshinnosuke_amd.backend import capi as libmod

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared_symbols():
    text = open(os.path.join(ROOT, "include", "xsmi355.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(xsmi_[a-z0-9_]+)\s*\(", text)))


def test_header_symbols_are_bound_and_exported():
    declared = _declared_symbols()
    assert len(declared) >= 20
    assert sorted(libmod.SIGNATURES) == declared          # the Python binding covers the whole header
    dll = ctypes.CDLL(libmod.library_path())
    for name in declared:
        assert hasattr(dll, name), name


def test_calls_before_init_fail_with_a_message():
    dll = ctypes.CDLL(libmod.library_path())
    dll.xsmi_last_error.restype = ctypes.c_char_p
    dll.xsmi_is_initialized.restype = ctypes.c_int
    if dll.xsmi_is_initialized():
        pytest.skip("library already initialised in this process")
    assert dll.xsmi_sync() == 3
    assert b"xsmi_init" in dll.xsmi_last_error()


def test_workspace_query_needs_no_device():
    f = libmod.lib.raw("xsmi_conv2d_workspace_bytes")
    c2 = f(32, 64, 56, 56, 64, 3, 3, 1, 1, 1)
    assert c2 >= 64 * 576 * 4
    assert f(32, 64, 56, 56, 64, 3, 3, 0, 1, 1) == 0      # invalid stride -> 0
    assert f(1, 1, 2, 2, 1, 5, 5, 1, 1, 0) == 0           # filter larger than the input -> 0


def test_workspace_queries_of_tensors_that_are_too_large_give_zero():
    """Tensors of 2^29 elements or more are refused by every pass; their counts of pixels and stages do not fit 32 bits."""
    whole = libmod.lib.raw("xsmi_conv2d_workspace_bytes")
    one = libmod.lib.raw("xsmi_conv2d_pass_workspace_bytes")
    for dims in ((65536, 16, 256, 256, 16, 3, 3, 1, 1, 1),            # 2^32 output pixels
                 (65536, 16, 256, 256, 16, 5, 5, 1, 1, 2), (1 << 20, 16, 1024, 1024, 16, 3, 3, 1, 1, 1),
                 (1, 1 << 15, 8, 8, 1 << 15, 3, 3, 1, 1, 1),          # a filter that is too large
                 (8192, 16, 64, 64, 16, 3, 3, 1, 1, 1)):              # 2^29 elements
        assert whole(*dims) == 0 and all(one(*dims, p, f) == 0 for p in range(3) for f in (0, libmod.CONV_BF16)), dims
    assert whole(8191, 16, 64, 64, 16, 3, 3, 1, 1, 1) > 0


def test_per_pass_workspace_queries_need_no_device():
    """The size of one pass alone never exceeds the size for all passes, the maximum over passes and flags is that
    size, a pass outside 0..2 and a bad geometry give 0; what the library holds itself is a constant."""
    whole = libmod.lib.raw("xsmi_conv2d_workspace_bytes")
    one = libmod.lib.raw("xsmi_conv2d_pass_workspace_bytes")
    for dims in ((32, 64, 56, 56, 64, 3, 3, 1, 1, 1), (32, 64, 56, 56, 128, 3, 3, 2, 2, 1), (32, 3, 224, 224, 64, 7, 7, 2, 2, 3),
                 (2, 5, 9, 11, 70, 3, 2, 1, 2, 2), (32, 512, 7, 7, 512, 3, 3, 1, 1, 1)):
        sizes = [one(*dims, p, f) for p in range(3) for f in (0, libmod.CONV_BF16)]
        assert all(0 < v <= whole(*dims) for v in sizes), dims
        assert max(sizes) == whole(*dims), dims
        assert one(*dims, 3, 0) == 0 and one(*dims, -1, 0) == 0
    # a layout workspace of the benchmark layer is the packed filter, not the split partials of the weight gradient
    c2 = (32, 64, 56, 56, 64, 3, 3, 1, 1, 1)
    assert one(*c2, 0, 0) < 1 << 20 and one(*c2, 1, 0) < 1 << 20 and one(*c2, 2, 0) > 8 << 20
    assert one(32, 64, 56, 56, 64, 3, 3, 0, 1, 1, 0, 0) == 0
    assert libmod.lib.raw("xsmi_scratch_bytes")() >= libmod.NOALLOC_SCRATCH_BYTES


def _split_wgrad_plan(n, c, h, w, k, r, s, sh, sw, pad):
    """Workspace bytes of the split weight gradient whose tile and split have the least estimated time of all (the model of
    conv_split_wgrad.hip, every tile and split tried); None where no tile fits."""
    up = lambda a, b: -(-a // b)  # noqa: E731
    oh, ow = (h + 2 * pad - r) // sh + 1, (w + 2 * pad - s) // sw + 1
    sx, pixels, pairs = 1 if s == 1 or ow == 1 else sw, n * oh * ow, up(up(c, 8) * r, 2)
    best = None
    for kt, px, nj, p in itertools.product((64, 32), (64, 32), (2, 3), (2, 3, 4, 5)):
        slots = (px - 1) * sx + (px - 1 + ow - 1) // ow * max(s - sx, 0) + s
        slots += (12 - slots % 8) % 8
        dy = kt // 8 * px
        subs = min(256 * p // kt // s, pairs)
        if slots > 510 or (nj == 3 and subs <= (1024 - dy) // (2 * slots)):
            continue
        subs = min(subs, (nj * 512 - dy) // (2 * slots))
        if subs < 1:
            continue
        across, rows, stages = up(pairs, subs), up(k, kt), up(pixels, px)
        tiles = across * rows
        stage = 55.0 * p * 6 * (px // 32) + 264.0 * ((dy + 2 * up(pairs, across) * slots) / 512) + 250.0
        once = 256 // tiles if tiles < 256 else 1
        for splits in (once, once // 2, once // 4, once // 8, 512 // tiles, 768 // tiles):
            splits = min(splits, 256, stages)
            if splits < 1:
                continue
            splits = up(stages, up(stages, splits))
            cost = up(tiles * splits, 256) * (up(stages, splits) + 1) * stage + tiles * splits * p * 16 * 0.6
            if best is None or cost < best[0]:
                best = cost, up(splits * tiles * 4096 * p * 4, 256) * 256 + up(splits * k * 4, 256) * 256
    return best and best[1]


def test_split_weight_gradient_plan_is_the_least_of_all_tiles():
    """The plan leaves tiles out by what they cost at least; it is the one that trying them all finds."""
    one = libmod.lib.raw("xsmi_conv2d_pass_workspace_bytes")
    option = lambda v: libmod.lib.call("xsmi_set_option", b"conv_split", v)  # noqa: E731
    rng = random.Random(7)
    log = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))  # noqa: E731
    seen = 0
    try:
        while seen < 2000:
            r, s, pad = rng.choice((1, 2, 3, 3, 5, 7, 16)), rng.choice((1, 2, 3, 3, 5, 7, 16)), rng.choice((0, 1, 3))
            dims = (log(1, 128), log(1, 600), log(1, 130), log(1, 130), log(1, 600), r, s, rng.choice((1, 1, 2, 3)), rng.choice((1, 1, 2, 3)), pad)
            option(0)
            plain = one(*dims, 2, 0)
            option(2)
            if plain:
                plan = _split_wgrad_plan(*dims)
                assert one(*dims, 2, 0) == max(plain, plan or 0), dims
                seen += plan is not None and plan > plain
    finally:
        option(1)
