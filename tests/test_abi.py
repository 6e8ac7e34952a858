"""The C-ABI library loads without a GPU and exports every entry point include/mi355moe.h declares; argument
validation fails cleanly before any device work."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HDR = os.path.join(ROOT, "include", "mi355moe.h")


def declared():
    src = open(HDR).read()
    src = re.sub(r"/\*.*?\*/", "", src, flags=re.S)
    return sorted(set(re.findall(r"\b(mm_[a-z0-9_]+)\s*\(", src)))


def test_header_declares_entry_points():
    names = declared()
    for must in ("mm_split", "mm_combine_host", "mm_permute", "mm_combine", "mm_expert_gemv", "mm_router_topk"):
        assert must in names


def test_library_exports_every_declared_symbol():
    from mi355moe import _lib
    L = _lib.load()
    out = subprocess.run(["nm", "-D", "--defined-only", _lib.LIB_PATH], capture_output=True, text=True, check=True).stdout
    exported = set(re.findall(r" T (mm_[a-z0-9_]+)$", out, flags=re.M))
    for name in declared():
        assert name in exported, name
        assert getattr(L, name) is not None
        assert name in _lib.EXPORTS, name


def test_argument_errors_without_device_work():
    from mi355moe import _lib
    L = _lib.load()
    assert L.mm_version() == 100
    rc = L.mm_split(None, None, None, 32, 4, 4096, 2000, None, None, None, None, None, None, None, 0, None, None, None,
                    None, None, None, None, None, None)
    assert rc == -1 and b"E <= 1024" in L.mm_last_error()
    rc = L.mm_permute(None, None, 10, 8, 0, None, None, None, None, None, None, None, None, None, 0, None)
    assert rc == -1
    rc = L.mm_expert_gemv(None, None, 0, 0, 1, 1, 1, None, None, None, None, None, 1, None, None, 0, 31, None)
    assert rc == -1 and b"incomplete layer" in L.mm_last_error()
    with pytest.raises(RuntimeError, match="mm_combine"):
        _lib.call("mm_combine", None, None, None, None, 1, 1, 4096, 8, 0, None)
    assert L.mm_permute_workspace(100, 384) == 0 and L.mm_permute_workspace(131072, 384) > 0
    # transformed gate/up inputs, 8 K parts of gate/up partial sums, the down input, 4 K parts of down partials
    assert L.mm_gemv_workspace(36, 385, 4096, 2048) >= (36 * 2 * 4096 * 2 + 8 * 36 * 2 * 2048 * 4 + 36 * 2048 * 2
                                                        + 4 * 36 * 4096 * 4)
    assert L.mm_gemv_workspace(0, 385, 4096, 2048) == 0


@pytest.mark.parametrize("H,I", [(1024, 512), (4096, 2048), (5120, 2304)])
def test_scratch_holds_every_call_of_64_mib_with_one_record_per_expert(H, I):
    """mm_moe_decode_noalloc takes every call (up to 1,024 routes) whose decode arrays, with one 48-byte record per active
    expert, fill at most 64 MiB: the records of 16 routes of larger calls come on top of that."""
    from mi355moe import _lib
    L = _lib.load()
    scratch = eval(re.search(r"#define MM_NOALLOC_SCRATCH_BYTES (.*)", open(HDR).read()).group(1).replace("(size_t)", ""))
    al = lambda v: (v + 255) & ~255
    for E in (8, 128, 384, 1024):
        for n in range(1, 1025):
            cap, nb = min(32, max(4, 8192 // n)), (H + 511) // 512
            one = (al(min(n, E) * 48) + al(8) + 5 * al(n * 4) + al(n * 2 * H * 2) + al(n * 2 * nb * 4)
                   + al(cap * n * 2 * I * 4) + al(n * I * 2) + al(n * (I // 128) * 4) + al(cap * n * H * 4))
            need = L.mm_gemv_workspace(n, E, H, I)
            assert one <= need <= one + al(n // 16 * 48), (E, n)
            if one <= 64 << 20:
                assert need <= scratch, (E, n)


def test_route_limit_counts_one_record_per_expert():
    """The limit on a partial launch's tile rows holds for one record per expert: 8,000 routes over 16 experts of 65,536 x
    65,536 pass it (records of 16 routes would not) and fail on the workspace, argument checks only."""
    import ctypes
    from mi355moe import _lib
    L = _lib.load()
    lay = _lib.MMLayer(*([256] * 7), 16, 65536, 65536, 10.0, 0)
    rc = L.mm_expert_gemv(ctypes.byref(lay), 256, 0, 0, 4000, 8000, 2, 256, 256, 256, 256, 256, 8000, 256, None, 0, 31, None)
    assert rc == -1 and b"workspace too small" in L.mm_last_error(), L.mm_last_error()


@pytest.mark.parametrize("E,H,I,k", [(384, 4096, 2048, 8), (384, 5120, 2304, 6), (8, 4096, 2048, 2), (64, 4096, 2048, 6),
                                     (32, 1024, 512, 4), (4, 256, 128, 1), (1024, 1024, 1024, 1)])
def test_fused_workspace_holds_every_smaller_call(E, H, I, k):
    """mm_fused_moe_workspace grows with the tokens, and is at least what a call asks for (read from the argument error of a
    call without any), on both sides of every change of path."""
    import ctypes
    from mi355moe import _lib
    L = _lib.load()
    lay = _lib.MMLayer(*([256] * 7), E, H, I, 10.0, 0)
    had = 0
    for T in sorted(set(range(1, 3000, 7)) | {384 // k, 384 // k + 1, 1024 // k, 1024 // k + 1}):
        rc = L.mm_fused_moe(ctypes.byref(lay), 256, 0, T, k, 256, 256, 32, 256, 256, 0, None)
        m = re.search(rb"workspace too small \(0 < (\d+)\)", L.mm_last_error())
        assert rc == -1 and m, L.mm_last_error()
        ws = L.mm_fused_moe_workspace(T, k, E, H, I, 32)
        assert ws >= int(m.group(1)) and ws >= had, T
        had = ws


@pytest.mark.parametrize("T,cap", [(16384, 32), (16384, 400), (16384, 1 << 30), (128, 400)])
def test_fused_call_is_not_refused_by_its_threshold(T, cap):
    """A fused call of 16,384 tokens, top-8 of 384 experts at H 4096 passes the argument checks whatever the threshold
    (E x cap positions of 400 would pass 2 GiB of inputs, but no path holds them) and fails on the missing workspace; thresholds
    below 1 and more routes than the decode path can address on it stay errors."""
    import ctypes
    from mi355moe import _lib
    L = _lib.load()
    lay = _lib.MMLayer(*([256] * 7), 384, 4096, 2048, 10.0, 0)
    rc = L.mm_fused_moe(ctypes.byref(lay), 256, 0, T, 8, 256, 256, cap, 256, 256, 0, None)
    assert rc == -1 and b"workspace too small" in L.mm_last_error(), L.mm_last_error()
    rc = L.mm_fused_moe(ctypes.byref(lay), 256, 0, T, 8, 256, 256, 0, 256, 256, 1 << 40, None)
    assert rc == -1 and b"cap < 1" in L.mm_last_error()
    wide = _lib.MMLayer(*([256] * 7), 384, 1 << 19, 128, 10.0, 0)
    rc = L.mm_fused_moe(ctypes.byref(wide), 256, 0, 128, 8, 256, 256, cap, 256, 256, 1 << 50, None)
    assert rc == -1 and b"too many routes" in L.mm_last_error(), L.mm_last_error()


def test_expert_seed_matches_oracle():
    import oracle as O
    from mi355moe import _lib
    L = _lib.load()
    for ls, e in ((1000, 0), (1039, 384), (2**40 + 3, 17)):
        assert L.mm_expert_seed(ls, e) == O.expert_seed(ls, e)
