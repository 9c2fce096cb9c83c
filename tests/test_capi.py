"""The C-ABI library loads (no GPU needed) and exports every declared symbol."""
import ctypes
import os
import re

from wnw_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared_functions():
    names = []
    for h in sorted(os.listdir(os.path.join(ROOT, "include"))):
        if not h.endswith(".h"):
            continue
        text = open(os.path.join(ROOT, "include", h)).read()
        text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
        names += re.findall(r"\b(wnw_[a-z0-9_]+)\s*\(", text)
    return sorted(set(names))


def test_header_declares_functions():
    names = _declared_functions()
    assert "wnw_decode_attn" in names and "wnw_interleave_append" in names and "wnw_rebuild_append_kv" in names


def test_library_exports_every_declared_symbol():
    handle = ctypes.CDLL(_lib.LIB_PATH)
    missing = [n for n in _declared_functions() if not hasattr(handle, n)]
    assert not missing, f"not exported: {missing}"


def test_python_binding_covers_every_symbol():
    declared = set(_declared_functions())
    bound = set(_lib.exported_symbols())
    assert declared <= bound, f"unbound: {sorted(declared - bound)}"
    _lib.lib()  # argtypes install without error


def test_host_only_queries_work_without_gpu():
    l = _lib.lib()
    assert l.wnw_abi_version() >= 1
    ws = l.wnw_decode_attn_workspace_bytes(64, 4, 128)
    assert ws > 0 and ws % 256 == 0
    assert l.wnw_decode_attn_workspace_bytes(64, 0, 128) == -1


def test_prefill_scores_refuses_reads_outside_its_tensors():
    """Heads outside the counts, negative strides and sizes beyond the
    kernel's are refused before anything is launched (the pointers are not
    looked at)."""
    good = dict(heads=8, kv_heads=2, a=[0, 7], kv=[1], strides=[65536, 8192, 128, 16384, 8192, 128, 4096, 64],
                most=256)

    def call(**change):
        c = {**good, **change}
        i32 = lambda x: (ctypes.c_int32 * len(x))(*x)  # noqa: E731
        p = ctypes.c_void_p(1 << 20)
        return _lib.lib().wnw_prefill_scores(
            p, p, p, (ctypes.c_int64 * 8)(*c["strides"]), 1, c["heads"], c["kv_heads"], 64, 128, i32([2]), i32([50]),
            i32(c["a"]), len(c["a"]), i32(c["kv"]), len(c["kv"]), 0, 0.1, _lib.DT_BF16, _lib.DT_BF16, 48, c["most"], p, p,
            p, 1 << 60, None)

    for i in range(8):
        assert call(strides=[-x if j == i else x for j, x in enumerate(good["strides"])]) == _lib.WNW_EINVAL
    for bad in (dict(a=[0, 8]), dict(a=[-1]), dict(kv=[2]), dict(kv=[0, -1]), dict(heads=7), dict(kv_heads=0),
                dict(heads=0), dict(most=1 << 31)):
        assert call(**bad) == _lib.WNW_EINVAL, bad
