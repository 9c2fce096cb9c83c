"""The operators' native plain form (_callpath): the same results as the
general path, and every call it does not take left to that path."""
import sys

import pytest
import torch

import wnw_amd
from wnw_amd import _lib
from wnw_amd.kv.fused_attn import AttnWorkspace, decode_attn
from wnw_amd.wnw.kernels import fused_score_accumulate


def test_host_tensors_are_left_to_the_general_path():
    q, k = torch.zeros(2, 4, 128), torch.zeros(8, 128)
    cu = torch.tensor([0, 4, 8], dtype=torch.int32)
    native = _lib.callpath()
    assert native.attn(q, k, k, cu, 1.0, None, None, None, None) is None
    assert native.score(q, k, cu, cu, cu, cu, q, cu, 4, 1.0) is None
    assert native.attn(None, 3, "k", cu, 1.0, None, None, None, None) is None
    with pytest.raises(TypeError):
        native.attn(q)
    with pytest.raises(_lib.WnwError, match="GPU tensors"):
        decode_attn(q, k, k, cu, 1.0)


def test_missing_extension_names_the_build(monkeypatch):
    monkeypatch.setattr(_lib, "_callpath", None)
    monkeypatch.setitem(sys.modules, "wnw_amd._callpath", None)
    monkeypatch.delattr(wnw_amd, "_callpath", raising=False)
    with pytest.raises(RuntimeError, match="_callpath.so.*build the HIP extension"):
        decode_attn(torch.zeros(2, 4, 128), torch.zeros(8, 128), torch.zeros(8, 128), torch.zeros(3), 1.0)


def _segments(gpu, dtype, group, append):
    gen = torch.Generator(device=gpu)
    gen.manual_seed(3)
    lens = [1, 16, 333, 0, 65] if not append else [1, 16, 333, 7, 65]
    d, n, slack = 128, len(lens), 8

    def rnd(*s):
        return torch.randn(*s, device=gpu, generator=gen).to(dtype)

    cu = torch.tensor([0] + lens, dtype=torch.int32, device=gpu).cumsum(0).to(torch.int32)
    caps = [x + slack for x in lens]
    base = torch.tensor([sum(caps[:i]) for i in range(n)], dtype=torch.int64, device=gpu)
    k, v = rnd(sum(caps), d), rnd(sum(caps), d)
    rows = sum(lens) + n
    new = (rnd(n, d), rnd(n, d), torch.empty_like(cu), torch.tensor(caps, dtype=torch.int32, device=gpu))
    return rnd(n, group, d), k, v, cu, base, rows, new if append else None


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("group,append", [(1, False), (4, True), (16, True)])
def test_same_as_the_general_path(gpu, dtype, group, append):
    q, k, v, cu, base, rows, new = _segments(gpu, dtype, group, append)
    res = []
    for general in (False, True):
        kk, vv = k.clone(), v.clone()
        app = None if new is None else (new[0], new[1], torch.zeros_like(cu), new[3])
        out = decode_attn(q, kk, vv, cu, 0.1, seg_base=base, total_rows=rows, append=app,
                          workspace=AttnWorkspace(gpu) if general else None)
        res.append((out, kk, vv) + ((app[2],) if app else ()))
    for a, b in zip(*res):
        assert torch.equal(a, b)
    given = torch.empty_like(q)  # out: written and returned itself
    assert decode_attn(q, k, v, cu, 0.1, seg_base=base, total_rows=rows, out=given) is given
    # forms the native call leaves: strided q, offsets and bases
    strided = torch.empty(group, q.shape[0], q.shape[2], device=gpu, dtype=dtype).copy_(q.transpose(0, 1)).transpose(0, 1)
    cu2 = torch.stack([cu, cu], dim=1)[:, 0]
    assert not strided.is_contiguous() or group == 1
    assert torch.equal(decode_attn(strided, k, v, cu2, 0.1, seg_base=base, total_rows=rows), given)


@pytest.mark.gpu
def test_refusals_and_transforms(gpu):
    q, k, v, cu, base, rows, new = _segments(gpu, torch.bfloat16, 4, True)
    for bad in (dict(total_rows=None), dict(append=(new[0][:-1], *new[1:])), dict(append=(new[0], new[1], cu, new[3])),
                dict(append=(new[0].float(), *new[1:]))):
        with pytest.raises(_lib.WnwError):
            decode_attn(q, k, v, cu, 0.1, **{**dict(seg_base=base, total_rows=rows), **bad})
    with pytest.raises(_lib.WnwError):
        decode_attn(q.float(), k, v, cu, 0.1, seg_base=base, total_rows=rows)
    with pytest.raises(OverflowError):  # the general path's float(scale)
        decode_attn(q, k, v, cu, 10**400, seg_base=base, total_rows=rows)
    with pytest.raises(_lib.WnwError, match="group must be"):
        decode_attn(q.repeat(1, 8, 1), k, v, cu, 0.1, seg_base=base, total_rows=rows)
    with pytest.raises(RuntimeError):  # no storage under vmap
        torch.vmap(lambda x: decode_attn(x, k, v, cu, 0.1, seg_base=base, total_rows=rows))(torch.stack([q, q]))


@pytest.mark.gpu
def test_score_same_as_the_general_path(gpu):
    gen = torch.Generator(device=gpu)
    gen.manual_seed(4)
    q = torch.randn(2, 4, 128, device=gpu, generator=gen).bfloat16()
    k = torch.randn(900, 128, device=gpu, generator=gen).bfloat16()
    i32 = lambda *x: torch.tensor(x, dtype=torch.int32, device=gpu)  # noqa: E731
    s0, s1, a0, a1, off = i32(0, 500), i32(500, 900), i32(3, 9), i32(480, 390), i32(0, 477, 858)
    accs = []
    for strided in (False, True):
        acc = torch.zeros(858, device=gpu)
        st = torch.stack([s0, s0], dim=1)[:, 0] if strided else s0
        fused_score_accumulate(q, k, st, s1, a0, a1, acc, off, max_audio=477)
        accs.append(acc)
    assert torch.equal(*accs) and accs[0].sum().item() > 0
    with pytest.raises(_lib.WnwError):
        fused_score_accumulate(q, k, s0.long(), s1, a0, a1, accs[0], off, max_audio=477)
