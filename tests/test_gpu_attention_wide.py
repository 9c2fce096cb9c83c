"""The streaming attention kernel's wide instances (q through registers):
groups of 9 to 16 heads, 512-byte rows (fp32 head_dim 128, 16-bit head_dim
256) and fp32 head_dim 64, against the float64 oracle at the edges of their
16-row steps, wave ranges and segment table: fused append, dense operator
and kept logits.  Tolerances as in test_gpu_attention.py (16-bit outputs
2e-3 + 1e-2 |ref|, fp32 1e-4 + 1e-3 |ref|) and test_gpu_score.py (scores
1e-6 + 1e-3 |ref|: sums of weights from 32-bit logits)."""
import numpy as np
import pytest

from tests.helpers import allclose_report
from tests.test_gpu_attention import _append_case, _check_append, _run_case, _tol
from wnw_amd import _lib

pytestmark = pytest.mark.gpu

WIDE = [("float32", 4, 64), ("float32", 16, 64), ("float32", 1, 128), ("float32", 9, 128), ("bfloat16", 9, 64),
        ("float16", 16, 64), ("bfloat16", 13, 128), ("float16", 16, 128), ("bfloat16", 1, 256), ("float16", 8, 256),
        ("bfloat16", 16, 256)]


def _lens(n):
    """n segments: empty, one-row, around one and two 16-row steps, long."""
    edge = [0, 1, 15, 16, 17, 31, 32, 33, 48, 5000, 2, 64, 300]
    rng = np.random.default_rng(n)
    return (edge + [int(x) for x in rng.integers(0, 70, max(0, n - len(edge)))])[:n]


@pytest.mark.parametrize("n", [13, 64, 65, 150])
@pytest.mark.parametrize("dtype,G,D", WIDE)
def test_append_and_dense(gpu, dtype, G, D, n):
    """64 / 65 segments: the direct table and the table pass."""
    _check_append(_append_case(gpu, _lens(n), G, D, dtype, seed=G + n), dtype)
    for n_wg in (0, 1, 3):
        got, ref = _run_case(gpu, _lens(n), G, D, dtype, n_wg=n_wg, seed=D + n)
        ok, msg = allclose_report(got, ref, *_tol(dtype))
        assert ok, msg


@pytest.mark.parametrize("dtype,G,D", WIDE)
def test_append_with_scores(gpu, dtype, G, D):
    """The kept logits of the appended segments, scored by the logit pass."""
    lens = [40, 300, 17, 1000, 64, 2, 513, 90]
    r = _append_case(gpu, lens, G, D, dtype, seed=4, score=(4, [0, 1, 0, 1], [3, 0], [17, 2]))
    _check_append(r, dtype)
    acc, ref = r["extra"]
    ok, msg = allclose_report(acc.cpu().numpy().astype(np.float64), ref, 1e-6, 1e-3)
    assert ok, msg


@pytest.mark.parametrize("dtype,G,D", [("float32", 4, 128), ("bfloat16", 16, 128), ("bfloat16", 4, 256)])
def test_capacity_is_refused(gpu, dtype, G, D):
    """A segment without room for its new row: WNW_DEVERR_CAPACITY, and the
    row is not stored."""
    _check_append(_append_case(gpu, [40, 300, 5, 77], G, D, dtype, seed=9, short_cap=1), dtype, err=_lib.DEVERR_CAPACITY)


@pytest.mark.parametrize("dtype,G,D", [("float32", 4, 128), ("bfloat16", 16, 128), ("bfloat16", 5, 256)])
def test_many_segments_per_wave(gpu, dtype, G, D):
    """One workgroup over 300 segments: the walk changes windows, more new
    rows end in a wave than it keeps until the end."""
    rng = np.random.default_rng(5)
    lens = [int(x) for x in rng.integers(0, 24, 300)]
    _check_append(_append_case(gpu, lens, G, D, dtype, seed=8, rows_hint=64), dtype)


@pytest.mark.parametrize("dtype,G,D", [("bfloat16", 4, 128), ("float16", 16, 128), ("bfloat16", 7, 64),
                                       ("float32", 2, 128)])
@pytest.mark.parametrize("n_wg", [97, 150, 256, 1100])
def test_two_level_merge(gpu, dtype, G, D, n_wg):
    """Segments of more than 32 pieces (merged block by block) side by side,
    with one-row and empty segments between, at piece counts around whole
    blocks of 16; twice on one workspace, whose counters must be left at zero."""
    lens = [9000, 1, 4096, 0, 2, 4096, 5000, 1, 1, 1, 700]
    for seed in (1, 2):
        got, ref = _run_case(gpu, lens, G, D, dtype, n_wg=n_wg, seed=seed)
        ok, msg = allclose_report(got, ref, *_tol(dtype))
        assert ok, msg


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("G", [4, 16])
@pytest.mark.parametrize("nats", [12.0, 17.5, 20.0])
def test_weights_in_32_bits_beside_a_sink(gpu, dtype, G, nats):
    """head_dim 256, one workgroup: a row whose V is zero and whose score is far
    above the others', so that the output is made of weights of 6e-6 to 2e-9
    of the maximum, below what f16 holds.  Bound: the output's own rounding
    (2^-11 / 2^-8, in 2-norm 0.3 to 0.6 of that) and the 32-bit sums."""
    import torch

    from wnw_amd.kv.fused_attn import decode_attn

    n, D, dt = 6000, 256, getattr(torch, dtype)
    gen = torch.Generator(device=gpu)
    gen.manual_seed(int(nats))
    k = torch.randn(n, D, device=gpu, generator=gen) * 0.05
    k[:, 0] = 0
    k[3, 0] = nats
    v = torch.rand(n, D, device=gpu, generator=gen) + 0.5
    v[3] = 0
    v *= 2.0 ** min(14, round(nats * 1.4427 - 12.5))  # the output in the range of normal f16
    q = torch.randn(1, G, D, device=gpu, generator=gen) * 0.1
    q[..., 0] = 16.0
    q, k, v = q.to(dt), k.to(dt), v.to(dt)
    ref = ((q[0].double() @ k.double().t()) / 16).softmax(-1) @ v.double()
    cu = torch.tensor([0, n], dtype=torch.int32, device=gpu)
    out = decode_attn(q, k, v, cu, 1 / 16, n_wg=1)[0].double()
    err = float((out - ref).norm() / ref.norm())
    assert err < (4e-4 if dtype == "float16" else 3e-3), err


@pytest.mark.parametrize("dtype,G,D", [("float32", 4, 64), ("float32", 16, 128), ("bfloat16", 4, 256),
                                       ("float16", 16, 256)])
@pytest.mark.parametrize("append", [False, True])
def test_infinite_values(gpu, dtype, G, D, append):
    """An infinity in V's last row of a segment (the step's rows after it are
    copies of it, with weight 0) or in the row before it: the output is that
    infinity, in its column alone."""
    import torch

    from wnw_amd.kv.fused_attn import decode_attn

    lens, dt = [1, 17, 200, 33, 16, 5], getattr(torch, dtype)
    n, cap = len(lens), [x + 1 for x in lens]
    gen = torch.Generator(device=gpu)
    gen.manual_seed(6)
    rnd = lambda *s: torch.randn(*s, device=gpu, generator=gen)  # noqa: E731
    base = [sum(cap[:i]) for i in range(n)]
    q, k, v = rnd(n, G, D).to(dt), rnd(sum(cap), D).to(dt), rnd(sum(cap), D).to(dt)
    new_k, new_v = rnd(n, D).to(dt), rnd(n, D).to(dt)
    last = [b + x - 1 for b, x in zip(base, lens)]
    v[last[2], 9], v[last[3], 3], v[last[1] - 1, 4], v[last[5], 0] = float("inf"), float("-inf"), float("inf"), float("inf")
    if append:
        new_v[4, 7] = float("-inf")
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=gpu)  # noqa: E731
    cu = i32([0] + lens).cumsum(0).to(torch.int32)
    want = torch.zeros(n, D, device=gpu)
    want[2, 9], want[3, 3], want[1, 4], want[5, 0] = float("inf"), float("-inf"), float("inf"), float("inf")
    want[4, 7] = float("-inf") if append else 0
    app = (new_k, new_v, torch.empty_like(cu), i32(cap)) if append else None
    for rows in (sum(lens) + n, 64):  # several workgroups and one
        out = decode_attn(q, k.clone(), v.clone(), cu, 0.05, seg_base=torch.tensor(base, device=gpu), total_rows=rows,
                          append=app).float()
        assert torch.equal(torch.where(torch.isfinite(out), 0.0, out), want[:, None].expand_as(out))
