"""The prompt kernels against 64-bit attention, and the inputs they leave to
PyTorch.

Attention: 16-bit outputs and 16-bit weights in the value product, relative
2-norm error of at most 4e-3 (bf16, 2^-8 steps) / 5e-4 (f16).  Scores: 32-bit
logits of exact 16-bit products, 32-bit sums: 1e-6 + 1e-4 |ref| (weights in
[0, 1], the exponential's argument error scales with the logits)."""
import ctypes

import pytest
import torch
import torch.nn.functional as F
from torch.nn.attention import SDPBackend, sdpa_kernel

from wnw_amd import _lib
from wnw_amd.wnw import prompt, session

pytestmark = pytest.mark.gpu


def _qkv(dev, B, H, S, D, dtype, seed, layout):
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    if layout == "rows":  # [B, S, H, D] viewed as [B, H, S, D], as projections leave it
        return [torch.randn(B, S, H, D, device=dev, generator=g).to(dtype).transpose(1, 2) for _ in range(3)]
    return [torch.randn(B, H, S, D, device=dev, generator=g).to(dtype) for _ in range(3)]


@pytest.mark.parametrize("S", [1, 2, 31, 32, 33, 63, 64, 65, 127, 128, 129, 193, 500])
@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 128), (torch.float16, 128), (torch.bfloat16, 64),
                                     (torch.float16, 64)])
@pytest.mark.parametrize("layout", ["heads", "rows"])
def test_causal_attention(gpu, S, dtype, D, layout):
    q, k, v = _qkv(gpu, 2, 3, S, D, dtype, S, layout)
    out = session.prefill_attention(q, k, v, None, 0.11)
    assert prompt.causal_attention(q, k, v, 0.11) is not None
    assert out.stride() == q.stride() and out.dtype == dtype
    s = (q.double() @ k.double().transpose(-1, -2).contiguous()) * 0.11
    s = s + torch.full((S, S), float("-inf"), device=gpu, dtype=torch.float64).triu_(1)
    ref = s.softmax(-1) @ v.double().contiguous()
    err = float((out.double() - ref).norm() / ref.norm())
    assert err < (4e-3 if dtype == torch.bfloat16 else 5e-4), err


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 128), (torch.float16, 64)])
@pytest.mark.parametrize("H,Hkv", [(8, 2), (7, 1)])
def test_causal_attention_grouped(gpu, dtype, D, H, Hkv):
    """The C entry point with fewer KV heads than query heads."""
    B, S, scale = 2, 150, 0.1
    q = _qkv(gpu, B, H, S, D, dtype, 1, "rows")[0]
    k, v, _ = _qkv(gpu, B, Hkv, S, D, dtype, 2, "heads")
    out = torch.empty_like(q)
    strides = (ctypes.c_int64 * 12)(*(t.stride(i) for t in (q, k, v, out) for i in range(3)))
    _lib.check(_lib.lib().wnw_prefill_attn(_lib.ptr(q), _lib.ptr(k), _lib.ptr(v), B, H, Hkv, S, D, strides, scale,
                                           _lib.dtype_code(dtype), _lib.ptr(out), _lib.stream_of(gpu)))
    kk, vv = (t.repeat_interleave(H // Hkv, dim=1) for t in (k, v))
    assert torch.equal(out, prompt.causal_attention(q, kk, vv, scale))
    s = (q.double() @ kk.double().transpose(-1, -2).contiguous()) * scale
    s = s + torch.full((S, S), float("-inf"), device=gpu, dtype=torch.float64).triu_(1)
    ref = s.softmax(-1) @ vv.double().contiguous()
    err = float((out.double() - ref).norm() / ref.norm())
    assert err < (4e-3 if dtype == torch.bfloat16 else 5e-4), err


def test_causal_attention_large_scores(gpu):
    """Scores in the thousands and equal rows: the running maximum carries the
    sums, no overflow."""
    q, k, v = _qkv(gpu, 1, 2, 300, 128, torch.bfloat16, 9, "heads")
    q = q * 30
    k[:, :, 100:140] = k[:, :, 100:101]
    ref = ((q.double() @ k.double().transpose(-1, -2).contiguous()) +
           torch.full((300, 300), float("-inf"), device=gpu, dtype=torch.float64).triu_(1)).softmax(-1) @ v.double()
    out = prompt.causal_attention(q, k, v, 1.0)
    assert float((out.double() - ref).norm() / ref.norm()) < 4e-3


@pytest.mark.parametrize("dtype,tol", [(torch.bfloat16, 4e-3), (torch.float16, 5e-4)])
@pytest.mark.parametrize("step", [2.0, 7.5, 8.5])
def test_causal_attention_rising_scores(gpu, dtype, tol, step):
    """Scores that rise from one 64-key tile to the next, by less and by more
    than 8 in log2, and fall again: tiles that rescale the sums and tiles that
    do not."""
    q, k, v = _qkv(gpu, 1, 2, 700, 128, dtype, 11, "heads")
    q[..., 0] = 8.0
    tiles = torch.tensor([0, 1, 2, 3, 3, 4, 2, 5, 0, 6, 7], device=gpu, dtype=torch.float32)
    k[..., 0] = (tiles.repeat_interleave(64)[:700] * (step * 0.6931 / (8.0 * 0.08))).to(dtype)
    ref = ((q.double() @ k.double().transpose(-1, -2).contiguous()) * 0.08 +
           torch.full((700, 700), float("-inf"), device=gpu, dtype=torch.float64).triu_(1)).softmax(-1) @ v.double()
    out = prompt.causal_attention(q, k, v, 0.08)
    assert float((out.double() - ref).norm() / ref.norm()) < tol


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 128), (torch.float16, 128), (torch.bfloat16, 64),
                                     (torch.float16, 64)])
@pytest.mark.parametrize("deviation", [0.5, 1.0, 2.0, 4.0])
def test_causal_attention_no_less_exact_than_sdpa(gpu, dtype, D, deviation):
    """Flat to peaked rows against 64 bits, beside SDPA's fused kernels: the
    same rounding points (the largest weight is 1, 16-bit weights in the value
    product, 32-bit sums), so errors that differ by the order of the 32-bit sums
    only.  1 % of a 16-bit rounding is far above that (measured 0.01 %)."""
    q, k, v = _qkv(gpu, 1, 4, 1111, D, dtype, 21, "heads")
    q, scale = (q.float() * deviation).to(dtype), D ** -0.5
    ref = ((q.double() @ k.double().transpose(-1, -2).contiguous()) * scale +
           torch.full((1111, 1111), float("-inf"), device=gpu, dtype=torch.float64).triu_(1)).softmax(-1) @ v.double()
    with sdpa_kernel([SDPBackend.FLASH_ATTENTION, SDPBackend.EFFICIENT_ATTENTION]):
        sdpa = F.scaled_dot_product_attention(q, k, v, is_causal=True, scale=scale)
    err, theirs = (float((x.double() - ref).norm() / ref.norm()) for x in (prompt.causal_attention(q, k, v, scale), sdpa))
    assert err <= 1.01 * theirs, (err, theirs)


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 128), (torch.float16, 64)])
@pytest.mark.parametrize("S", [1, 33, 65, 127, 200, 256])
@pytest.mark.parametrize("value", [float("inf"), float("-inf")])
def test_causal_attention_infinite_last_value(gpu, dtype, D, S, value):
    """An infinity in the last row of V: the last query's output is that
    infinity, as SDPA gives it, and no query before the row's 64-key tile sees
    it (within the tile 0 * infinity is NaN there too)."""
    q, k, v = _qkv(gpu, 1, 2, S, D, dtype, S, "heads")
    v[:, :, -1, 5] = value
    out = prompt.causal_attention(q, k, v, 0.1)
    assert (out[:, :, -1, 5] == value).all()
    assert torch.isfinite(out[:, :, :(S - 1) // 64 * 64]).all()
    assert torch.isfinite(torch.cat([out[..., :5], out[..., 6:]], dim=-1)).all()


def test_inputs_left_to_torch(gpu):
    q, k, v = _qkv(gpu, 1, 2, 40, 128, torch.bfloat16, 3, "heads")
    assert prompt.causal_attention(q, k, v, 0.1) is not None
    assert prompt.causal_attention(q, k, v, -0.1) is None  # the running maximum needs a positive scale
    assert prompt.causal_attention(q, k[:, :, :30], v[:, :, :30], 0.1) is None
    assert prompt.causal_attention(q.float(), k.float(), v.float(), 0.1) is None
    wide = torch.randn(1, 2, 40, 129, device=gpu).to(torch.bfloat16)
    assert prompt.causal_attention(wide[..., 1:], k, v, 0.1) is None  # rows not 16-byte aligned
    for t in (q, k, v):
        t.requires_grad_(True)
    assert prompt.causal_attention(q, k, v, 0.1) is None
    out = session.prefill_attention(q, k, v, None, 0.1)
    out.float().sum().backward()
    assert q.grad is not None and k.grad is not None and v.grad is not None
    with torch.no_grad():
        assert prompt.causal_attention(q, k, v, 0.1) is not None
    q, k, v = (t.detach() for t in (q, k, v))
    got = torch.func.vmap(lambda a: session.prefill_attention(a, k, v, None, 0.1))(torch.stack([q, q]))
    torch.testing.assert_close(got[0], session.prefill_attention(q, k, v, None, 0.1), atol=2e-2, rtol=2e-2)


def test_traced_programs_record_torch_operators(gpu):
    """torch.jit.trace sees operators only: a launch behind its back would
    leave the traced program with unwritten memory."""
    q, k, v = _qkv(gpu, 1, 4, 96, 128, torch.bfloat16, 3, "heads")
    q2 = _qkv(gpu, 1, 4, 96, 128, torch.bfloat16, 4, "heads")[0]
    traced = torch.jit.trace(lambda a, b, c: session.prefill_attention(a, b, c, None, 0.1), (q, k, v), check_trace=False)
    want = session.prefill_attention(q2, k, v, None, 0.1)
    torch.testing.assert_close(traced(q2, k, v), want, atol=2e-2, rtol=2e-2)
    cache = _Cache(_Config([0], 2, "mean_text"), [2], [90])

    def scores(a, b):
        class_a, per_head = session.compute_prefill_scores(a, b, None, cache, 0, 2, 2, 0.1)
        return class_a[0], per_head[0][1]

    traced = torch.jit.trace(scores, (q, k[:, :2]), check_trace=False)
    for x, y in zip(traced(q2, k[:, :2]), scores(q2, k[:, :2])):
        torch.testing.assert_close(x, y, atol=1e-3, rtol=2e-2)


class _Config:
    def __init__(self, a_heads, group, mode):
        self.prefill_score_mode, self._a, self._g = mode, a_heads, group

    def get_layer_class_a(self, layer):
        return self._a

    def is_class_a_kv_head(self, layer, h):
        return h in {x // self._g for x in self._a}


class _Cache:
    def __init__(self, config, starts, ends):
        self.config, self._raw_audio_starts, self._raw_audio_ends = config, starts, ends


@pytest.mark.parametrize("dtype,D,G,H,S", [(torch.bfloat16, 128, 4, 4, 700), (torch.float16, 64, 7, 2, 257),
                                           (torch.float32, 128, 2, 3, 300), (torch.bfloat16, 256, 1, 2, 65),
                                           (torch.float32, 256, 3, 2, 130)])
@pytest.mark.parametrize("mode", ["last", "mean_text"])
@pytest.mark.parametrize("mask", ["none", "float", "bool", "lowest"])
def test_token_scores(gpu, dtype, D, G, H, S, mode, mask):
    """Two samples: text after the audio of one (more queries than fit the LDS
    at a time at 700 rows), none after the other's; masks additive, boolean,
    and with the type's lowest value instead of -inf."""
    B, starts, ends = 2, [5, 1], [S // 3, S]
    q = _qkv(gpu, B, G * H, S, D, dtype, 1, "rows")[0]
    k = _qkv(gpu, B, H, S, D, dtype, 2, "heads")[0]
    base = torch.ones(B, 1, S, S, device=gpu).tril_().bool()
    base[1, :, :, :2] = False
    base[1, :, :2, :2] = True
    m = {"none": None, "bool": base,
         "float": torch.where(base, 0.0, float("-inf")).to(dtype) + torch.rand(S, device=gpu).to(dtype),
         "lowest": torch.where(base, 0.0, torch.finfo(dtype).min).to(dtype)}[mask]
    a_heads = [0, G - 1] if G > 1 else [0]
    cache = _Cache(_Config(a_heads, G, mode), starts, ends)
    got = session.compute_prefill_scores(q, k, m, cache, 0, H, G, D ** -0.5)
    m64 = None if m is None else (torch.where(m, 0.0, float("-inf")) if mask == "bool" else m).double()
    want = _scores64(q.double(), k.double(), m64, cache, H, G, D ** -0.5)
    assert _lib.device_error() == 0
    for b in range(B):
        pairs = [(got[0][b], want[0][b])] + list(zip(got[1][b], want[1][b]))
        for x, y in pairs:
            assert (x is None) == (y is None)
            if x is not None:
                assert x.dtype == torch.float32 and x.shape == y.shape
                torch.testing.assert_close(x.double(), y, atol=1e-6, rtol=1e-4)


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("deviation", [1.0, 3.0])
def test_fp32_token_scores_no_less_exact_than_torch(gpu, monkeypatch, D, deviation):
    """fp32 scores against 64 bits, beside the PyTorch form's, root mean square
    over 16 inputs: 0.5 to 0.95 of it by the order of the sums; a dot as one
    chain of multiply-adds is at 1.5 to 3."""
    H, G, S = 3, 4, 900
    cache = _Cache(_Config([0, 2], G, "last"), [14], [850])
    native, sums = session.token_scores, {}
    for seed in range(16):
        q, k, _ = _qkv(gpu, 1, H * G, S, D, torch.float32, seed, "heads")
        q, k = q * deviation, k[:, :H].contiguous()
        want = _scores64(q.double(), k.double(), None, cache, H, G, D ** -0.5)
        for name, f in (("kernel", native), ("torch", lambda *a: None)):
            monkeypatch.setattr(session, "token_scores", f)
            got = session.compute_prefill_scores(q, k, None, cache, 0, H, G, D ** -0.5)
            for part, x, y in (("class A", got[0][0], want[0][0]), ("head", got[1][0][1], want[1][0][1])):
                e = float((x.double() - y).norm() / y.norm())
                sums[name, part] = sums.get((name, part), 0.0) + e * e
    for part in ("class A", "head"):
        ours, theirs = (sums[n, part] ** 0.5 / 4 for n in ("kernel", "torch"))
        print(f"prompt scores D={D} deviation={deviation} {part}: {ours:.3e}, torch {theirs:.3e}", flush=True)
        assert ours <= 1.2 * theirs, (part, ours, theirs)


def _scores64(q, k, m, cache, H, G, scale):
    """compute_prefill_scores in 64 bits."""
    B, _, S, _ = q.shape
    if m is None:
        m = torch.full((S, S), float("-inf"), device=q.device, dtype=torch.float64).triu_(1).expand(B, 1, S, S)
    cfg = cache.config
    a, per = [], []
    for b in range(B):
        ra, re = cache._raw_audio_starts[b], cache._raw_audio_ends[b]
        ca = cfg.get_layer_class_a(0)
        a.append(((q[b, ca, -1] @ k[b, ca[0] // G].t()) * scale + m[b, 0, -1]).softmax(-1)[:, ra:re].sum(0))
        row = []
        for h in range(H):
            if cfg.is_class_a_kv_head(0, h):
                row.append(None)
                continue
            rows = slice(S - 1, S) if cfg.prefill_score_mode == "last" else slice(re, S)
            if rows.start == S:
                row.append(torch.zeros(re - ra, device=q.device, dtype=torch.float64))
                continue
            s = (q[b, h * G:(h + 1) * G, rows] @ k[b, h].t()) * scale + m[b, 0, rows]
            row.append(s.softmax(-1)[:, :, ra:re].mean(dim=1).sum(0))
        per.append(row)
    return a, per
