"""fused_score_accumulate on matrix instructions against the float64 oracle:
types, head counts and head sizes, items whose slices end inside 16-row
tiles or are empty, audio ranges that start and end inside a slice, many
items (8 slices each) and one (128), a query view that is not 16-byte
aligned.  Tolerance 1e-6 + 1e-3 |ref|, as test_gpu_score.py (weights from
32-bit logits of exact 16-bit products)."""
import numpy as np
import pytest
import torch

import oracle
from tests.helpers import DTYPE_CODES, allclose_report, rand_rows, to_torch
from wnw_amd import _lib
from wnw_amd.wnw import kernels as wk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,nh,D", [("bfloat16", 4, 128), ("float16", 16, 64), ("float32", 7, 128),
                                        ("float32", 2, 256), ("bfloat16", 9, 256), ("float32", 16, 64)])
@pytest.mark.parametrize("lens", [[23000], [1, 15, 16, 17, 127, 128, 129, 1000, 5, 2050], list(range(30, 730, 10))])
@pytest.mark.parametrize("aligned", [True, False])
def test_against_oracle(gpu, dtype, nh, D, lens, aligned):
    rng = np.random.default_rng(nh + D + len(lens))
    S = len(lens)
    starts = np.concatenate([[3], 3 + np.cumsum(lens)[:-1] + 2 * np.arange(1, S)]).astype(np.int64)
    ends = starts + np.asarray(lens)
    k = rand_rows(rng, int(ends[-1]) + 5, D, dtype)
    q = rand_rows(rng, S * nh, D, dtype).reshape(S, nh, D)
    a_s = np.array([min(9, n // 3) for n in lens], np.int32)
    a_e = np.array([n - n // 7 for n in lens], np.int32)
    offs = np.concatenate([[0], np.cumsum(a_e - a_s)]).astype(np.int32)
    acc0 = rng.random(int(offs[-1])).astype(np.float32)
    ref = oracle.segment_scores(q, k, starts, ends, a_s, a_e, offs[:-1], D ** -0.5, acc0.astype(np.float64),
                                dtype=DTYPE_CODES[dtype])
    tq = to_torch(q, dtype, gpu)
    if not aligned:
        buf = torch.empty(tq.numel() + 1, dtype=tq.dtype, device=gpu)
        buf[1:] = tq.reshape(-1)
        tq = buf[1:].view(S, nh, D)
        assert tq.data_ptr() % 16 and tq.is_contiguous()
    t = lambda a: torch.from_numpy(np.asarray(a, np.int32)).to(gpu)  # noqa: E731
    acc = torch.from_numpy(acc0).to(gpu)
    print(f"group score {dtype} nh={nh} D={D} S={S} aligned={aligned}", flush=True)
    wk.fused_score_accumulate(tq, to_torch(k, dtype, gpu), t(starts), t(ends), t(a_s), t(a_e), acc, t(offs))
    torch.cuda.synchronize()
    assert _lib.device_error() == 0
    ok, msg = allclose_report(acc.cpu().numpy().astype(np.float64), ref, 1e-6, 1e-3)
    assert ok, msg


def _tree_dots(q, k):
    """q . K in 32 bits as chains of 16 bytes of fused multiply-adds, added pairwise."""
    c = 16 // q.element_size()
    qc, kc = (t.double().reshape(t.shape[0], -1, c) for t in (q, k))
    d = torch.zeros(k.shape[0], q.shape[0], qc.shape[1], device=q.device)
    for e in range(c):
        d = (d.double() + kc[:, None, :, e] * qc[None, :, :, e]).float()
    while d.shape[2] > 1:
        d = d[:, :, 0::2] + d[:, :, 1::2]
    return d[:, :, 0]


@pytest.mark.parametrize("dtype,nh,D", [(torch.float32, 4, 64), (torch.float32, 4, 128), (torch.float32, 2, 256),
                                        (torch.bfloat16, 4, 64), (torch.bfloat16, 4, 128), (torch.float16, 4, 128),
                                        (torch.bfloat16, 2, 256)])
def test_no_less_exact_than_short_chains(gpu, dtype, nh, D):
    """Peaked rows (scores of standard deviation 3), where a weight's error is
    that of its dot: the error against 64 bits beside that of dots rounded in
    a tree of short chains with all else in 64 bits.  The two agree up to the
    luck of the few largest weights (0.95 to 1.10 over these 40 items) and the
    exponential's rounding, 6e-8 a weight.  Longer chains, with the scaled dot
    rounded in one of the two passes, are at 1.06 to 1.9."""
    S, n, scale = 40, 1200, D ** -0.5
    g = torch.Generator(device=gpu)
    g.manual_seed(D + nh)
    q = (3 * torch.randn(S, nh, D, device=gpu, generator=g)).to(dtype)
    k = torch.randn(S * n, D, device=gpu, generator=g).to(dtype)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=gpu)  # noqa: E731
    bounds, acc = [i * n for i in range(S + 1)], torch.zeros(S * n, device=gpu)
    wk.fused_score_accumulate(q, k, i32(bounds[:-1]), i32(bounds[1:]), i32([0] * S), i32([n] * S), acc, i32(bounds))
    ours = trees = 0.0
    for i in range(S):
        ki = k[i * n:(i + 1) * n]
        exact = ki.double() @ q[i].double().t() * scale
        w = exact.softmax(0).sum(1)
        tree = (_tree_dots(q[i], ki).double() * scale).softmax(0).sum(1)
        ours += float((acc[i * n:(i + 1) * n].double() - w).norm() / w.norm()) ** 2 / S
        trees += float((tree - w).norm() / w.norm()) ** 2 / S
    print(f"group score error {dtype} nh={nh} D={D}: {ours ** 0.5:.3e}, short chains {trees ** 0.5:.3e}", flush=True)
    assert ours <= 1.2 ** 2 * trees + 1e-14, (ours ** 0.5, trees ** 0.5)
