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
