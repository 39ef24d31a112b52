"""NaN and infinity through calls whose key range is split over workgroups: the
per-head call, the batched split (causal too) and the decode kernel, whose
partial rows are merged afterwards.

A query row with a NaN has NaN scores for every FP16 key, so its maximum over
them stays -inf: such a part must make the row NaN, as it does unsplit, and not
count as one that saw no key. An infinite value reaches the rows that weigh its
key, also from the last split, whose partial rows a short batch of the merge
reads more than once. Other rows equal the fp64 result (1e-5 + 1e-4|x| precise,
2e-3 with probabilities rounded to fp16).
"""
from __future__ import annotations

import numpy as np
import pytest

from helpers import dev, dev_half

pytestmark = pytest.mark.gpu

# heads, M, N, d, causal, precise, routed: first half of the keys INT8, the others FP16; per_head entry point
CASES = {
    "per-head": (1, 300, 2000, 128, False, True, False, True),
    "per-head-routed": (1, 200, 2048, 64, False, True, True, True),
    "per-head-decode": (1, 16, 3000, 128, False, True, False, True),
    "batched": (2, 300, 2000, 128, False, False, False, False),
    "batched-routed": (2, 300, 2048, 128, False, False, True, False),
    "batched-causal": (2, 1100, 1100, 128, True, False, False, False),
    "batched-precise-d72": (2, 200, 1500, 72, False, True, True, False),
    "decode": (2, 4, 5000, 128, False, False, False, False),
    "decode-routed": (3, 16, 4096, 64, False, False, True, False),
    "decode-precise-d100": (2, 7, 3000, 100, False, True, True, False),
}


def _words(tm, M, N, heads, routed):
    from tilemix import routing

    if not routed:
        return None
    codes = np.zeros(((M + 15) // 16, (N + 31) // 32), np.uint8)
    codes[:, :N // 64] = 1
    return dev(np.concatenate([routing.pack_cells(codes, 1)[0]] * heads))


def _call(tm, case, q, k, v):
    import torch

    heads, M, N, d, causal, precise, routed, per_head = case
    Q, K, V = (dev_half(x) for x in (q, k, v))
    O = torch.full((heads, M, d), 96.0, device="cuda:0")
    route = _words(tm, M, N, heads, routed)
    Q8, K8 = (torch.empty((heads, rows, d), dtype=torch.int8, device="cuda:0") for rows in (M, N))
    qs, ks = (torch.empty((heads, -(-rows // b)), dtype=torch.int16, device="cuda:0") for rows, b in ((M, 128), (N, 64)))
    tm.check(tm.quantize_tilemix_qk_batched(Q, K, Q8, K8, qs, ks, heads, M, N, d))
    scale = float(np.float32(d ** -0.5))
    if per_head:
        options = (None, None)
        if routed:
            options = (tm.TileMixRouting(route, route.numel(), 1), tm.TileMixQuantized(Q8, K8, qs, ks))
        tm.check(tm.launch_fused_fp16_attention(Q, K, V, O, M, N, d, scale, None, *options))
    else:
        options = dict(quantize=0, route_words=route, Q8=Q8, K8=K8, q_scales=qs, k_scales=ks) if routed else dict(quantize=0)
        tm.check(tm.attention_batched(tm.BatchedArgs(Q=Q, K=K, V=V, O=O, heads=heads, M=M, N=N, d=d, score_scale=scale,
                                                     causal=causal, precise=precise, key_tiles_per_group=1, **options)))
    torch.cuda.synchronize()
    return O.cpu().numpy()


def _inputs(oracle_lib, case):
    heads, M, N, d = case[:4]
    rng = np.random.default_rng(M + N + d)
    return [oracle_lib.float_to_half(rng.standard_normal((heads, r, d)).astype(np.float32)) for r in (M, N, N)]


@pytest.mark.parametrize("name", list(CASES))
def test_nan_query_row(tm, oracle_lib, cuda, name):
    heads, M, N, d, causal, precise, routed, _ = case = CASES[name]
    q, k, v = _inputs(oracle_lib, case)
    print(f"split, NaN in a query row: {name}", flush=True)
    clean = _call(tm, case, q, k, v)
    head, row = heads - 1, M - 2
    q[head, row, d // 2] = 0x7E00
    out = _call(tm, case, q, k, v)
    assert np.isnan(out[head, row]).all(), f"{np.isnan(out[head, row]).sum()} of {d} values are NaN"
    rest = np.ones((heads, M), bool)
    rest[head, row] = False
    assert np.isfinite(out[rest]).all()
    for h in range(heads):
        q8, q_s = oracle_lib.quantize(q[h], 128)
        k8, k_s = oracle_lib.quantize(k[h], 64)
        codes = np.zeros(((M + 15) // 16, (N + 31) // 32), np.uint8)
        if routed:
            codes[:, :N // 64] = 1
        with np.errstate(invalid="ignore"):
            want = oracle_lib.tilemix(q[h], k[h], v[h], q8, k8, q_s, k_s, codes, float(np.float32(d ** -0.5)), causal)
        err = np.abs(out[h] - want)[rest[h]]
        bound = (1e-5 + 1e-4 * np.abs(want) if precise else np.full_like(want, 2e-3))[rest[h]]
        assert (err <= bound).all(), (h, float(err.max()))
    if not routed:  # the NaN changes no other row
        assert np.array_equal(out[rest].view(np.uint32), clean[rest].view(np.uint32))


@pytest.mark.parametrize("name", ["batched", "batched-causal", "decode"])
def test_infinite_value_of_the_last_key(tm, oracle_lib, cuda, name):
    """The last key scores 0 for every row, so every row that sees it weighs it."""
    heads, M, N, d, causal = CASES[name][:5]
    q, k, v = _inputs(oracle_lib, CASES[name])
    k[:, -1] = 0
    v[:, -1, 3] = 0x7C00
    print(f"split, infinite value: {name}", flush=True)
    out = _call(tm, CASES[name], q, k, v)
    sees = np.arange(M) >= (N - 1 if causal else 0)
    assert (out[:, sees, 3] == np.inf).all()
    assert np.isfinite(np.delete(out, 3, axis=2)).all()
    if causal:  # 0 * inf inside the diagonal tile only
        assert np.isfinite(out[:, :N - N % 64, 3]).all()
