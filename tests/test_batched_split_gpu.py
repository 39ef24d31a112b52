"""Batched calls of few, long row blocks, whose key range is split over several
workgroups per 128-row block and merged by a second kernel: ragged shapes with
and without a causal mask, ranges past the diagonal, skipped cells and rows
without a visible key, both P.V forms, every load width, output types and
layouts, against the fp64 TileMix oracle (2e-3 / 2e-4 for the fast P.V,
1e-5 + 1e-4|x| for the precise one), and the call with verification outputs
against the one without, to the bit (Q8, K8 and the scales, cleared before each
call, too).
"""
from __future__ import annotations

import numpy as np
import pytest

from helpers import compare, dev, dev_half, host

pytestmark = pytest.mark.gpu

# heads, M, N, d, g, causal, precise, p_skip, out, layout
CASES = [
    (2, 300, 2000, 128, 1, False, False, 0.2, "f32", "hsd"), (2, 1100, 1100, 128, 2, True, False, 0.0, "f32", "hsd"),
    (3, 1030, 1030, 64, 1, True, True, 0.3, "f32", "shd"), (2, 1200, 1500, 96, 2, True, False, 0.0, "f32", "hsd"),
    (2, 1500, 1200, 32, 1, True, True, 0.2, "f32", "hsd"), (2, 130, 1024, 72, 1, False, True, 0.2, "f32", "hsd"),
    (1, 1025, 1025, 100, 2, True, False, 0.1, "f32", "hsd"), (2, 70, 1290, 33, 1, False, True, 0.2, "f32", "hsd"),
    (4, 257, 4099, 128, 2, False, False, 0.0, "bf16", "shd"), (5, 200, 1600, 64, 2, False, False, 0.0, "f16", "shd"),
    (1, 2600, 2600, 128, 2, True, True, 0.9, "f32", "hsd"), (2, 64, 3000, 128, 2, False, False, 1.0, "f32", "hsd"),
]


@pytest.mark.parametrize("case", CASES, ids=["-".join(map(str, c)) for c in CASES])
def test_batched_split_vs_oracle(tm, oracle_lib, cuda, case):
    import torch

    from tilemix import routing

    heads, M, N, d, g, causal, precise, p_skip, out, layout = case
    rng = np.random.default_rng(M + 3 * N + d)
    q, k, v = (oracle_lib.float_to_half(rng.standard_normal((heads, r, d)).astype(np.float32)) for r in (M, N, N))
    groups = ((N + 31) // 32 + g - 1) // g
    u = rng.random((heads, (M + 15) // 16, groups))
    codes = np.where(u < p_skip, 2, np.where(u < p_skip + (1 - p_skip) / 2, 1, 0)).astype(np.uint8)
    codes = np.ascontiguousarray(np.repeat(codes, g, axis=2)[:, :, :(N + 31) // 32])
    packed = [routing.pack_cells(x, g) for x in codes]
    empty = np.zeros(routing.word_count(M, N, g), np.uint64)
    route = dev(np.concatenate([r for r, _ in packed]))
    skip = dev(np.concatenate([empty if s is None else s for _, s in packed]))

    def laid_out(x):
        return x if layout == "hsd" else x.transpose(0, 1).contiguous().transpose(0, 1)

    Q, K, V = (laid_out(dev_half(x)) for x in (q, k, v))
    o_type = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[out]
    Q8 = torch.empty((heads, M, d), dtype=torch.int8, device="cuda:0")
    K8 = torch.empty((heads, N, d), dtype=torch.int8, device="cuda:0")
    qs = torch.empty((heads, (M + 127) // 128), dtype=torch.int16, device="cuda:0")
    ks = torch.empty((heads, (N + 63) // 64), dtype=torch.int16, device="cuda:0")
    outs = []
    for traced in (False, True):
        for t in (Q8, K8, qs, ks):
            t.fill_(99)
        O = laid_out(torch.full((heads, M, d), 96.0, dtype=o_type, device="cuda:0"))
        trace = torch.full(codes.shape, 9, dtype=torch.uint8, device="cuda:0")
        args = tm.BatchedArgs(
            Q=Q, K=K, V=V, O=O, heads=heads, M=M, N=N, d=d, score_scale=d ** -0.5, causal=causal, precise=precise,
            quantize=1, route_words=route, skip_words=skip, key_tiles_per_group=g, Q8=Q8, K8=K8, q_scales=qs,
            k_scales=ks, o_dtype={"f32": 0, "f16": 1, "bf16": 2}[out], decoded_bits=trace if traced else None,
            q_head_stride=Q.stride(0), k_head_stride=K.stride(0), v_head_stride=V.stride(0), o_head_stride=O.stride(0),
            q_row_stride=Q.stride(1), k_row_stride=K.stride(1), v_row_stride=V.stride(1), o_row_stride=O.stride(1))
        print(f"batched split {case} traced={traced}", flush=True)
        tm.check(tm.attention_batched(args))
        torch.cuda.synchronize()
        outs.append(O.float().cpu().numpy())
        if traced:
            assert np.array_equal(host(trace), codes)
        for h in range(heads):
            q8, q_s = oracle_lib.quantize(q[h], 128)
            k8, k_s = oracle_lib.quantize(k[h], 64)
            assert np.array_equal(host(Q8)[h], q8) and np.array_equal(host(K8)[h], k8)
            assert np.array_equal(host(qs)[h].view(np.uint16), q_s)
            assert np.array_equal(host(ks)[h].view(np.uint16), k_s)
    assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))
    for h in range(heads):
        q8, q_s = oracle_lib.quantize(q[h], 128)
        k8, k_s = oracle_lib.quantize(k[h], 64)
        want = oracle_lib.tilemix(q[h], k[h], v[h], q8, k8, q_s, k_s, codes[h], float(np.float32(d ** -0.5)), causal)
        got = outs[0][h]
        if precise:
            compare(got, want, 1e-5, 1e-4, f"head {h}")
        else:
            rounding = {"f32": 0.0, "f16": 2.0 ** -11, "bf16": 2.0 ** -8}[out] * np.abs(want)
            err = np.maximum(np.abs(got.astype(np.float64) - want) - rounding, 0.0)
            assert err.max() <= 2e-3 and err.mean() <= 2e-4, (h, float(err.max()), float(err.mean()))
