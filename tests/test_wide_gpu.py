"""Large launches, which the 256-row kernel takes when there are whole rounds of
long walks. A call that asks for the routing trace always takes the 128-row
kernel, so each call is made both ways: O must agree to the bit, and with the
fp64 TileMix oracle (2e-3 / 2e-4) on sampled rows.

Shapes: whole and ragged tiles, an odd number of 128-row blocks, more tiles than
one window of the route table and an odd number of visited ones, causal
diagonals through both halves of a block, cells that mix routes inside a wave,
skipped tiles, heads and rows without a visible key, a negative score scale,
16-bit outputs, [S, H, D] layouts, reversed rounds of row blocks, and a NaN in
one of a block's two Q quantization blocks. Q8 and the scales are cleared before
each call, and each call's are checked, on all heads against the other call's
and on sampled heads against the oracle's.
"""
from __future__ import annotations

import numpy as np
import pytest

from helpers import dev, host

pytestmark = pytest.mark.gpu

# name: heads, M, N, d, g, causal, p_skip, cell rows x key groups per drawn code, out, layout, scale sign
CASES = {
    "d128": (32, 2048, 2048, 128, 2, False, 0.0, 4, "f32", "hsd", 1),
    "d64-cells-skip": (64, 1000, 2049, 64, 1, False, 0.3, 1, "f32", "hsd", 1),
    "causal-cells": (64, 2048, 2048, 128, 3, True, 0.1, 1, "f32", "hsd", 1),
    "causal-d64-ragged": (64, 4095, 4095, 64, 2, True, 0.0, 4, "f32", "shd", 1),
    "causal-d112-skip": (64, 2047, 2047, 112, 2, True, 0.2, 4, "f32", "shd", 1),
    "odd-blocks-d112": (128, 300, 2100, 112, 2, False, 0.3, 4, "f32", "hsd", 1),
    "windows-odd-count": (64, 1024, 4100, 128, 2, False, 0.0, 8, "bf16", "hsd", 1),
    "negative-scale": (32, 2048, 2300, 128, 2, False, 0.0, 4, "f16", "shd", -1),
    "dense": (32, 2048, 2048, 48, 1, False, None, 1, "f32", "hsd", 1),
    "reversed-rounds": (16, 16384, 2048, 64, 2, False, 0.4, 4, "f32", "hsd", 1),
    "short-keys-causal": (64, 4096, 2048, 128, 2, True, 0.0, 8, "f32", "hsd", 1),
}


@pytest.mark.parametrize("name", list(CASES))
def test_wide_equals_128_row_kernel_and_oracle(tm, oracle_lib, cuda, name):
    import torch

    from tilemix import routing

    heads, M, N, d, g, causal, p_skip, rows, out, layout, sign = CASES[name]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(M + N + d)
    Q, K, V = (torch.randn(heads, r, d, generator=gen, device="cuda").half() for r in (M, N, N))
    options = dict(quantize=0)
    codes = np.zeros((heads, (M + 15) // 16, (N + 31) // 32), np.uint8)
    if p_skip is not None:
        rng = np.random.default_rng(M + N)
        q_tiles, groups = codes.shape[1], (codes.shape[2] + g - 1) // g
        u = rng.random((heads, (q_tiles + rows - 1) // rows, groups))
        u = np.repeat(np.repeat(u, rows, axis=1)[:, :q_tiles], g, axis=2)[:, :, :codes.shape[2]]
        codes = np.where(u < p_skip, 2, np.where(u < p_skip + (1 - p_skip) / 2, 1, 0)).astype(np.uint8)
        if p_skip > 0:
            codes[1] = 2  # a head without a visible key
            codes[2, 3:9] = 2  # rows without one
        packed = [routing.pack_cells(x, g) for x in codes]
        empty = np.zeros(routing.word_count(M, N, g), np.uint64)
        Q8 = torch.empty((heads, M, d), dtype=torch.int8, device="cuda")
        K8 = torch.empty((heads, N, d), dtype=torch.int8, device="cuda")
        qs = torch.empty((heads, (M + 127) // 128), dtype=torch.int16, device="cuda")
        ks = torch.empty((heads, (N + 63) // 64), dtype=torch.int16, device="cuda")
        if name == "d128":
            Q[0, 5, 7] = float("nan")  # the first Q block of head 0's first 256 rows
        options = dict(quantize=1, route_words=dev(np.concatenate([r for r, _ in packed])),
                       skip_words=dev(np.concatenate([empty if s is None else s for _, s in packed])) if p_skip else None,
                       Q8=Q8, K8=K8, q_scales=qs, k_scales=ks)

    def laid_out(x):
        return x if layout == "hsd" else x.transpose(0, 1).contiguous().transpose(0, 1)

    Q, K, V = laid_out(Q), laid_out(K), laid_out(V)
    scale = float(np.float32(sign / np.sqrt(d)))
    o_type = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[out]
    outs, quantized = [], []
    for traced in (False, True):
        if p_skip is not None:
            for t in (Q8, K8, qs, ks):
                t.fill_(99)
        O = laid_out(torch.full((heads, M, d), 96.0, dtype=o_type, device="cuda"))
        trace = torch.empty(codes.shape, dtype=torch.uint8, device="cuda")
        args = tm.BatchedArgs(
            Q=Q, K=K, V=V, O=O, heads=heads, M=M, N=N, d=d, score_scale=scale, causal=causal, key_tiles_per_group=g,
            o_dtype={"f32": 0, "f16": 1, "bf16": 2}[out], decoded_bits=trace if traced else None,
            q_head_stride=Q.stride(0), k_head_stride=K.stride(0), v_head_stride=V.stride(0), o_head_stride=O.stride(0),
            q_row_stride=Q.stride(1), k_row_stride=K.stride(1), v_row_stride=V.stride(1), o_row_stride=O.stride(1),
            **options)
        print(f"wide {name} traced={traced}", flush=True)
        tm.check(tm.attention_batched(args))
        torch.cuda.synchronize()
        outs.append(O.clone())
        if p_skip is not None:
            quantized.append([t.clone() for t in (Q8, K8, qs, ks)])
    assert torch.equal(outs[0].contiguous().view(torch.uint8), outs[1].contiguous().view(torch.uint8))
    assert np.array_equal(host(trace), codes)
    for wide, narrow in zip(*quantized):
        assert torch.equal(wide, narrow)
    got = outs[0].float().cpu().numpy()
    rng = np.random.default_rng(1)
    for h in (0, 2, heads - 1):
        q, k, v = (x[h].contiguous().cpu().view(torch.int16).numpy().view(np.uint16) for x in (Q, K, V))
        q8, q_s = oracle_lib.quantize(q, 128)
        k8, k_s = oracle_lib.quantize(k, 64)
        if p_skip is not None:
            wide_q8, wide_k8, wide_qs, wide_ks = (host(t)[h] for t in quantized[0])
            assert np.array_equal(wide_q8, q8) and np.array_equal(wide_qs.view(np.uint16), q_s)
            assert np.array_equal(wide_k8, k8) and np.array_equal(wide_ks.view(np.uint16), k_s)
        sample = np.unique(np.concatenate([rng.choice(M, 200), np.arange(16), np.arange(M - 16, M)])).astype(np.int32)
        if h == 0 and name == "d128":
            sample = sample[sample != 5]  # the row with the NaN
        want = oracle_lib.tilemix(q, k, v, q8, k8, q_s, k_s, codes[h], scale, causal, rows=sample)
        rounding = {"f32": 0.0, "f16": 2.0 ** -11, "bf16": 2.0 ** -8}[out] * np.abs(want)
        err = np.maximum(np.abs(got[h, sample].astype(np.float64) - want) - rounding, 0.0)
        assert err.max() <= 2e-3 and err.mean() <= 2e-4, (h, float(err.max()), float(err.mean()))
    if p_skip:
        assert not got[1].any(), "a head without a visible key is zero"
