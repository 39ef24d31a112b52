"""Calls whose key range is split over workgroups, captured in a HIP graph: a
captured call leaves the library's workspace alone and takes the same ranges of
keys in turn, so every replay equals the eager call to the bit, in every output.

Batched splits (ragged, causal, routed with skipped cells, precise, every load
width, 16-bit outputs, more ranges than one batch of the merge), split decode
(four and eight waves, every load width, heads without a visible key; the
per-head call of 16 rows among them); the eager call runs again between the
replays, and a repeated eager call gives the same bits too.
"""
from __future__ import annotations

import numpy as np
import pytest

from helpers import dev

pytestmark = pytest.mark.gpu

# heads, M, N, d, causal, precise, p_skip (None: dense), out, layout, per_head
CASES = {
    "chunk": (8, 512, 8192, 128, False, False, None, "bf16", "shd", False),
    "chunk-routed": (4, 500, 5000, 128, False, False, 0.3, "f32", "hsd", False),
    "causal": (2, 1100, 1100, 128, True, False, 0.0, "f32", "hsd", False),
    "causal-d64-skip": (3, 1030, 1030, 64, True, True, 0.4, "f32", "shd", False),
    "precise-d72": (12, 1003, 1003, 72, True, True, None, "f32", "hsd", False),
    "d100": (2, 300, 2000, 100, False, False, 0.2, "f16", "hsd", False),
    "d33": (2, 70, 1290, 33, False, True, 0.2, "f32", "hsd", False),
    "d32-many-ranges": (1, 128, 8192, 32, False, False, 0.2, "f32", "hsd", False),
    "all-skipped": (2, 64, 3000, 128, False, False, 1.0, "f32", "hsd", False),
    "decode": (4, 4, 5000, 128, False, False, 0.2, "f32", "hsd", False),
    "decode-d64": (3, 16, 9000, 64, False, True, None, "bf16", "shd", False),
    "decode-d72": (8, 1, 3000, 72, False, False, 0.5, "f32", "hsd", False),
    "decode-d100": (2, 7, 3000, 100, False, True, 0.0, "f32", "hsd", False),
    "decode-d121": (2, 3, 2500, 121, False, False, None, "f32", "hsd", False),
    "decode-four-waves": (16, 4, 33000, 128, False, False, 0.0, "f32", "hsd", False),
    "per-head-decode": (1, 16, 2500, 128, False, True, 0.0, "f32", "hsd", True),
    "precise-d48": (1, 777, 3001, 48, False, True, None, "f32", "hsd", False),
}


def _problem(name):
    import torch

    from tilemix import routing

    heads, M, N, d, causal, precise, p_skip, out, layout, per_head = CASES[name]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(M + N + d)

    def laid_out(x):
        return x if layout == "hsd" else x.transpose(0, 1).contiguous().transpose(0, 1)

    Q, K, V = (laid_out(torch.randn(heads, r, d, generator=gen, device="cuda").half()) for r in (M, N, N))
    route = skip = None
    if p_skip is not None:
        rng = np.random.default_rng(M + N)
        u = rng.random((heads, (M + 15) // 16, ((N + 31) // 32 + 1) // 2)).repeat(2, axis=2)[:, :, :(N + 31) // 32]
        codes = np.where(u < p_skip, 2, np.where(u < p_skip + (1 - p_skip) / 2, 1, 0)).astype(np.uint8)
        packed = [routing.pack_cells(x, 2) for x in codes]
        empty = np.zeros(routing.word_count(M, N, 2), np.uint64)
        route = dev(np.concatenate([r for r, _ in packed]))
        skip = dev(np.concatenate([empty if s is None else s for _, s in packed])) if p_skip else None
    return Q, K, V, route, skip, laid_out


@pytest.mark.parametrize("name", list(CASES))
def test_captured_split_call_equals_eager(tm, cuda, name):
    import torch

    heads, M, N, d, causal, precise, p_skip, out, layout, per_head = CASES[name]
    Q, K, V, route, skip, laid_out = _problem(name)
    o_dtype, o_type = {"f32": (0, torch.float32), "f16": (1, torch.float16), "bf16": (2, torch.bfloat16)}[out]

    def buffers():
        return dict(O=laid_out(torch.empty((heads, M, d), dtype=o_type, device="cuda")),
                    Q8=torch.empty((heads, M, d), dtype=torch.int8, device="cuda"),
                    K8=torch.empty((heads, N, d), dtype=torch.int8, device="cuda"),
                    qs=torch.empty((heads, (M + 127) // 128), dtype=torch.int16, device="cuda"),
                    ks=torch.empty((heads, (N + 63) // 64), dtype=torch.int16, device="cuda"))

    def step(b):
        if per_head:
            options = (None, None)
            if route is not None:
                tm.check(tm.quantize_tilemix_qk(Q, K, b["Q8"], b["K8"], b["qs"], b["ks"], M, N, d))
                options = (tm.TileMixRouting(route, route.numel(), 2),
                           tm.TileMixQuantized(b["Q8"], b["K8"], b["qs"], b["ks"]))
            tm.check(tm.launch_fused_fp16_attention(Q, K, V, b["O"], M, N, d, d ** -0.5, None, *options))
            return
        options = dict(quantize=0)
        if route is not None:
            options = dict(quantize=1, route_words=route, skip_words=skip, Q8=b["Q8"], K8=b["K8"], q_scales=b["qs"],
                           k_scales=b["ks"])
        O = b["O"]
        tm.check(tm.attention_batched(tm.BatchedArgs(
            Q=Q, K=K, V=V, O=O, heads=heads, M=M, N=N, d=d, score_scale=d ** -0.5, causal=causal, precise=precise,
            key_tiles_per_group=2, o_dtype=o_dtype, q_head_stride=Q.stride(0), k_head_stride=K.stride(0),
            v_head_stride=V.stride(0), o_head_stride=O.stride(0), q_row_stride=Q.stride(1), k_row_stride=K.stride(1),
            v_row_stride=V.stride(1), o_row_stride=O.stride(1), **options)))

    def cleared(b):
        for t in b.values():
            t.fill_(float("nan") if t.is_floating_point() else 99)
        torch.cuda.synchronize()

    def same(a, b, what):
        for n in a if route is not None else ("O",):
            x, y = (t[n].contiguous().view(torch.uint8) for t in (a, b))
            assert torch.equal(x, y), f"{what}: {n} differs"

    print(f"graph bits {name}: eager", flush=True)
    eager, again, captured = buffers(), buffers(), buffers()
    for b in (eager, again, captured):
        cleared(b)
        step(b)
    torch.cuda.synchronize()
    same(eager, again, "eager call repeated")
    graph = torch.cuda.CUDAGraph()
    print(f"graph bits {name}: capture", flush=True)
    with torch.cuda.graph(graph):
        step(captured)
    for replay in range(3):
        cleared(captured)
        graph.replay()
        cleared(again)
        step(again)
        torch.cuda.synchronize()
        same(eager, captured, f"replay {replay}")
        same(eager, again, f"eager call after replay {replay}")


@pytest.mark.parametrize("name", ["chunk-routed", "causal-d64-skip", "d100", "decode", "decode-d72"])
def test_captured_verification_outputs(tm, cuda, name):
    """The routing trace and the int32 dots of a captured split call, and O beside them."""
    import torch

    heads, M, N, d, causal, precise = CASES[name][:6]
    Q, K, V, route, skip, laid_out = _problem(name)
    Q8, K8 = (torch.empty((heads, rows, d), dtype=torch.int8, device="cuda") for rows in (M, N))
    qs, ks = (torch.empty((heads, -(-rows // b)), dtype=torch.int16, device="cuda") for rows, b in ((M, 128), (N, 64)))
    O = laid_out(torch.empty((heads, M, d), device="cuda"))
    trace = torch.empty((heads, (M + 15) // 16, (N + 31) // 32), dtype=torch.uint8, device="cuda")
    dots = torch.empty((heads, M, N), dtype=torch.int32, device="cuda")
    args = tm.BatchedArgs(
        Q=Q, K=K, V=V, O=O, heads=heads, M=M, N=N, d=d, score_scale=d ** -0.5, causal=causal, precise=precise, quantize=1,
        route_words=route, skip_words=skip, key_tiles_per_group=2, Q8=Q8, K8=K8, q_scales=qs, k_scales=ks,
        decoded_bits=trace, score_dots=dots, q_head_stride=Q.stride(0), k_head_stride=K.stride(0),
        v_head_stride=V.stride(0), o_head_stride=O.stride(0), q_row_stride=Q.stride(1), k_row_stride=K.stride(1),
        v_row_stride=V.stride(1), o_row_stride=O.stride(1))

    def cleared():
        for t in (O, trace, dots):
            t.fill_(77)
        torch.cuda.synchronize()

    print(f"graph bits {name}: verification outputs", flush=True)
    cleared()
    tm.check(tm.attention_batched(args))
    torch.cuda.synchronize()
    eager = [t.clone() for t in (O, trace, dots)]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        tm.check(tm.attention_batched(args))
    for replay in range(2):
        cleared()
        graph.replay()
        torch.cuda.synchronize()
        for what, a, b in zip(("O", "trace", "dots"), eager, (O, trace, dots)):
            assert torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8)), f"{what}, replay {replay}"
