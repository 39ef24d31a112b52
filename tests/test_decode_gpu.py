"""Calls with at most 16 query rows per head (decode against a key cache), which
one kernel of their own serves, against the fp64 TileMix oracle.

The shapes sit where that kernel can go wrong: the edges of a 32-key step, of a
workgroup's range of steps and of the split over workgroups, every width of
load that d and the alignment allow, one and sixteen rows, routes that change
from cell to cell, skipped cells and heads with no visible key, each quantize
mode, output type and layout; keys and values of more than 128 MiB, which are
read with a non-temporal hint and by four or eight waves; NaN and infinity in Q.
Every head is followed by NaN rows. Bounds are those of the batched sweep: 1e-5 +
1e-4|x| with precise P.V, max-abs 2e-3 and mean-abs 2e-4 with probabilities
rounded to fp16 (plus the rounding of a 16-bit O: at most 2^-8 |x| for bf16, 2^-11
|x| for fp16).
"""
from __future__ import annotations

import numpy as np
import pytest

from helpers import GUARD_DOT, dev, dev_half, host

pytestmark = pytest.mark.gpu

PAD = 64


def _case(heads, M, N, d, g=2, p_skip=0.0, quantize=2, precise=False, out="f32", layout="hsd", aligned=True,
          scale=1.0, routed=True):
    return dict(heads=heads, M=M, N=N, d=d, g=g, p_skip=p_skip, quantize=quantize, precise=precise, out=out,
                layout=layout, aligned=aligned, scale=scale, routed=routed)


CASES = [
    _case(2, 1, 1, 128), _case(1, 16, 31, 64, precise=True), _case(3, 4, 32, 128, g=1), _case(2, 5, 33, 72, g=1),
    _case(2, 16, 255, 128, g=1, p_skip=0.3), _case(2, 3, 256, 64, precise=True), _case(5, 7, 257, 80, quantize=1),
    _case(1, 16, 513, 128, precise=True, quantize=0), _case(2, 4, 1000, 100, g=3, p_skip=0.25),
    _case(3, 2, 777, 40, precise=True, quantize=0), _case(1, 9, 1003, 7, g=1, quantize=0),
    _case(2, 16, 1500, 121, quantize=1, precise=True), _case(2, 8, 2048, 120, quantize=0, p_skip=0.5, g=1),
    _case(1, 4, 9000, 128, p_skip=0.3, precise=True), _case(4, 1, 4097, 128, out="bf16", layout="shd"),
    _case(3, 6, 3000, 64, out="f16", layout="shd", quantize=1), _case(2, 4, 1200, 96, aligned=False),
    _case(2, 4, 1200, 72, aligned=False, out="bf16"), _case(2, 3, 700, 128, scale=-1.0, p_skip=0.2),
    _case(2, 3, 700, 64, scale=0.0, precise=True), _case(2, 16, 2000, 128, routed=False, precise=True),
    _case(2, 1, 5000, 33, routed=False), _case(300, 2, 600, 32, p_skip=0.3), _case(600, 1, 300, 64),
    _case(1, 16, 33000, 128, g=5, p_skip=0.1), _case(2, 4, 900, 128, p_skip=1.0),
]


def _id(c):
    return "-".join(f"{k}{v}" for k, v in c.items())


def _codes(rng, N, g, p_skip, routed):
    tiles = (N + 31) // 32
    if not routed:
        return np.zeros((1, tiles), np.uint8)
    u = rng.random((1, (tiles + g - 1) // g))
    codes = np.where(u < p_skip, 2, np.where(u < p_skip + 0.5 * (1 - p_skip), 1, 0)).astype(np.uint8)
    return np.repeat(codes, g, axis=1)[:, :tiles].copy()


def _half_rows(rng, oracle_lib, heads, rows, d):
    return [oracle_lib.float_to_half(rng.standard_normal((rows, d)).astype(np.float32)) for _ in range(heads)]


def _padded(parts, rows, layout):
    """NaN-padded heads as a device tensor viewed [heads, rows + PAD, d]."""
    out = np.full((len(parts), rows + PAD, parts[0].shape[1]), 0x7E00, dtype=np.uint16)
    for h, part in enumerate(parts):
        out[h, :rows] = part
    if layout == "hsd":
        return dev_half(out)
    return dev_half(np.ascontiguousarray(out.transpose(1, 0, 2))).transpose(0, 1)


def _problem(oracle_lib, c):
    rng = np.random.default_rng(c["M"] * 7919 + c["N"] * 31 + c["d"])
    p = dict(q=_half_rows(rng, oracle_lib, c["heads"], c["M"], c["d"]),
             k=_half_rows(rng, oracle_lib, c["heads"], c["N"], c["d"]),
             v=_half_rows(rng, oracle_lib, c["heads"], c["N"], c["d"]))
    p["codes"] = [_codes(rng, c["N"], c["g"], c["p_skip"], c["routed"]) for _ in range(c["heads"])]
    return p


def _device(tm, c, p):
    """(BatchedArgs, everything they point to)."""
    import torch

    from tilemix import routing

    heads, M, N, d = c["heads"], c["M"], c["N"], c["d"]
    Q, K, V = (_padded(p[n], r, c["layout"]) for n, r in (("q", M), ("k", N), ("v", N)))
    b = dict(Q=Q, K=K, V=V, Q8=torch.full((heads, M, d), 99, dtype=torch.int8, device="cuda:0"),
             K8=torch.full((heads, N, d), 99, dtype=torch.int8, device="cuda:0"),
             qs=torch.empty((heads, 1), dtype=torch.int16, device="cuda:0"),
             ks=torch.empty((heads, (N + 63) // 64), dtype=torch.int16, device="cuda:0"))
    o_type = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[c["out"]]
    lead = 16 if c["aligned"] else 1
    flat = torch.full((lead + heads * (M + 1) * d,), 96.0, dtype=o_type, device="cuda:0")
    O = flat[lead:].view(heads, M + 1, d) if c["layout"] == "hsd" else flat[lead:].view(M + 1, heads, d).transpose(0, 1)
    b.update(flat=flat, O=O, trace=torch.full((heads, (N + 31) // 32), 9, dtype=torch.uint8, device="cuda:0"),
             dots=torch.full((heads, M, N), int(GUARD_DOT), dtype=torch.int32, device="cuda:0"))
    options = dict(quantize=0)
    if c["routed"]:
        packed = [routing.pack_cells(x, c["g"]) for x in p["codes"]]
        empty = np.zeros(routing.word_count(M, N, c["g"]), np.uint64)
        b["route"] = dev(np.concatenate([r for r, _ in packed]))
        b["skip"] = dev(np.concatenate([empty if s is None else s for _, s in packed])) if c["p_skip"] else None
        if c["quantize"] != 1:
            both = c["quantize"] == 0
            tm.check(tm.quantize_tilemix_qk_strided(
                Q if both else None, K, b["Q8"] if both else None, b["K8"], b["qs"] if both else None, b["ks"], heads,
                M, N, d, Q.stride(0), K.stride(0), Q.stride(1), K.stride(1)))
        options = dict(quantize=c["quantize"], route_words=b["route"], skip_words=b["skip"], Q8=b["Q8"], K8=b["K8"],
                       q_scales=b["qs"], k_scales=b["ks"])
    args = tm.BatchedArgs(
        Q=Q, K=K, V=V, O=O, heads=heads, M=M, N=N, d=d, score_scale=c["scale"] / np.sqrt(d), precise=c["precise"],
        key_tiles_per_group=c["g"], o_dtype={"f32": 0, "f16": 1, "bf16": 2}[c["out"]],
        q_head_stride=Q.stride(0), k_head_stride=K.stride(0), v_head_stride=V.stride(0), o_head_stride=O.stride(0),
        q_row_stride=Q.stride(1), k_row_stride=K.stride(1), v_row_stride=V.stride(1), o_row_stride=O.stride(1),
        **options)
    return args, b


def _check(oracle_lib, c, p, b):
    heads, M, d = c["heads"], c["M"], c["d"]
    out = b["O"].float().cpu().numpy()
    assert (out[:, M:] == 96.0).all(), "rows past M written"
    assert (b["flat"][:16 if c["aligned"] else 1].float() == 96.0).all()
    for h in sorted({0, 1, heads // 2, heads - 1} & set(range(heads))):
        q8, qs = oracle_lib.quantize(p["q"][h], 128)
        k8, ks = oracle_lib.quantize(p["k"][h], 64)
        if c["routed"]:
            assert np.array_equal(b["Q8"][h].cpu().numpy(), q8) and np.array_equal(b["K8"][h].cpu().numpy(), k8)
            assert np.array_equal(b["qs"][h].cpu().numpy().view(np.uint16), qs)
        scale = float(np.float32(c["scale"] / np.sqrt(d)))
        want = oracle_lib.tilemix(p["q"][h], p["k"][h], p["v"][h], q8, k8, qs, ks, p["codes"][h], scale)
        got = out[h, :M].astype(np.float64)
        assert np.isfinite(got).all()
        rounding = {"f32": 0.0, "f16": 2.0 ** -11, "bf16": 2.0 ** -8}[c["out"]] * np.abs(want)
        err = np.maximum(np.abs(got - want) - rounding, 0.0)
        if c["precise"]:
            assert (err <= 1e-5 + 1e-4 * np.abs(want)).all(), (h, float(err.max()))
        else:
            assert err.max() <= 2e-3 and err.mean() <= 2e-4, (h, float(err.max()), float(err.mean()))


@pytest.mark.parametrize("case", CASES, ids=[_id(c) for c in CASES])
def test_decode_vs_oracle(tm, oracle_lib, cuda, case):
    import torch

    p = _problem(oracle_lib, case)
    args, b = _device(tm, case, p)
    torch.cuda.synchronize()
    print(f"decode {_id(case)}", flush=True)
    tm.check(tm.attention_batched(args))
    torch.cuda.synchronize()
    _check(oracle_lib, case, p, b)
    # With the verification outputs: the same O, the route of every cell, the dots of INT8 cells.
    first = b["flat"].clone()
    args.decoded_bits, args.score_dots = b["trace"], b["dots"] if case["routed"] else None
    tm.check(tm.attention_batched(args))
    torch.cuda.synchronize()
    assert torch.equal(first.view(torch.uint8), b["flat"].view(torch.uint8))
    codes = np.concatenate(p["codes"])
    assert np.array_equal(host(b["trace"]), codes)
    if case["routed"]:
        h = case["heads"] - 1
        cells = np.repeat(codes[h], 32)[:case["N"]] == 1
        q8, k8 = (b[n][h].cpu().numpy().astype(np.int64) for n in ("Q8", "K8"))
        assert np.array_equal(host(b["dots"])[h], np.where(cells[None, :], q8 @ k8.T, int(GUARD_DOT)))


def test_decode_calls_share_the_workspace_in_turn(tm, oracle_lib, cuda):
    """Split calls on two streams with nothing between them, and per-head split calls among them."""
    import torch

    cases = [_case(4, 4, 5000, 128, p_skip=0.2), _case(2, 16, 9000, 64, precise=True), _case(8, 1, 3000, 72)]
    made = []
    for c in cases:
        p = _problem(oracle_lib, c)
        made.append((c, p) + _device(tm, c, p))
    q, k, v = (dev_half(x) for x in oracle_lib.make_inputs(1000, 2000, 128, "random"))
    outs = [torch.empty((1000, 128), device="cuda:0") for _ in range(7)]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    print("decode and per-head calls on two streams", flush=True)
    for i in range(6):
        tm.check(tm.attention_batched(made[i % 3][2], streams[i % 2]))
        tm.check(tm.launch_fused_fp16_attention(q, k, v, outs[i], 1000, 2000, 128, 0.1, streams[(i // 2) % 2]))
    torch.cuda.synchronize()
    for c, p, _, b in made:
        _check(oracle_lib, c, p, b)
    tm.check(tm.launch_fused_fp16_attention(q, k, v, outs[6], 1000, 2000, 128, 0.1))
    torch.cuda.synchronize()
    for o in outs[:6]:
        assert np.array_equal(host(o), host(outs[6]))


def test_decode_under_graph_capture(tm, oracle_lib, cuda):
    import torch

    c = _case(4, 4, 5000, 128, p_skip=0.2)
    p = _problem(oracle_lib, c)
    args, b = _device(tm, c, p)
    graph = torch.cuda.CUDAGraph()
    print("decode under graph capture", flush=True)
    with torch.cuda.graph(graph):
        tm.check(tm.attention_batched(args, torch.cuda.current_stream()))
    for _ in range(3):
        b["flat"].fill_(96.0)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        _check(oracle_lib, c, p, b)
        tm.check(tm.attention_batched(args))  # eager, split, between the replays
        torch.cuda.synchronize()
        _check(oracle_lib, c, p, b)


# heads, M, N, d, routed, precise, out: more than 128 MiB of keys and values. From the top: four waves with the
# hint (64 steps a workgroup), eight with it (47), four at d <= 64, precise, 8-byte K8 rows, and rows in dword pieces.
LARGE = [
    (32, 4, 16384, 128, True, False, "f32"), (100, 4, 3000, 128, True, False, "bf16"), (64, 2, 9000, 64, True, False, "f32"),
    (40, 3, 11000, 112, True, True, "f32"), (32, 16, 17000, 72, False, False, "f32"), (32, 2, 16500, 100, True, False, "f32"),
    (256, 1, 1100, 128, False, True, "f32"), (520, 4, 700, 102, True, False, "f32"), (520, 4, 700, 128, True, False, "f32"),
]


@pytest.mark.parametrize("case", LARGE, ids=["-".join(map(str, c)) for c in LARGE])
def test_decode_large(tm, oracle_lib, cuda, case):
    import torch

    from tilemix import routing

    heads, M, N, d, routed, precise, out = case
    assert heads * N * d * 4 > 128 << 20
    gen = torch.Generator(device="cuda")
    gen.manual_seed(heads + N)
    Q, K, V = (torch.randn(heads, r, d, generator=gen, device="cuda", dtype=torch.float16) for r in (M, N, N))
    O = torch.full((heads, M, d), 96.0, dtype=torch.bfloat16 if out == "bf16" else torch.float32, device="cuda")
    codes = [_codes(np.random.default_rng(h), N, 2, 0.2, routed) for h in range(heads)]
    options = dict(quantize=0)
    if routed:
        packed = [routing.pack_cells(x, 2) for x in codes]
        empty = np.zeros(routing.word_count(M, N, 2), np.uint64)
        K8 = torch.empty((heads, N, d), dtype=torch.int8, device="cuda")
        ks = torch.empty((heads, (N + 63) // 64), dtype=torch.int16, device="cuda")
        options = dict(quantize=1, route_words=dev(np.concatenate([r for r, _ in packed])),
                       skip_words=dev(np.concatenate([empty if s is None else s for _, s in packed])), K8=K8,
                       k_scales=ks)
    print(f"large decode {case}", flush=True)
    tm.check(tm.attention_batched(tm.BatchedArgs(
        Q=Q, K=K, V=V, O=O, heads=heads, M=M, N=N, d=d, score_scale=d ** -0.5, precise=precise, key_tiles_per_group=2,
        o_dtype=2 if out == "bf16" else 0, **options)))
    torch.cuda.synchronize()
    got = O.float().cpu().numpy().astype(np.float64)
    assert np.isfinite(got).all()
    for h in (0, heads // 2, heads - 1):
        q, k, v = (host(x[h]) for x in (Q, K, V))
        q8, q_s = oracle_lib.quantize(q, 128)
        k8, k_s = oracle_lib.quantize(k, 64)
        want = oracle_lib.tilemix(q, k, v, q8, k8, q_s, k_s, codes[h], float(np.float32(d ** -0.5)))
        err = np.maximum(np.abs(got[h] - want) - (2.0 ** -8 * np.abs(want) if out == "bf16" else 0.0), 0.0)
        if precise:
            assert (err <= 1e-5 + 1e-4 * np.abs(want)).all(), (h, float(err.max()))
        else:
            assert err.max() <= 2e-3 and err.mean() <= 2e-4, (h, float(err.max()), float(err.mean()))


@pytest.mark.parametrize("heads,M,N,d", [(3, 16, 700, 128), (2, 5, 3000, 64), (2, 9, 513, 72), (2, 16, 900, 100),
                                         (3, 4, 1200, 33)])
def test_decode_special_values_in_q(tm, oracle_lib, cuda, heads, M, N, d):
    """Q quantized in the kernel, with a NaN in every head's block, the last of all NaN, the first also with the
    largest fp16 value: Q8 and the scales are the quantizer's, and rows without a NaN are the oracle's."""
    import torch

    from tilemix import routing

    rng = np.random.default_rng(N + d)
    q, k, v = (oracle_lib.float_to_half(rng.standard_normal((heads, r, d)).astype(np.float32)) for r in (M, N, N))
    for h in range(heads):
        q[h, (3 * h + 1) % M, (7 * h) % d] = 0x7E00 if h % 2 else 0xFE00
    q[0, 0, d - 1] = 0xFBFF
    q[heads - 1] = 0x7E00
    codes = [_codes(rng, N, 1, 0.0, True) for _ in range(heads)]
    route = dev(np.concatenate([routing.pack_cells(x, 1)[0] for x in codes]))
    Q, K, V = (dev_half(x) for x in (q, k, v))
    outs = dict(Q8=torch.full((heads, M, d), 99, dtype=torch.int8, device="cuda"),
                K8=torch.full((heads, N, d), 99, dtype=torch.int8, device="cuda"),
                q_scales=torch.full((heads, 1), 99, dtype=torch.int16, device="cuda"),
                k_scales=torch.full((heads, (N + 63) // 64), 99, dtype=torch.int16, device="cuda"))
    wanted = {n: torch.empty_like(t) for n, t in outs.items()}
    tm.check(tm.quantize_tilemix_qk_batched(Q, K, *wanted.values(), heads, M, N, d))
    O = torch.full((heads, M, d), 96.0, device="cuda")
    print(f"decode, NaN in Q: {heads} x {M} x {N} x {d}", flush=True)
    tm.check(tm.attention_batched(tm.BatchedArgs(Q=Q, K=K, V=V, O=O, heads=heads, M=M, N=N, d=d, score_scale=d ** -0.5,
                                                 precise=True, key_tiles_per_group=1, quantize=1, route_words=route,
                                                 **outs)))
    torch.cuda.synchronize()
    for n in outs:
        assert torch.equal(outs[n], wanted[n]), n
    got = O.cpu().numpy()
    for h in range(heads):
        q8, q_s = oracle_lib.quantize(q[h], 128)
        k8, k_s = oracle_lib.quantize(k[h], 64)
        assert np.array_equal(host(outs["Q8"])[h], q8) and np.array_equal(host(outs["q_scales"])[h].view(np.uint16), q_s)
        bad = ((q[h] & 0x7FFF) > 0x7C00).any(axis=1)
        assert np.isnan(got[h][bad]).all() and np.isfinite(got[h][~bad]).all()
        with np.errstate(invalid="ignore"):
            want = oracle_lib.tilemix(q[h], k[h], v[h], q8, k8, q_s, k_s, codes[h], float(np.float32(d ** -0.5)))
        assert (np.abs(got[h] - want)[~bad] <= (1e-5 + 1e-4 * np.abs(want))[~bad]).all()
