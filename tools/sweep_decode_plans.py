#!/usr/bin/env python3
"""Pieces per sequence of decode launches: what the constants of the plans were fitted to (pa_partitions_per_piece in
paged_attention_mfma.hip, unified_decode_segments in unified_decode.hip).  Random batches; of each the device time (HIP graphs of 9 calls over
three states) in one piece, in the pieces that the plan would cut it into, and as the plan has it.
usage: python tools/sweep_decode_plans.py [v2|rocm|uni] [seed] [batches]"""
import math, os, random, sys
import torch
sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
from perf import cases
from vllm_amd import _custom_ops as ops, _lib

SHAPES = [(32, 8, 80), (16, 8, 80), (32, 8, 96), (40, 8, 112), (16, 16, 112), (32, 8, 120), (24, 4, 192), (16, 8, 256), (32, 8, 128), (32, 8, 128),
          (8, 1, 128), (8, 1, 128), (64, 8, 128), (32, 32, 128), (32, 8, 64), (32, 8, 64), (12, 12, 64), (16, 1, 64), (4, 1, 128), (20, 4, 128)]
UNI_SHAPES = [s for s in SHAPES if s[2] in (64, 96, 128, 192, 256)]
STATES = 3


def cdiv(a, b):
    return -(-a // b)


def graph_us(fn, calls=9, repeats=5):
    fn(0)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        keep = [fn(j) for j in range(calls)]
    for _ in range(3):
        g.replay()
    torch.cuda.synchronize()
    ts = []
    for _ in range(repeats):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        g.replay()
        g.replay()
        b.record()
        torch.cuda.synchronize()
        ts.append(a.elapsed_time(b) / (2 * calls) * 1e3)
    del keep
    return sorted(ts)[repeats // 2]


def cut_partitions(part, P, base, d):
    """Partitions per piece of pa_partitions_per_piece without its one-piece rules."""
    slots = 256 if d > 128 else 512
    if base < slots:
        sp = max(min(cdiv(base * P, slots), 2048 // part), cdiv(base * P, 4 * slots))
    else:
        sp, best = P, math.inf
        for c in range(P, 0, -1):
            if c * part < 2048:
                break
            cost = cdiv(base * cdiv(P, c), slots) * (c * part + 256)
            if cost < best * 0.97:
                best, sp = cost, c
    return min(max(sp, 1), P)


def cut_segments(L, pairs, row):
    """Segments of unified_decode_segments without its one-piece rule."""
    cap, slots = min(cdiv(L, 256), 16), 256 if row > 128 else 512
    if pairs * cap <= slots:
        return cap
    cost = [cdiv(pairs * n, slots) / n * (1 + n * 160 / L) for n in range(1, cap + 1)]
    return next(n for n in range(1, cap + 1) if cost[n - 1] <= min(cost) * 1.05)


def main():
    kind = sys.argv[1] if len(sys.argv) > 1 else "v2"
    rng = random.Random(int(sys.argv[2]) if len(sys.argv) > 2 else 0)
    n = int(sys.argv[3]) if len(sys.argv) > 3 else 200
    log = lambda a, b: int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))
    part = 512 if kind == "v2" else 256
    print("   heads   D    kv block batch tokens pieces |   one    cut   rule, all alike |   one    cut   rule, from 1/8 on", flush=True)
    for _ in range(n):
        h, kvh, d = rng.choice(UNI_SHAPES if kind == "uni" else SHAPES)
        kv, block = rng.choice(["auto", "fp8"]), rng.choice([16, 16, 32])
        d = 112 if kv == "fp8" and d % 16 else d
        seqs = max(1, round(log(1, 768) / kvh))
        base = seqs * kvh * cdiv(h // kvh, 16)
        L = min(log(part + 1, 9000), (500 << 20) // (2 * kvh * d * (1 if kv == "fp8" else 2)) // seqs)
        P = cdiv(L, part)
        pieces = cut_segments(L, base, d) if kind == "uni" else cdiv(P, cut_partitions(part, P, base, d))
        if L <= part or pieces == 1 or (kind == "uni" and base >= 1024):
            continue
        cells = []
        for ragged in (False, True):
            if ragged and seqs == 1:
                cells.append(" " * 21)
                continue
            c = {"kind": "engine" if kind == "uni" else "decode", "chunks": 0, "new": 0, "cached": 0, "decodes": seqs, "seqs": seqs, "ctx": L,
                 "ragged": ragged, "heads": h, "kv_heads": kvh, "head": d, "block": block, "kv": kv, "dtype": "bf16"}
            states = [cases.prepare(c, k) for k in range(STATES)]

            def call(j):
                s = states[j % STATES]
                if kind == "uni":
                    return cases.run(s)
                out = torch.empty_like(s["q"])
                tmp = torch.empty((seqs, h, P, d), dtype=out.dtype, device="cuda")
                sums = torch.empty((seqs, h, P), dtype=torch.float32, device="cuda")
                args = (out, sums, torch.empty_like(sums), tmp, s["q"], *s["cache"], kvh, d ** -0.5, s["table"], s["lens"])
                if kind == "v2":
                    ops.paged_attention_v2(*args, block, s["max_len"], None, kv, s["scale"], s["scale"])
                else:
                    ops.paged_attention_rocm(*args, None, block, s["max_len"], None, kv, s["scale"], s["scale"])
                return out

            graph_us(call, repeats=3)
            if kind == "uni":
                key, forms = "uni_seg", (1, pieces, 0)
            else:
                key, forms = "pa_sp", (P, cut_partitions(part, P, base, d), 0)
            us = [math.inf] * 3
            for _ in range(2):
                for i, v in enumerate(forms):
                    _lib.set_tuning(key, v)
                    us[i] = min(us[i], graph_us(call))
            _lib.set_tuning(key, 0)
            cells.append("".join(f"{t:7.2f}" for t in us))
            del states
        print(f"{f'{h}/{kvh}':>8} {d:3d} {kv:>5} {block:5d} {seqs:5d} {L:6d} {pieces:6d} |{cells[0]}           |{cells[1]}", flush=True)
        torch.cuda.empty_cache()


if __name__ == "__main__":
    main()
