"""GPU parity: unified_attention (flash-layout cache, causal, window / softcap / ALiBi / fp8)
vs the CPU oracle's restatement of the Triton kernel.  Shapes and tolerance follow the
reference's tests/kernels/attention/test_triton_unified_attention.py:80-200 (atol 1.5e-2,
rtol 1e-2 on N(0,1) data), head sizes 128 (tile / decode kernels) and 256 (wide-head kernel)."""
import pytest
import torch

from helpers import make_unified_case

pytestmark = pytest.mark.gpu

ATOL, RTOL = 1.5e-2, 1e-2


def run(orc, c, dtype, window=None, softcap=0.0, alibi=None, out_scale=None, fp8=False, view=None):
    from vllm_amd.attention.ops import unified_attention
    ws = (window - 1, 0) if window is not None else (-1, -1)
    D = c["q"].shape[2]
    sm = D ** -0.5
    odt = torch.uint8 if out_scale is not None else dtype
    ref = torch.zeros(c["q"].shape, dtype=odt)
    kd = c["scale"] if fp8 else None
    orc.unified_attention(c["q"], c["k"], c["v"], ref, c["cu_seqlens_q"], c["max_seqlen_q"],
                          c["seqused_k"], c["max_seqlen_k"], sm, True, ws, c["block_table"],
                          softcap, None, kd, kd, alibi, out_scale)
    kc, vc = c["k"].cuda(), c["v"].cuda()
    if view is not None:
        kc, vc = view(kc), view(vc)
    out = torch.zeros(c["q"].shape, dtype=odt, device="cuda")
    unified_attention(c["q"].cuda(), kc, vc, out, c["cu_seqlens_q"].cuda(), c["max_seqlen_q"],
                      c["seqused_k"].cuda(), c["max_seqlen_k"], sm, True, ws,
                      c["block_table"].cuda(), softcap, None,
                      None if kd is None else kd.cuda(), None if kd is None else kd.cuda(),
                      None if alibi is None else alibi.cuda(),
                      None if out_scale is None else out_scale.cuda())
    if out_scale is not None:
        a = out.cpu().view(torch.float8_e4m3fn).float() * float(out_scale)
        b = ref.view(torch.float8_e4m3fn).float() * float(out_scale)
        torch.testing.assert_close(a, b, atol=8e-3 + ATOL, rtol=0.13)
    else:
        torch.testing.assert_close(out.cpu().float(), ref.float(), atol=ATOL, rtol=RTOL)


@pytest.mark.parametrize("seq_lens", [[(1, 1328), (5, 18), (129, 463)], [(1, 523), (1, 37), (1, 2011)]])
@pytest.mark.parametrize("num_heads", [(4, 4), (8, 2), (16, 2)])
@pytest.mark.parametrize("block_size", [16, 32])
@pytest.mark.parametrize("sliding_window", [None, 256])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("soft_cap", [None, 10.0, 50.0])
@pytest.mark.parametrize("head_size", [128, 256])
def test_unified_reference_grid(oracle, seq_lens, num_heads, block_size, sliding_window, dtype, soft_cap, head_size):
    """The reference test's grid (HEAD_SIZES = [128, 256])."""
    c = make_unified_case(seq_lens, num_heads[0], num_heads[1], head_size, block_size, dtype,
                          seed=len(seq_lens) + num_heads[0] + block_size)
    run(oracle, c, dtype, window=sliding_window, softcap=soft_cap or 0.0)


@pytest.mark.parametrize("D", [160, 192, 224, 256])
@pytest.mark.parametrize("mode", ["plain", "fp8", "alibi", "fp8_out"])
@pytest.mark.parametrize("kernel", ["tile", "valu"])
def test_unified_wide_heads(oracle, D, mode, kernel):
    """Head sizes 160 .. 256 of TritonAttentionBackend.get_supported_head_sizes (triton_attn.py:147-148):
    the tile kernel's 256-wide instantiation (default) and the plain VALU kernel ("pf_rows" = 2), mixed batch,
    fp8 cache / ALiBi / fp8 output."""
    from vllm_amd import _lib
    _lib.set_tuning("pf_rows", 2 if kernel == "valu" else 0)
    try:
        _wide_heads(oracle, D, mode)
    finally:
        _lib.set_tuning("pf_rows", 0)


def _wide_heads(oracle, D, mode):
    fp8 = mode in ("fp8", "fp8_out")
    c = make_unified_case([(90, 400), (1, 700), (17, 17), (1, 1), (3, 260)], 8, 2, D, 16, torch.bfloat16,
                          fp8=fp8, seed=D, kv_scale=0.5)
    slopes = 2.0 ** -(torch.arange(8).float() * 0.5 + 1) if mode == "alibi" else None
    run(oracle, c, torch.bfloat16, fp8=fp8, alibi=slopes, window=300 if mode == "alibi" else None,
        out_scale=torch.tensor([0.03]) if mode == "fp8_out" else None)


@pytest.mark.parametrize("seq_lens", [[(700, 700), (300, 1500), (64, 64), (1, 1)], [(257, 1000), (130, 131)]])
@pytest.mark.parametrize("D", [128, 64])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("window", [None, 100])
def test_unified_long_prefill(oracle, seq_lens, D, dtype, window):
    """Several row blocks per sequence: interior, diagonal and skipped tiles, pure prefill
    (ctx 0) and chunked prefill, window narrower than a row block."""
    c = make_unified_case(seq_lens, 8, 2, D, 16, dtype, seed=D + len(seq_lens))
    run(oracle, c, dtype, window=window)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("block_size", [16, 32])
@pytest.mark.parametrize("D", [128, 64])
@pytest.mark.parametrize("soft_cap", [None, 30.0])
def test_unified_fp8_cache(oracle, dtype, block_size, D, soft_cap):
    c = make_unified_case([(200, 900), (1, 77), (33, 33)], 8, 2, D, block_size, dtype, fp8=True,
                          seed=block_size + D, kv_scale=0.75)
    run(oracle, c, dtype, softcap=soft_cap or 0.0, fp8=True)


@pytest.mark.parametrize("block_size", [64, 128])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("seq_lens", [[(1, 1328), (5, 18), (129, 463), (64, 64)], [(1, 523), (1, 37), (1, 2011), (1, 128)],
                                      [(1, 70)] * 10 + [(40, 300), (1, 129), (1, 1)] * 3])
def test_unified_large_blocks(oracle, block_size, fp8, seq_lens):
    """Pages of 64 / 128 tokens (the block size is a run-time power of two in both kernels): mixed,
    decode-only (split) and >= 16-sequence batches (decode kernel + tile kernel)."""
    c = make_unified_case(seq_lens, 8, 2, 128, block_size, torch.bfloat16, fp8=fp8, seed=block_size + len(seq_lens),
                          kv_scale=0.5)
    run(oracle, c, torch.bfloat16, fp8=fp8)
    run(oracle, c, torch.bfloat16, fp8=fp8, window=100, softcap=25.0)


@pytest.mark.parametrize("D", [32, 80, 96, 120, 128])
def test_unified_head_sizes(oracle, D):
    c = make_unified_case([(90, 400), (17, 17)], 4, 2, D, 16, torch.bfloat16, seed=D)
    run(oracle, c, torch.bfloat16)


@pytest.mark.parametrize("window", [None, 64])
def test_unified_alibi(oracle, window):
    c = make_unified_case([(150, 600), (1, 300), (40, 41)], 8, 4, 128, 16, torch.float16, seed=5)
    slopes = 2.0 ** -(torch.arange(8).float() * 0.5 + 1)
    run(oracle, c, torch.float16, alibi=slopes, window=window)


@pytest.mark.parametrize("heads", [(8, 2), (32, 8), (16, 1), (6, 2)])
@pytest.mark.parametrize("D", [128, 64])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("mode", ["plain", "window", "alibi", "softcap"])
def test_unified_decode_batches(oracle, heads, D, fp8, mode):
    """Decode-only batches (every query length 1): the decode kernel and the GQA-packed tile
    launch (tile rows = the q heads of a kv head's group).  Lengths around the 64-key tile and
    the page size."""
    c = make_unified_case([(1, 1), (1, 64), (1, 65), (1, 300), (1, 17), (1, 1000)], heads[0], heads[1],
                          D, 16, torch.bfloat16, fp8=fp8, seed=heads[0] + D, kv_scale=0.5)
    slopes = 2.0 ** -(torch.arange(heads[0]).float() * 0.25 + 1) if mode == "alibi" else None
    from vllm_amd import _lib
    try:
        for knob in (1, 0):   # the decode kernel, then the packed tile kernel
            _lib.set_tuning("uni_decode", knob)
            run(oracle, c, torch.bfloat16, fp8=fp8, alibi=slopes, window=48 if mode == "window" else None,
                softcap=20.0 if mode == "softcap" else 0.0)
    finally:
        _lib.set_tuning("uni_decode", 1)


@pytest.mark.parametrize("heads", [(8, 2), (32, 8), (6, 2), (14, 2), (16, 1)])
@pytest.mark.parametrize("D", [128, 64])
@pytest.mark.parametrize("mode", ["plain", "window", "alibi"])
def test_unified_mixed_batch_packed(oracle, heads, D, mode):
    """Prefill chunks and decode tokens in one call, GQA groups that do and do not divide the
    tile's 64 / 128 rows (6, 7): rows are (token, head) pairs, blocks of 64 // group tokens."""
    c = make_unified_case([(1, 500), (70, 70), (1, 64), (33, 200), (9, 9), (150, 1100), (1, 1)],
                          heads[0], heads[1], D, 16, torch.float16, seed=heads[0] * 3 + D)
    slopes = 2.0 ** -(torch.arange(heads[0]).float() * 0.25 + 1) if mode == "alibi" else None
    run(oracle, c, torch.float16, alibi=slopes, window=40 if mode == "window" else None)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("block_size", [16, 32])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("nseq", [3, 140, 260])
def test_unified_decode_kernel(oracle, dtype, block_size, fp8, nseq):
    """The flash-layout decode kernel (unified_decode.hip): split over key segments (3 and 140
    sequences: 12 and 560 workgroups) and unsplit with the XCD-grouped order (260: 1040), both
    block sizes and dtypes, lengths around the step (32 / 64 tokens), the page and the
    64-token segment tile."""
    lens = [1, 31, 32, 33, 63, 64, 65, 127, 128, 129, 255, 257, 700, 1, 16, 17]
    seqs = [(1, lens[i % len(lens)] + (i // len(lens))) for i in range(nseq)]
    if nseq == 3:
        seqs = [(1, 2500), (1, 64), (1, 1023)]
    c = make_unified_case(seqs, 8, 4, 128, block_size, dtype, fp8=fp8, seed=nseq + block_size, kv_scale=0.5)
    run(oracle, c, dtype, fp8=fp8)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("D,nseq", [(64, 3), (128, 3), (128, 40), (256, 3), (256, 40)])
@pytest.mark.parametrize("segs", [1, 2, 3, 16])
def test_unified_decode_segments(oracle, fp8, D, nseq, segs):
    """Every batch in one piece and cut, whichever of them the heuristic takes: more segments than a sequence has tiles, lengths
    around the edges of a segment, one key."""
    from vllm_amd import _lib
    lens = [900, 1, 64, 65, 128, 129, 192, 383, 385, 577]
    c = make_unified_case([(1, lens[i % len(lens)]) for i in range(nseq)], 8, 4, D, 16, torch.bfloat16, fp8=fp8, seed=nseq + segs, kv_scale=0.5)
    _lib.set_tuning("uni_seg", segs)
    try:
        run(oracle, c, torch.bfloat16, fp8=fp8)
    finally:
        _lib.set_tuning("uni_seg", 0)


@pytest.mark.parametrize("D", [32, 48, 80, 96, 112, 120, 136, 160, 192, 224, 256])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("nseq", [5, 260])
def test_unified_decode_head_sizes(oracle, D, fp8, nseq):
    """Head sizes below the kernel's padded 64 / 128 / 256 (whole 16-byte K chunks): split and unsplit
    launches, and a mixed batch of >= 16 sequences."""
    if fp8 and D % 16:
        pytest.skip("an fp8 cache needs head sizes that are multiples of 16")
    lens = [1, 31, 64, 65, 129, 300, 700]
    seqs = [(1, lens[i % len(lens)] + i // 7) for i in range(nseq)]
    c = make_unified_case(seqs, 8, 4, D, 16, torch.bfloat16, fp8=fp8, seed=D + nseq, kv_scale=0.5)
    run(oracle, c, torch.bfloat16, fp8=fp8)
    if nseq == 5:
        c = make_unified_case(seqs * 4 + [(37, 120)], 8, 4, D, 16, torch.bfloat16, fp8=fp8, seed=D, kv_scale=0.5)
        run(oracle, c, torch.bfloat16, fp8=fp8, window=90)


@pytest.mark.parametrize("D_heads", [(128, (8, 4)), (64, (16, 8)), (64, (8, 4)), (32, (8, 8)), (128, (16, 2)), (64, (32, 4))])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("hp", [1, 2, 4])
@pytest.mark.parametrize("mode", ["plain", "alibi", "window", "fp8_out"])
@pytest.mark.parametrize("nseq", [5, 150])
def test_unified_decode_packed_kv_heads(oracle, D_heads, fp8, hp, mode, nseq):
    """Token-major caches: "uni_hp" adjacent kv heads are taken as one row of the decode kernel (their q heads are the
    columns of one Q^T operand, zero outside the own head's d range; 1 = never, 2 / 4 = that many where the shape allows,
    else fewer) -- split (5 sequences) and unsplit launches, every per-column feature, against the oracle."""
    from vllm_amd import _lib
    D, (H, KVH) = D_heads
    lens = [3, 64, 65, 300, 1000]
    seqs = [(1, lens[i % 5] + i // 5) for i in range(nseq)]
    c = make_unified_case(seqs, H, KVH, D, 16, torch.bfloat16, fp8=fp8, seed=D + H + nseq, kv_scale=0.5)
    slopes = 2.0 ** -(torch.arange(H).float() * 0.25 + 1) if mode == "alibi" else None
    _lib.set_tuning("uni_hp", hp)
    try:
        run(oracle, c, torch.bfloat16, fp8=fp8, alibi=slopes, window=90 if mode == "window" else None,
            out_scale=torch.tensor([0.02]) if mode == "fp8_out" else None)
    finally:
        _lib.set_tuning("uni_hp", 0)


@pytest.mark.parametrize("heads", [(32, 1), (48, 2), (20, 1), (17, 1)])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("nseq", [4, 600])
def test_unified_decode_wide_groups(oracle, heads, fp8, nseq):
    """GQA groups of more than 16 q heads (MQA): 16 heads per workgroup, the last chunk partial;
    split and unsplit launches, ALiBi per head."""
    lens = [1, 33, 64, 130, 500]
    seqs = [(1, lens[i % len(lens)] + i // 5) for i in range(nseq)]
    c = make_unified_case(seqs, heads[0], heads[1], 64, 16, torch.float16, fp8=fp8, seed=heads[0] + nseq, kv_scale=0.5)
    slopes = 2.0 ** -(torch.arange(heads[0]).float() * 0.125 + 1)
    run(oracle, c, torch.float16, fp8=fp8, alibi=slopes)


@pytest.mark.parametrize("mode", ["window", "alibi", "softcap", "fp8_out", "hnd"])
@pytest.mark.parametrize("fp8", [False, True])
def test_unified_decode_kernel_features(oracle, mode, fp8):
    """Window edges inside / across steps and segments, ALiBi, softcap, fp8 output and a
    head-major (HND) cache allocation; unsplit launch (1040 workgroups; the split launches of
    these features are in test_unified_decode_batches)."""
    lens = [5, 100, 129, 300, 640, 1000]
    seqs = [(1, lens[i % len(lens)] + i // 6) for i in range(260)]
    c = make_unified_case(seqs, 8, 4, 64 if mode == "alibi" else 128, 16, torch.bfloat16, fp8=fp8, seed=77,
                          kv_scale=0.5)
    slopes = 2.0 ** -(torch.arange(8).float() * 0.25 + 1) if mode == "alibi" else None
    view = (lambda t: t.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3)) if mode == "hnd" else None
    run(oracle, c, torch.bfloat16, fp8=fp8, alibi=slopes, window=100 if mode == "window" else None,
        softcap=15.0 if mode == "softcap" else 0.0,
        out_scale=torch.tensor([0.02]) if mode == "fp8_out" else None, view=view)


@pytest.mark.parametrize("mode", ["window", "alibi", "softcap", "fp8_out", "hnd", "f16", "mqa"])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("nseq", [6, 300])
def test_unified_decode_kernel_wide_heads(oracle, mode, fp8, nseq):
    """The decode kernel's 256-wide instantiation (head sizes 136 .. 256: one workgroup per CU, the 16 q heads
    written in two passes): split (6 sequences) and unsplit launches, every feature, groups of 16 and 20 q heads."""
    lens = [5, 100, 129, 300, 640, 1000]
    seqs = [(1, lens[i % len(lens)] + i // 6) for i in range(nseq)]
    dtype = torch.float16 if mode == "f16" else torch.bfloat16
    H, KVH = (20, 1) if mode == "mqa" else (16, 2) if mode == "hnd" else (8, 4)
    c = make_unified_case(seqs, H, KVH, 192 if mode == "alibi" else 256, 16, dtype, fp8=fp8, seed=78 + nseq, kv_scale=0.5)
    slopes = 2.0 ** -(torch.arange(H).float() * 0.25 + 1) if mode == "alibi" else None
    view = (lambda t: t.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3)) if mode == "hnd" else None
    run(oracle, c, dtype, fp8=fp8, alibi=slopes, window=100 if mode == "window" else None,
        softcap=15.0 if mode == "softcap" else 0.0,
        out_scale=torch.tensor([0.02]) if mode == "fp8_out" else None, view=view)


@pytest.mark.parametrize("heads", [(8, 2), (32, 8), (4, 4), (24, 1)])
@pytest.mark.parametrize("D", [128, 64])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("mode", ["plain", "window", "alibi", "softcap"])
def test_unified_mixed_batch_two_kernels(oracle, heads, D, fp8, mode):
    """Mixed batches of >= 16 sequences: the decode kernel takes the sequences of query length
    1 (also a one-token prefill chunk), the tile kernel the rest."""
    seqs = [(1, 500), (70, 70), (1, 64), (33, 200), (1, 1), (9, 9), (1, 129), (150, 1100), (1, 31),
            (1, 1000), (2, 2), (1, 333), (1, 65), (17, 80), (1, 256), (1, 255), (1, 77), (5, 600)]
    c = make_unified_case(seqs, heads[0], heads[1], D, 16, torch.bfloat16, fp8=fp8, seed=heads[0] + D,
                          kv_scale=0.5)
    slopes = 2.0 ** -(torch.arange(heads[0]).float() * 0.25 + 1) if mode == "alibi" else None
    run(oracle, c, torch.bfloat16, fp8=fp8, alibi=slopes, window=40 if mode == "window" else None,
        softcap=20.0 if mode == "softcap" else 0.0)


def test_unified_decode_kernel_equals_packed(oracle):
    """Same decode batch through the decode kernel and the packed tile kernel ("uni_decode" = 0)."""
    from vllm_amd import _lib
    from vllm_amd.attention.ops import unified_attention
    c = make_unified_case([(1, 700), (1, 33), (1, 4000)], 16, 4, 128, 16, torch.bfloat16, fp8=True, seed=4,
                          kv_scale=0.5)
    outs = []
    sc = c["scale"].cuda()
    for knob in (1, 0):
        _lib.set_tuning("uni_decode", knob)
        out = torch.zeros(c["q"].shape, dtype=torch.bfloat16, device="cuda")
        unified_attention(c["q"].cuda(), c["k"].cuda(), c["v"].cuda(), out, c["cu_seqlens_q"].cuda(), 1,
                          c["seqused_k"].cuda(), 4000, 128 ** -0.5, True, (-1, -1),
                          c["block_table"].cuda(), 0.0, None, sc, sc)
        outs.append(out.cpu())
    _lib.set_tuning("uni_decode", 1)
    torch.testing.assert_close(outs[0].float(), outs[1].float(), atol=4e-3, rtol=4e-3)


def test_unified_decode_packed_equals_unpacked(oracle):
    """Same decode batch through the packed and the per-head launch ("pf_rows" = 1)."""
    from vllm_amd import _lib
    from vllm_amd.attention.ops import unified_attention
    c = make_unified_case([(1, 700), (1, 33)], 16, 4, 128, 32, torch.float16, seed=4)
    outs = []
    for knob in (0, 1):
        _lib.set_tuning("pf_rows", knob)
        out = torch.zeros(c["q"].shape, dtype=torch.float16, device="cuda")
        unified_attention(c["q"].cuda(), c["k"].cuda(), c["v"].cuda(), out, c["cu_seqlens_q"].cuda(), 1,
                          c["seqused_k"].cuda(), 700, 128 ** -0.5, True, (-1, -1),
                          c["block_table"].cuda(), 0.0, None, None, None)
        outs.append(out.cpu())
    _lib.set_tuning("pf_rows", 0)
    torch.testing.assert_close(outs[0].float(), outs[1].float(), atol=2e-3, rtol=2e-3)


def test_unified_fp8_output(oracle):
    c = make_unified_case([(130, 500), (1, 90)], 8, 2, 128, 16, torch.bfloat16, fp8=True, seed=9,
                          kv_scale=0.5)
    run(oracle, c, torch.bfloat16, fp8=True, out_scale=torch.tensor([0.02]))


def test_unified_strided_cache(oracle):
    """Caches as permuted views of an HND allocation (strides, not shapes, address the cache)."""
    c = make_unified_case([(70, 300), (3, 50)], 4, 2, 128, 16, torch.bfloat16, seed=11)
    view = lambda t: t.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3)
    run(oracle, c, torch.bfloat16, view=view)


def test_unified_rejects_what_it_does_not_cover():
    from vllm_amd.attention.ops import unified_attention
    c = make_unified_case([(4, 40)], 4, 4, 264, 16, torch.bfloat16)
    out = torch.zeros(c["q"].shape, dtype=torch.bfloat16, device="cuda")
    with pytest.raises(RuntimeError, match="unsupported head size"):
        unified_attention(c["q"].cuda(), c["k"].cuda(), c["v"].cuda(), out, c["cu_seqlens_q"].cuda(),
                          4, c["seqused_k"].cuda(), 40, 0.1, True, (-1, -1), c["block_table"].cuda(),
                          0, None, None, None)


@pytest.mark.parametrize("fp8", [False, True])
def test_unified_mixed_batch_with_caller_segments_c_abi(oracle, fp8):
    """C-ABI level (include/vllm_amd.h): a mixed batch of >= 16 sequences with query lengths
    1..4 whose caller passes num_segments = 16 scratch.  The decode tokens are written by the
    decode kernel; the segment merge of the tile path must leave them alone (their segm_* rows
    are never written: poisoned with NaN here)."""
    from vllm_amd import _lib
    from vllm_amd._lib import check, lib
    from vllm_amd._torch_ops import _ptr, _stream
    dtype, H, KVH, D, BS = torch.bfloat16, 8, 2, 128, 16
    seq_lens = [(1 + (i % 4) if i % 3 else 1, 40 + 97 * i) for i in range(20)]
    c = make_unified_case(seq_lens, H, KVH, D, BS, dtype, fp8=fp8, seed=5, kv_scale=0.05 if fp8 else 1.0)
    sm = D ** -0.5
    kd = c["scale"] if fp8 else None
    ref = torch.zeros(c["q"].shape, dtype=dtype)
    oracle.unified_attention(c["q"], c["k"], c["v"], ref, c["cu_seqlens_q"], c["max_seqlen_q"],
                             c["seqused_k"], c["max_seqlen_k"], sm, True, (-1, -1), c["block_table"],
                             0.0, None, kd, kd, None, None)
    q, k, v = c["q"].cuda(), c["k"].cuda(), c["v"].cuda()
    cu, sk, bt = c["cu_seqlens_q"].cuda(), c["seqused_k"].cuda(), c["block_table"].cuda()
    kdd = None if kd is None else kd.cuda()
    out = torch.zeros_like(q)
    nseg = 16
    T = q.shape[0]
    segm_out = torch.full((T, H, nseg, D), float("nan"), dtype=torch.float32, device="cuda")
    segm_max = torch.full((T, H, nseg), float("nan"), dtype=torch.float32, device="cuda")
    segm_sum = torch.full((T, H, nseg), float("nan"), dtype=torch.float32, device="cuda")
    check(lib.vllm_amd_unified_attention(
        _ptr(out), _ptr(q), _ptr(k), _ptr(v), _ptr(cu), _ptr(sk), _ptr(bt), _ptr(kdd), _ptr(kdd),
        None, None, len(seq_lens), H, KVH, D, BS, c["max_seqlen_q"], bt.stride(0), q.stride(0),
        q.stride(1), out.stride(0), out.stride(1), k.stride(0), k.stride(1), k.stride(2),
        v.stride(0), v.stride(1), v.stride(2), float(sm), 0, 0.0, T, c["max_seqlen_k"],
        _ptr(segm_out), _ptr(segm_max), _ptr(segm_sum), nseg, _lib.BF16,
        _lib.KV_FP8_E4M3 if fp8 else _lib.KV_AUTO, _stream(q)))
    torch.cuda.synchronize()
    assert not out.isnan().any()
    torch.testing.assert_close(out.cpu().float(), ref.float(), atol=ATOL, rtol=RTOL)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("shape", [(64, 16, 8), (200, 4, 2), (256, 8, 8)])   # the last: XCD-grouped
def test_unified_decode_longest_first_order(oracle, fp8, shape):
    """Unsplit decode launches of 257..1024 workgroups hand the sequences out longest first
    (pa_lpt_wg, common.cuh): the output equals the oracle's and is bit-identical to the hardware
    order ("pa_order" = 0), with ties among the lengths and a mixed batch (non-decode sequences
    leave their workgroups at once)."""
    from vllm_amd import _lib
    from vllm_amd.attention.ops import unified_attention
    S, H, KVH = shape
    g = torch.Generator().manual_seed(S)
    kvl = torch.randint(1, 400, (S,), generator=g).tolist()
    kvl[2] = kvl[11] = kvl[S - 1] = 123
    for mixed in (False, True):
        sl = [(1, n) for n in kvl]
        if mixed:
            sl[4] = (3, kvl[4] + 3)
            sl[20] = (40, 40)
        c = make_unified_case(sl, H, KVH, 128, 16, torch.bfloat16, fp8=fp8, seed=S + mixed, kv_scale=0.5)
        run(oracle, c, torch.bfloat16, fp8=fp8)
        if not mixed:
            run(oracle, c, torch.bfloat16, fp8=fp8, window=100)   # keys clamp at the window
        kd = c["scale"].cuda() if fp8 else None
        outs = []
        for order in (1, 0):
            _lib.set_tuning("pa_order", order)
            out = torch.zeros(c["q"].shape, dtype=torch.bfloat16, device="cuda")
            unified_attention(c["q"].cuda(), c["k"].cuda(), c["v"].cuda(), out, c["cu_seqlens_q"].cuda(),
                              c["max_seqlen_q"], c["seqused_k"].cuda(), c["max_seqlen_k"], 128 ** -0.5,
                              True, (-1, -1), c["block_table"].cuda(), 0.0, None, kd, kd)
            outs.append(out)
        _lib.set_tuning("pa_order", 1)
        torch.cuda.synchronize()
        assert torch.equal(outs[0], outs[1])


@pytest.fixture
def force_fa():
    """The 256-row kernel (prefill_fa.hip) for every launch that it supports ("pf_fa" = 2), not only long chunks."""
    from vllm_amd import _lib
    _lib.set_tuning("pf_fa", 2)
    yield
    _lib.set_tuning("pf_fa", 0)


@pytest.mark.parametrize("heads", [(8, 2), (32, 8), (4, 4), (6, 2), (14, 2), (16, 1), (24, 1)])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("seq_lens", [[(700, 700), (300, 1500), (64, 64), (1, 1)],
                                      [(257, 1000), (130, 131), (1, 900), (5, 18), (63, 64), (65, 65)]])
def test_unified_fa_kernel(oracle, force_fa, heads, fp8, dtype, seq_lens):
    """The 256-row kernel on every GQA packing (groups that divide 256 rows, 3 and 7 that do not, 24 = unpacked
    rows): pure and chunked prefill, row blocks with one valid row, interior / diagonal / skipped tiles, stale NaN
    slots behind the sequences, both cache types."""
    c = make_unified_case(seq_lens, heads[0], heads[1], 128, 16, dtype, fp8=fp8, seed=heads[0] + len(seq_lens),
                          kv_scale=0.5)
    run(oracle, c, dtype, fp8=fp8)


@pytest.mark.parametrize("mode", ["fp8_out", "hnd", "bs64", "mixed16"])
@pytest.mark.parametrize("fp8", [False, True])
def test_unified_fa_kernel_features(oracle, force_fa, mode, fp8):
    """fp8 output, a head-major cache allocation, 64-token pages, and a batch of >= 16 sequences whose decode tokens
    go to the decode kernel while the 256-row kernel skips them."""
    seqs = [(200, 900), (1, 77), (33, 33), (400, 400)]
    if mode == "mixed16":
        seqs = seqs + [(1, 100 + 37 * i) for i in range(14)]
    c = make_unified_case(seqs, 8, 2, 128, 64 if mode == "bs64" else 16, torch.bfloat16, fp8=fp8, seed=11, kv_scale=0.75)
    view = (lambda t: t.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3)) if mode == "hnd" else None
    run(oracle, c, torch.bfloat16, fp8=fp8, out_scale=torch.tensor([0.03]) if mode == "fp8_out" else None, view=view)


@pytest.mark.parametrize("heads,D", [((8, 2), 128), ((32, 8), 80), ((24, 1), 128), ((4, 4), 128)])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("n,mode", [(16, "plain"), (19, "fp8_out"), (70, "plain")])
def test_unified_mixed_one_launch(oracle, force_fa, heads, D, fp8, n, mode):
    """Chunks and decode tokens in one launch (head-major cache memory): decodes of one key, of fewer steps than the eight waves,
    of one step per wave and one key more, chunks in front of, among and behind them, groups of more than 16 q heads, row
    blocks in a number that is no multiple of 8; with and without the longest-first order."""
    from vllm_amd import _lib
    seqs = [(1, (1, 16, 33, 255, 257, 512, 513, 900)[i % 8]) for i in range(n)]
    seqs[0], seqs[n // 2], seqs[n - 1] = (70, 600), (65, 65), (130, 333)
    c = make_unified_case(seqs, heads[0], heads[1], D, 16, torch.bfloat16, fp8=fp8, seed=n + D, kv_scale=0.5)
    hnd = lambda t: t.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3)
    for order in (1, 0) if n == 70 else (1,):
        _lib.set_tuning("pa_order", order)
        try:
            run(oracle, c, torch.bfloat16, fp8=fp8, out_scale=torch.tensor([0.03]) if mode == "fp8_out" else None, view=hnd)
        finally:
            _lib.set_tuning("pa_order", 1)


def _mixed_launches(key=b"pf_mixed_launches"):
    import ctypes
    from vllm_amd import _lib
    n = ctypes.c_int()
    _lib.check(_lib.lib.vllm_amd_get_tuning(key, ctypes.byref(n)))
    return n.value


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("heads,D,BS", [((8, 2), 128, 32), ((32, 8), 80, 64), ((24, 1), 96, 16), ((4, 4), 128, 128)])
def test_unified_mixed_forms(oracle, force_fa, heads, D, BS, dtype, fp8):
    """The same mixed step in one launch and in two, which each is looked up: both 16-bit types, pages of more than one 16-slot tile."""
    from vllm_amd import _lib
    seqs = [(1, (1, 16, 31, 33, 64, 129, 257, 512, 700)[i % 9]) for i in range(19)]
    seqs[0], seqs[9], seqs[18] = (70, 300), (65, 65), (130, 190)
    c = make_unified_case(seqs, heads[0], heads[1], D, BS, dtype, fp8=fp8, seed=BS + D, kv_scale=0.5)
    hnd = lambda t: t.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3)
    for mixed in (1, 0):
        _lib.set_tuning("pf_mixed", mixed)
        try:
            before = _mixed_launches()
            run(oracle, c, dtype, fp8=fp8, view=hnd)
            assert _mixed_launches() - before == mixed
        finally:
            _lib.set_tuning("pf_mixed", 1)


@pytest.mark.parametrize("n,one", [(64, 1), (65, 0)])
def test_unified_mixed_launch_limit(oracle, force_fa, n, one):
    """512 (sequence, kv head) pairs go along with the chunks, 520 have a launch of their own."""
    seqs = [(1, 1 + 3 * i % 70) for i in range(n)]
    seqs[5], seqs[n - 1] = (66, 80), (35, 35)
    c = make_unified_case(seqs, 8, 8, 128, 16, torch.bfloat16, seed=n)
    before = _mixed_launches()
    run(oracle, c, torch.bfloat16, view=lambda t: t.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3))
    assert _mixed_launches() - before == one


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("heads,D", [((8, 2), 128), ((32, 8), 80), ((24, 1), 96)])
@pytest.mark.parametrize("seqs,one", [
    ([(1, 700), (130, 190)], 1), ([(70, 300), (1, 1), (65, 65), (1, 513)], 1), ([(1, 900), (1, 5), (1, 257), (450, 450)], 1),
    ([(40, 500), (90, 90), (3, 7)], 1),           # no decode, and nothing that tells
    ([(90, 500), (91, 91)], 0), ([(1, 99)] + [(50, 50)] * 5, 0),   # none, and too many tokens for one; one that does not matter
])
def test_unified_few_sequences_one_launch(oracle, force_fa, heads, D, fp8, seqs, one):
    """Fewer than 16 sequences: decodes that may be among the chunks go along as workgroups of the decode kernel."""
    from vllm_amd import _lib
    c = make_unified_case(seqs, heads[0], heads[1], D, 16, torch.bfloat16, fp8=fp8, seed=len(seqs) + D, kv_scale=0.5)
    _lib.set_tuning("pf_segs", 1)
    try:
        before = _mixed_launches()
        run(oracle, c, torch.bfloat16, fp8=fp8, view=lambda t: t.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3))
        assert _mixed_launches() - before == one
    finally:
        _lib.set_tuning("pf_segs", 0)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("heads,D", [((8, 2), 64), ((16, 8), 256), ((4, 4), 128)])
@pytest.mark.parametrize("softcap", [0.0, 20.0])
def test_unified_few_sequences_decodes_apart(oracle, heads, D, fp8, softcap):
    """The same, where the chunks' kernel takes no decodes along: the decode kernel in front of it, and every token written once."""
    from vllm_amd import _lib
    c = make_unified_case([(1, 2100), (300, 310), (1, 1), (2, 900)], heads[0], heads[1], D, 16, torch.bfloat16, fp8=fp8, seed=D, kv_scale=0.5)
    _lib.set_tuning("pf_segs", 1)
    try:
        run(oracle, c, torch.bfloat16, fp8=fp8, softcap=softcap)
    finally:
        _lib.set_tuning("pf_segs", 0)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("heads,D", [((8, 1), 128), ((16, 2), 64), ((8, 2), 256), ((24, 1), 80)])
@pytest.mark.parametrize("window,out8", [(None, False), (700, False), (None, True)])
def test_unified_decodes_cut_beside_segments(oracle, heads, D, fp8, window, out8):
    """Few decodes beside a chunk whose keys are cut into segments: cut too, and merged by the chunk's merge; pieces without a key, of
    one tile and one key more, chunks in front of and behind the decodes."""
    seqs = [(40, 2300)] + [(1, (1, 63, 64, 65, 128, 129, 900, 2200, 1025)[i % 9]) for i in range(15)] + [(9, 30)]
    c = make_unified_case(seqs, heads[0], heads[1], D, 16, torch.bfloat16, fp8=fp8, seed=D, kv_scale=0.5)
    run(oracle, c, torch.bfloat16, fp8=fp8, window=window, out_scale=torch.tensor([0.03]) if out8 else None)


def test_unified_fa_kernel_sharp_rows(oracle, force_fa):
    """Rows whose maximum keeps growing along the keys (the lazy rescale must fire on some tiles and not on others):
    keys scaled up with their position."""
    c = make_unified_case([(300, 1200)], 8, 2, 128, 16, torch.bfloat16, seed=3)
    bt = c["block_table"][0]
    for t in range(1200):
        c["k"][int(bt[t // 16]), t % 16] *= (0.2 + 2.5 * t / 1200)
    run(oracle, c, torch.bfloat16)


@pytest.mark.parametrize("window", [1, 16, 64, 100, 257, 1000])
@pytest.mark.parametrize("heads", [(8, 2), (4, 4), (6, 2)])
@pytest.mark.parametrize("fp8", [False, True])
def test_unified_fa_kernel_window(oracle, force_fa, window, heads, fp8):
    """Sliding windows narrower than a key tile, than a row block's span, and wider: tiles left of the window skipped
    (not even staged for the workgroup's first rows), left-edge tiles masked, interior, diagonal."""
    c = make_unified_case([(700, 700), (300, 1500), (64, 64), (1, 900), (130, 131)], heads[0], heads[1], 128, 16,
                          torch.bfloat16, fp8=fp8, seed=window + heads[0], kv_scale=0.5)
    run(oracle, c, torch.bfloat16, fp8=fp8, window=window)


@pytest.mark.parametrize("D", [72, 80, 96, 112, 120, 136, 160, 192, 224, 256])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_unified_fa_kernel_head_sizes(oracle, force_fa, D, fp8, dtype):
    """Head sizes 72 .. 120 run the 256-row kernel padded to 128 (zero columns from clamped addresses, the last
    sequence ending at the end of the cache allocation), 136 .. 256 its four-wave form padded to 256."""
    if fp8 and D % 16:
        pytest.skip("an fp8 cache needs head sizes that are multiples of 16")
    c = make_unified_case([(300, 700), (1, 90), (70, 70)], 8, 2, D, 16, dtype, fp8=fp8, seed=D, kv_scale=0.5)
    run(oracle, c, dtype, fp8=fp8)
    run(oracle, c, dtype, fp8=fp8, window=50)
    if D == 256:   # unpacked rows, a group that does not divide the 128 rows, fp8 output
        c = make_unified_case([(200, 333), (64, 64)], 6, 2, D, 32, dtype, fp8=fp8, seed=1, kv_scale=0.5)
        run(oracle, c, dtype, fp8=fp8)
        c = make_unified_case([(200, 333), (64, 64)], 4, 4, D, 16, dtype, fp8=fp8, seed=2, kv_scale=0.5)
        run(oracle, c, dtype, fp8=fp8, out_scale=torch.tensor([0.03]))


@pytest.mark.parametrize("soft_cap", [10.0, 50.0])
@pytest.mark.parametrize("D", [128, 256, 96])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("window", [None, 100])
def test_unified_fa_kernel_softcap(oracle, force_fa, soft_cap, D, fp8, window):
    """Soft-capped scores (Gemma-2: 50 with head 256 and alternating sliding windows) in the 256-row kernel: interior and
    masked tiles (a masked score must stay -inf, not -softcap), both head widths, fp8 cache."""
    for dtype in (torch.bfloat16, torch.float16):
        c = make_unified_case([(300, 700), (129, 463), (1, 90), (70, 70)], 8, 2, D, 16, dtype, fp8=fp8,
                              seed=int(soft_cap) + D, kv_scale=0.5)
        run(oracle, c, dtype, fp8=fp8, softcap=soft_cap, window=window)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("D", [128, 112, 256])
@pytest.mark.parametrize("window", [None, 130])
def test_unified_fa_kernel_whole_tiles(oracle, force_fa, window, D, fp8):
    """Runs of at least four whole 64-key tiles are staged without checks while two more follow: sequences of 1 .. 12 whole
    tiles, ending on a tile, one key before and one behind, with and without keys before the chunk; a head size with padding
    columns, which has no such run."""
    for lens in ([(320, 320), (64, 128), (129, 257), (255, 446), (192, 384), (65, 258), (257, 513), (128, 449)],
                 [(449, 449), (384, 769), (33, 416), (130, 514), (512, 512), (64, 512), (383, 766), (577, 577)]):
        c = make_unified_case(lens, 4, 2, D, 16, torch.bfloat16, fp8=fp8, seed=D, kv_scale=0.5)
        run(oracle, c, torch.bfloat16, fp8=fp8, window=window)


@pytest.mark.parametrize("segs", [2, 5, 32])
@pytest.mark.parametrize("num_heads,head_size", [((8, 2), 128), ((8, 8), 64), ((8, 1), 80), ((4, 2), 256)])
@pytest.mark.parametrize("mode", ["plain", "fp8", "window", "softcap", "fp8_out", "mixed"])
def test_unified_prefill_key_segments(oracle, segs, num_heads, head_size, mode):
    """Few row blocks over long key ranges: the 256-row kernel split over the keys.  Segments that end inside a sequence,
    more segments than tiles, rows that see nothing of a segment (the causal edge, the window), a one-token sequence;
    "mixed": 16 sequences, whose one-token ones the decode kernel takes and the merge must leave alone."""
    from vllm_amd import _lib
    lens = [(70, 700), (1, 300), (150, 150), (33, 97)]
    if mode == "mixed":
        lens += [(1, 20 + 40 * i) for i in range(12)]
    fp8 = mode in ("fp8", "fp8_out", "mixed")
    c = make_unified_case(lens, num_heads[0], num_heads[1], head_size, 16, torch.bfloat16, fp8=fp8, seed=segs + head_size,
                          kv_scale=0.5)
    _lib.set_tuning("pf_segs", segs)
    try:
        run(oracle, c, torch.bfloat16, window=100 if mode == "window" else None, softcap=20.0 if mode == "softcap" else 0.0,
            out_scale=torch.tensor([0.02]) if mode == "fp8_out" else None, fp8=fp8)
    finally:
        _lib.set_tuning("pf_segs", 0)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("D", [128, 256])
def test_unified_prefill_key_segments_nan(oracle, D, fp8):
    """A NaN query, and NaN keys that a whole sequence sees (a whole tile: the first of a segment, for some of the segment
    counts), make exactly the rows NaN that see them -- split over the keys as unsplit."""
    from vllm_amd import _lib
    from vllm_amd.attention.ops import unified_attention
    c = make_unified_case([(70, 700), (33, 97), (90, 350)], 8, 2, D, 16, torch.bfloat16, fp8=fp8, seed=D, kv_scale=0.5)
    kd = c["scale"] if fp8 else None
    ref = torch.zeros_like(c["q"])
    oracle.unified_attention(c["q"], c["k"], c["v"], ref, c["cu_seqlens_q"], c["max_seqlen_q"], c["seqused_k"],
                             c["max_seqlen_k"], D ** -0.5, True, (-1, -1), c["block_table"], 0.0, None, kd, kd, None, None)
    bad = torch.zeros(c["q"].shape[:2], dtype=torch.bool)
    c["q"][40, 5] = float("nan")
    bad[40, 5] = True
    for n in range(128, 192):   # the third sequence's third tile, kv head 1
        c["k"][int(c["block_table"][2, n // 16]), n % 16, 1] = 0x7f if fp8 else float("nan")
    bad[103:, 4:] = True
    d = {k: v.cuda() for k, v in c.items() if torch.is_tensor(v)}
    kd = d["scale"] if fp8 else None
    _lib.set_tuning("pf_fa", 2)
    try:
        for segs in (1, 2, 3, 5, 32):
            _lib.set_tuning("pf_segs", segs)
            out = torch.zeros_like(d["q"])
            unified_attention(d["q"], d["k"], d["v"], out, d["cu_seqlens_q"], c["max_seqlen_q"], d["seqused_k"], c["max_seqlen_k"], D ** -0.5,
                              True, (-1, -1), d["block_table"], 0.0, None, kd, kd)
            out = out.cpu()
            assert torch.equal(out.isnan().any(-1), bad) and torch.equal(out.isnan().all(-1), bad), segs
            torch.testing.assert_close(out.float()[~bad], ref.float()[~bad], atol=ATOL, rtol=RTOL)
    finally:
        _lib.set_tuning("pf_segs", 0)
        _lib.set_tuning("pf_fa", 0)


@pytest.mark.parametrize("D", [32, 80, 120, 192, 256])
@pytest.mark.parametrize("nseq", [5, 260])
@pytest.mark.parametrize("window", [None, 100])
def test_unified_decode_keys_of_minus_infinity(oracle, D, nseq, window):
    """A key whose score is -inf has probability 0: the columns that pad the head size inside the decode kernel must not
    make a NaN of it (0 * inf).  Split and unsplit launches, one kv head per row ("uni_hp" = 1)."""
    from vllm_amd import _lib
    lens = [33, 64, 130, 500]
    c = make_unified_case([(1, lens[i % 4] + i // 4) for i in range(nseq)], 8, 2, D, 16, torch.bfloat16, seed=D + nseq)
    c["q"][..., 3] = c["q"][..., 3].abs() + 0.5
    for i, n in enumerate(c["seqused_k"].tolist()):
        for t in {n // 2, n - 1, 5}:
            c["k"][int(c["block_table"][i, t // 16]), t % 16, :, 3] = float("-inf")
    _lib.set_tuning("uni_hp", 1)
    try:
        run(oracle, c, torch.bfloat16, window=window)
    finally:
        _lib.set_tuning("uni_hp", 0)


@pytest.mark.parametrize("kernel", ["64 rows", "256 rows", "split"])
def test_unified_rows_in_front_of_the_first_sequence(oracle, kernel):
    """cu_seqlens_q that starts above 0 (the last sequences of a longer batch): the others' rows are left alone."""
    from vllm_amd import _lib
    from vllm_amd.attention.ops import unified_attention
    c = make_unified_case([(300, 340), (70, 570), (1, 78), (90, 290)], 8, 2, 128, 16, torch.bfloat16, seed=3)
    ref = torch.zeros_like(c["q"])
    oracle.unified_attention(c["q"], c["k"], c["v"], ref, c["cu_seqlens_q"], c["max_seqlen_q"], c["seqused_k"],
                             c["max_seqlen_k"], 128 ** -0.5, True, (-1, -1), c["block_table"], 0.0, None, None, None, None, None)
    d = {k: v.cuda() for k, v in c.items() if torch.is_tensor(v)}
    _lib.set_tuning("pf_fa", 1 if kernel == "64 rows" else 2)
    _lib.set_tuning("pf_segs", 3 if kernel == "split" else 0)
    try:
        for first in (1, 3):
            out = torch.zeros_like(d["q"])
            unified_attention(d["q"], d["k"], d["v"], out, d["cu_seqlens_q"][first:], c["max_seqlen_q"], d["seqused_k"][first:],
                              c["max_seqlen_k"], 128 ** -0.5, True, (-1, -1), d["block_table"][first:], 0.0, None, None, None)
            out, at = out.cpu(), int(c["cu_seqlens_q"][first])
            assert float(out[:at].abs().max()) == 0.0
            torch.testing.assert_close(out[at:].float(), ref[at:].float(), atol=ATOL, rtol=RTOL)
    finally:
        _lib.set_tuning("pf_segs", 0)
        _lib.set_tuning("pf_fa", 0)


@pytest.mark.parametrize("segs", [1, 3, 6, 16])
def test_unified_decode_rows_that_are_not_the_sequence_number(oracle, segs):
    """Decode tokens behind rows of other sequences, and an empty sequence among them: the merge finds each one's own row."""
    from vllm_amd import _lib
    from vllm_amd.attention.ops import unified_attention
    c = make_unified_case([(1, n) for n in (5, 300, 1100, 64, 900, 1025)], 8, 2, 128, 16, torch.bfloat16, seed=segs)
    ref = torch.zeros_like(c["q"])
    oracle.unified_attention(c["q"], c["k"], c["v"], ref, c["cu_seqlens_q"], 1, c["seqused_k"],
                             c["max_seqlen_k"], 128 ** -0.5, True, (-1, -1), c["block_table"], 0.0, None, None, None, None, None)
    d = {k: v.cuda() for k, v in c.items() if torch.is_tensor(v)}
    cu, at = torch.tensor([2, 3, 3, 4, 5, 6], dtype=torch.int32, device="cuda"), torch.tensor([2, 0, 3, 4, 5], device="cuda")
    out = torch.zeros_like(d["q"])
    _lib.set_tuning("uni_seg", segs)
    try:
        unified_attention(d["q"], d["k"], d["v"], out, cu, 1, d["seqused_k"][at].contiguous(), c["max_seqlen_k"], 128 ** -0.5, True,
                          (-1, -1), d["block_table"][at].contiguous(), 0.0, None, None, None)
    finally:
        _lib.set_tuning("uni_seg", 0)
    ref[:2] = 0
    torch.testing.assert_close(out.cpu().float(), ref.float(), atol=ATOL, rtol=RTOL)


def test_unified_scales_of_an_unquantised_cache_are_not_read(oracle):
    """A cache in the query's type: k_descale / v_descale may be anywhere (a layer's scales on the host); with fp8 they may not."""
    from vllm_amd.attention.ops import unified_attention
    for fp8 in (False, True):
        c = make_unified_case([(70, 170), (1, 30)], 4, 2, 128, 16, torch.bfloat16, fp8=fp8, seed=1, kv_scale=0.5)
        d = {k: v.cuda() for k, v in c.items() if torch.is_tensor(v)}
        out = torch.zeros_like(d["q"])
        call = lambda: unified_attention(d["q"], d["k"], d["v"], out, d["cu_seqlens_q"], c["max_seqlen_q"], d["seqused_k"],
                                         c["max_seqlen_k"], 128 ** -0.5, True, (-1, -1), d["block_table"], 0.0, None, c["scale"],
                                         c["scale"])
        if fp8:
            with pytest.raises(RuntimeError, match="device tensors"):
                call()
        else:
            call()
            ref = torch.zeros_like(c["q"])
            oracle.unified_attention(c["q"], c["k"], c["v"], ref, c["cu_seqlens_q"], c["max_seqlen_q"], c["seqused_k"],
                                     c["max_seqlen_k"], 128 ** -0.5, True, (-1, -1), c["block_table"], 0.0, None, None, None, None,
                                     None)
            torch.testing.assert_close(out.cpu().float(), ref.float(), atol=ATOL, rtol=RTOL)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("n", [20, 64, 65, 140])
def test_unified_prefill_key_segments_among_decodes(oracle, n, fp8):
    """Chunks anywhere among many decode tokens, split over the keys: workgroups go to the chunks' row blocks only, which are
    looked for in rounds of 64 sequences; a fresh chunk stays whole."""
    from vllm_amd import _lib
    seqs = [(1, 5 + 3 * i) for i in range(n)]
    seqs[0], seqs[n // 2], seqs[n - 1] = (70, 600), (40, 40), (5, 333)
    c = make_unified_case(seqs, 8, 2, 128, 16, torch.bfloat16, fp8=fp8, seed=n, kv_scale=0.5)
    for segs in (2, 4):
        _lib.set_tuning("pf_segs", segs)
        try:
            run(oracle, c, torch.bfloat16, fp8=fp8)
        finally:
            _lib.set_tuning("pf_segs", 0)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("D,heads", [(80, (8, 2)), (128, (32, 8)), (256, (8, 4)), (64, (8, 2))])
@pytest.mark.parametrize("window", [100, 600, 1500])
@pytest.mark.parametrize("soft_cap", [None, 30.0])
def test_unified_window_far_behind(oracle, fp8, D, heads, window, soft_cap):
    """Windows that leave more than 16 key tiles of the longest sequence out: chunks of any length take the 256-row kernel, in
    one piece (100), cut by the keys that a row block walks (600) or by all of them (1500); shorter sequences beside it."""
    c = make_unified_case([(200, 2600), (3, 1500), (70, 70), (1, 700)], *heads, D, 16, torch.bfloat16, fp8=fp8, seed=D + window)
    run(oracle, c, torch.bfloat16, window=window, softcap=soft_cap or 0.0, fp8=fp8)


# (query, key) lengths -> row blocks of 256 / group tokens and their halves
ROW_BLOCKS = {
    "halves": ([(33, 33), (32, 32), (96, 96), (129, 129), (200, 500), (1, 70), (64, 65), (2, 300)], (8, 2)),     # 1, 2, 3, 5, 7 halves of 32 tokens
    "one head": ([(129, 129), (257, 400), (128, 300), (300, 300)], (4, 4)),                                       # halves of 128 tokens
    "group of 16": ([(9, 9), (8, 80), (17, 17), (40, 200)], (16, 1)),
    "group of 3": ([(43, 43), (85, 85), (86, 300), (171, 171)], (6, 2)),                                          # does not divide 128: no pairs
    "one round": ([(2 + i, 10 + 3 * i) for i in range(32)], (8, 8)),                                              # 256 row blocks
    "past one round": ([(2 + i, 10 + 3 * i) for i in range(33)], (8, 8)),                                         # 264
    "past 64 sequences": ([(2 + i % 40, 3 + 2 * i) if i % 7 else (1, 50) for i in range(80)], (4, 2)),
}


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("blocks", ROW_BLOCKS)
def test_unified_row_blocks(oracle, force_fa, fp8, blocks):
    """The unsplit 256-row kernel where its row blocks are dealt out: half blocks paired from the front and the back of a chunk up to
    one round of workgroups, whole ones above, more sequences than lanes."""
    from vllm_amd import _lib
    seqs, heads = ROW_BLOCKS[blocks]
    c = make_unified_case(seqs, heads[0], heads[1], 128, 16, torch.bfloat16, fp8=fp8, seed=len(seqs), kv_scale=0.5)
    _lib.set_tuning("pf_segs", 1)
    try:
        run(oracle, c, torch.bfloat16, fp8=fp8)
    finally:
        _lib.set_tuning("pf_segs", 0)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("heads,D,seqs", [
    ((8, 2), 128, [(40 + 31 * (i % 5), 40 + 31 * (i % 5) + 7 * (i % 3)) for i in range(60)]),           # 2 heads: 4 XCDs each, 300 blocks
    ((16, 1), 128, [(100 + 53 * (i % 4), 150 + 61 * (i % 4)) for i in range(25)]),                      # 1 head, halves of 8 tokens, 300 blocks
    ((16, 4), 128, [(300 + i, 300 + i) for i in range(15)] + [(1, 9)]),                                 # 4 heads, 304 blocks, the last of one token
    ((8, 8), 128, [(1 + 17 * i % 290, 20 + 29 * i) for i in range(36)]),                                # whole heads per XCD, short and long contexts
    ((16, 8), 256, [(3 + 40 * (i % 6), 3 + 40 * (i % 6)) for i in range(14)]),                          # 128-row blocks
    ((128, 8), 128, [(530, 530), (512, 512)]),                                                          # two prompts, 528 blocks
])
def test_unified_row_block_order(oracle, force_fa, fp8, heads, D, seqs):
    """More than one round of row blocks: in the order of their last keys, in shares per XCD for few heads; every block once."""
    from vllm_amd import _lib
    c = make_unified_case(seqs, heads[0], heads[1], D, 16, torch.bfloat16, fp8=fp8, seed=len(seqs), kv_scale=0.5)
    _lib.set_tuning("pf_segs", 1)
    try:
        run(oracle, c, torch.bfloat16, fp8=fp8)
    finally:
        _lib.set_tuning("pf_segs", 0)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("heads,seqs", [
    ((16, 1), [(1, 30 + 7 * i) for i in range(66)] + [(100 + 53 * (i % 4), 150 + 61 * (i % 4)) for i in range(25)]),   # 300 row blocks
    ((8, 2), [(1, 5 + 3 * i) for i in range(64)] + [(40 + 31 * (i % 5), 40 + 31 * (i % 5) + 7 * (i % 3)) for i in range(60)]),
    ((16, 4), [(300 + i, 300 + i) for i in range(8)] + [(1, 9 + i) for i in range(70)] + [(310 + i, 310 + i) for i in range(8)]),
    ((16, 1), [(1, 40)] * 70 + [(60 + i, 600 + i) for i in range(70)]),                                                # short ones over long contexts: runs
])
def test_unified_row_block_order_behind_decodes(oracle, force_fa, fp8, heads, seqs):
    """1, 2 or 4 heads and more than one round of row blocks behind more decodes than lanes: every block once."""
    from vllm_amd import _lib
    c = make_unified_case(seqs, heads[0], heads[1], 128, 16, torch.bfloat16, fp8=fp8, seed=len(seqs), kv_scale=0.5)
    _lib.set_tuning("pf_segs", 1)
    try:
        run(oracle, c, torch.bfloat16, fp8=fp8)
    finally:
        _lib.set_tuning("pf_segs", 0)


def test_unified_shares_behind_decodes():
    """One kv head, two prompts of 5000 tokens: the row blocks are dealt out in shares whether 40 or 80 decodes stand in front of them.
    (In runs, as when only the first 64 sequences were looked at, the step took 1.6 times as long; what the decodes add is 2 %.)"""
    from vllm_amd.attention.ops import unified_attention
    g = torch.Generator(device="cuda").manual_seed(0)
    r = lambda *s: torch.randn(s, generator=g, device="cuda").to(torch.bfloat16)
    cache = r(2, 700, 16, 1, 128)
    def step(n):
        lens = [(1, 200)] * n + [(5000, 5000), (5000, 5000)]
        q = r(sum(a for a, _ in lens), 8, 128)
        cu = torch.tensor([0] + [a for a, _ in lens], dtype=torch.int32, device="cuda").cumsum(0).to(torch.int32)
        table = torch.randint(700, (n + 2, 313), generator=g, device="cuda", dtype=torch.int32)
        used, out = torch.tensor([b for _, b in lens], dtype=torch.int32, device="cuda"), torch.empty_like(q)
        return lambda: unified_attention(q, cache[0], cache[1], out, cu, 5000, used, 5000, 0.088, True, (-1, -1), table, 0.0, None, None, None)
    def us(f):
        t = []
        for _ in range(8):
            a, b = torch.cuda.Event(True), torch.cuda.Event(True)
            a.record(); f(); b.record(); torch.cuda.synchronize(); t.append(a.elapsed_time(b))
        return sorted(t)[2]
    few, many = step(40), step(80)
    us(few), us(many)
    assert us(many) < 1.25 * us(few)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("heads,seqs", [
    ((64, 32), [(400, 400), (350, 350), (300, 300), (290, 290), (280, 280), (401, 401)]),            # six of two q heads: 560 blocks
    ((32, 32), [(256 + 20 * i, 256 + 20 * i) for i in range(8)] + [(1, 1)]),                          # nine of one: 544 blocks
    ((128, 32), [(400, 400), (430, 430), (300, 300)]),                                                # three of four: 576
    ((128, 32), [(400, 401), (430, 430), (300, 300)]),                                                # one of them over a context: by sequence
])
def test_unified_row_blocks_of_more_rounds_by_last_keys(oracle, force_fa, fp8, heads, seqs):
    """More than two rounds of row blocks without a context, by their last keys where few chunks share an XCD."""
    from vllm_amd import _lib
    c = make_unified_case(seqs, heads[0], heads[1], 128, 16, torch.bfloat16, fp8=fp8, seed=len(seqs), kv_scale=0.5)
    _lib.set_tuning("pf_segs", 1)
    try:
        run(oracle, c, torch.bfloat16, fp8=fp8)
    finally:
        _lib.set_tuning("pf_segs", 0)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("heads,D", [((8, 2), 64), ((16, 8), 256), ((4, 4), 128)])
@pytest.mark.parametrize("softcap", [0.0, 20.0])
def test_unified_few_sequences_long_decodes(oracle, heads, D, fp8, softcap):
    """Fewer than 16 sequences with a decode of 3100 keys: in a launch of their own where the chunks' kernel takes none along, and as row
    blocks where a key is 1024 bytes; every token written once."""
    from vllm_amd import _lib
    c = make_unified_case([(1, 3100), (300, 310), (1, 1), (2, 900)], heads[0], heads[1], D, 16, torch.bfloat16, fp8=fp8, seed=D + 1, kv_scale=0.5)
    _lib.set_tuning("pf_segs", 1)
    try:
        run(oracle, c, torch.bfloat16, fp8=fp8, softcap=softcap)
    finally:
        _lib.set_tuning("pf_segs", 0)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("seqs", [
    [(1, 1100), (150, 400), (1, 7), (170, 170), (1, 900), (163, 300), (1, 1030)],        # the decodes start behind 192 of 256 row blocks
    [(150, 400), (170, 180), (163, 600), (160, 160), (2, 700)],                          # none
])
def test_unified_decodes_between_row_blocks(oracle, force_fa, fp8, seqs):
    """Decodes behind the first 192 workgroup ids, row blocks on both sides of them: with a group of 16 q heads 16 tokens are a row
    block, and 8 kv heads make 240 of them."""
    from vllm_amd import _lib
    c = make_unified_case(seqs, 128, 8, 128, 16, torch.bfloat16, fp8=fp8, seed=len(seqs), kv_scale=0.5)
    _lib.set_tuning("pf_segs", 1)
    try:
        before = _mixed_launches()
        run(oracle, c, torch.bfloat16, fp8=fp8, view=lambda t: t.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3))
        assert _mixed_launches() - before == 1
    finally:
        _lib.set_tuning("pf_segs", 0)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("heads,D,decodes,most,cut", [
    ((8, 1), 128, 15, 2200, 1), ((16, 2), 64, 15, 2200, 1), ((8, 2), 256, 15, 2200, 1), ((24, 1), 80, 15, 2200, 1),
    ((8, 1), 128, 63, 2200, 0),       # 65 (sequence, kv head) pairs
    ((8, 1), 128, 15, 1900, 0),       # fewer than 2048 keys
])
def test_unified_decodes_cut_beside_segments_taken(oracle, heads, D, decodes, most, cut, fp8):
    """The same, with a look at whether the chunk's merge took the decodes along."""
    seqs = [(40, most)] + [(1, (1, 63, 64, 65, 128, 129, 900, most - 100, 1025)[i % 9]) for i in range(decodes)] + [(9, 30)]
    c = make_unified_case(seqs, heads[0], heads[1], D, 16, torch.bfloat16, fp8=fp8, seed=D, kv_scale=0.5)
    before = _mixed_launches(b"pf_cut_launches")
    run(oracle, c, torch.bfloat16, fp8=fp8)
    assert _mixed_launches(b"pf_cut_launches") - before == cut
