"""CPU tests (no GPU) of the host-side mirrors: PagedAttention helper (shapes, v1/v2
heuristic, scratch shapes), Fp8LinearOp plumbing, TP sharding, and a world_size-2 gloo
run of the N>1 path (KV-head-sharded attention + row-parallel GEMM + all-reduce) with the
oracle standing in for the kernels."""
import os
import socket

import pytest
import torch
import torch.multiprocessing as mp

from helpers import make_attn_case


def test_kv_cache_shape_and_split():
    from vllm_amd.attention import PagedAttention
    assert PagedAttention.get_kv_cache_shape(10, 16, 8, 128) == (2, 10, 16 * 8 * 128)
    kv = torch.zeros(PagedAttention.get_kv_cache_shape(10, 16, 8, 128), dtype=torch.bfloat16)
    k, v = PagedAttention.split_kv_cache(kv, 8, 128)
    assert k.shape == (10, 8, 16, 16, 8) and v.shape == (10, 8, 128, 16)
    kv8 = torch.zeros(PagedAttention.get_kv_cache_shape(10, 16, 8, 128), dtype=torch.uint8)
    k, v = PagedAttention.split_kv_cache(kv8, 8, 128)
    assert k.shape == (10, 8, 8, 16, 16) and v.shape == (10, 8, 128, 16)
    assert 120 in PagedAttention.get_supported_head_sizes()


@pytest.mark.parametrize("S,H,max_len,want,KVH", [
    (64, 32, 4096, "v1", 8),      # configs[1]: S*H = 2048 > 512
    (8, 64, 131072, "v2", 8),     # configs[4]: > 8192
    (4, 32, 300, "v1", 8),        # one partition
    (4, 32, 2048, "v2", 8),       # S*H = 128 <= 512 and 4 partitions
    (256, 8, 32768, "v2", 8),     # configs[3]
    (128, 8, 4096, "v2", 1),      # S*H = 1024 > 512, but 128 (sequence, kv head) workgroups: partitioned here
    (256, 8, 2048, "v1", 1),      # 256 workgroups: one per CU
])
def test_forward_decode_heuristic(monkeypatch, S, H, max_len, want, KVH):
    """vllm/attention/ops/paged_attn.py:117-193: same choice (refined where this implementation's workgroup count
    differs from the reference's, see forward_decode) and scratch shapes."""
    from vllm_amd.attention import paged_attn
    calls = {}
    monkeypatch.setattr(paged_attn.ops, "paged_attention_v1",
                        lambda *a, **k: calls.setdefault("v1", a))
    monkeypatch.setattr(paged_attn.ops, "paged_attention_v2",
                        lambda *a, **k: calls.setdefault("v2", a))
    q = torch.zeros((S, H, 128), dtype=torch.bfloat16)
    kc = torch.zeros((4, 8, 16, 16, 8), dtype=torch.bfloat16)
    vc = torch.zeros((4, 8, 128, 16), dtype=torch.bfloat16)
    bt = torch.zeros((S, (max_len + 15) // 16), dtype=torch.int32)
    sl = torch.ones(S, dtype=torch.int32)
    one = torch.ones(1)
    out = paged_attn.PagedAttention.forward_decode(q, kc, vc, bt, sl, max_len, "auto", KVH, 0.1,
                                                   None, one, one)
    assert out.shape == q.shape and list(calls) == [want]
    if want == "v2":
        P = (max_len + 511) // 512
        _, es, ml, tmp = calls["v2"][:4]
        assert es.shape == (S, H, P) and ml.shape == (S, H, P) and tmp.shape == (S, H, P, 128)
        assert es.dtype == torch.float32 and tmp.dtype == q.dtype


@pytest.mark.parametrize("S,H,KVH,D,BS,dtype,kv,want", [
    (1, 32, 8, 128, 16, torch.bfloat16, "fp8", "decode"),
    (8, 32, 8, 128, 16, torch.bfloat16, "auto", "decode"),
    (8, 32, 8, 128, 8, torch.bfloat16, "auto", "decode"),
    (4, 16, 8, 256, 32, torch.float16, "auto", "decode"),
    (4, 16, 8, 64, 16, torch.float32, "auto", "decode"),
    (40, 32, 8, 128, 16, torch.bfloat16, "auto", "v1"),       # 320 workgroups: one per CU and more
    (200, 32, 1, 128, 16, torch.bfloat16, "fp8", "v1"),       # 32 q heads per kv head: two workgroups each
])
def test_forward_decode_two_partitions(monkeypatch, S, H, KVH, D, BS, dtype, kv, want):
    """Between 513 and 1024 keys the operator that knows the plan decides, whatever the types and shapes; no scratch from here."""
    from vllm_amd.attention import paged_attn
    calls = {}
    for mod, name, key in ((paged_attn.ops, "paged_attention_v1", "v1"), (paged_attn.ops, "paged_attention_v2", "v2"),
                           (paged_attn._torch_ops, "paged_attention_decode", "decode")):
        monkeypatch.setattr(mod, name, lambda *a, key=key, **k: calls.setdefault(key, a))
    x = 16 // (torch.empty(0, dtype=dtype).element_size() if kv == "auto" else 1)
    cdt = dtype if kv == "auto" else torch.uint8
    q = torch.zeros((S, H, D), dtype=dtype)
    kc, vc = torch.zeros((4, KVH, D // x, BS, x), dtype=cdt), torch.zeros((4, KVH, D, BS), dtype=cdt)
    bt, sl, one = torch.zeros((S, 4096 // BS), dtype=torch.int32), torch.ones(S, dtype=torch.int32), torch.ones(1)
    out = paged_attn.PagedAttention.forward_decode(q, kc, vc, bt, sl, 777, kv, KVH, 0.1, None, one, one, blocksparse_vert_stride=None)
    assert out.shape == q.shape and list(calls) == [want]
    if want == "decode":   # the arguments of v1
        a = calls["decode"]
        assert a[0] is out and a[1] is q and a[8:10] == (BS, 777) and a[11] == kv and len(a) == 19


def test_paged_attention_v2_pieces():
    """The plan without a device: one piece, two, and every call that is not the matrix-core kernel's."""
    from vllm_amd._lib import BF16, F32, KV_AUTO, KV_FP8_E4M3, lib

    def pieces(S=1, H=32, D=128, KVH=8, BS=16, L=777, P=2, dt=BF16, kv=KV_FP8_E4M3, out=1 << 20, q=1 << 21, q_stride=None, head_stride=None, vert=0):
        return lib.vllm_amd_paged_attention_v2_pieces(out, q, S, H, D, KVH, BS, L, P, dt, kv, H * D if q_stride is None else q_stride,
                                                      D * BS if head_stride is None else head_stride, vert)

    assert pieces() == 1 and pieces(S=16, L=1000) == 1 and pieces(kv=KV_AUTO) == 1
    assert pieces(S=8, L=1000, kv=KV_AUTO) == 2 and pieces(S=4, L=1024, kv=KV_AUTO) == 2
    assert pieces(L=300, P=1) == 1 and pieces(S=0) == 1
    for other in (dict(dt=F32, kv=KV_AUTO), dict(BS=8), dict(vert=2), dict(q=(1 << 21) + 8), dict(q_stride=32 * 128 + 4), dict(head_stride=128 * 16 + 16),
                  dict(out=(1 << 20) + 8)):
        assert pieces(**other) == 2, other
    assert pieces(L=8000, P=16) > 1


@pytest.mark.parametrize("M,N,K,kernel", [
    (32, 1280, 8192, 3711), (64, 1024, 4096, 3711), (40, 1248, 15360, 3711), (64, 2048, 8192, 3721), (40, 2480, 1536, 3712),
    (94, 1280, 8192, 3721), (84, 2048, 16384, 3731), (63, 4096, 4096, 3722), (150, 1280, 1152, 3722), (138, 1296, 1024, 3722),
    # 32 columns over a short K: all rows in one workgroup
    (39, 2560, 1024, 37), (48, 2144, 1152, 37), (48, 2144, 1280, 3712), (50, 3504, 512, 37), (56, 3280, 1920, 37), (56, 3280, 2048, 3722),
    # a nearly empty last group over a long one
    (33, 2192, 14336, 37), (35, 2192, 14336, 37), (36, 2192, 14336, 3712), (36, 2560, 20480, 37), (37, 2560, 20480, 3712),
    (33, 2240, 8192, 3712), (33, 2192, 13312, 3712), (53, 4096, 15360, 37), (55, 3584, 20480, 37), (56, 3584, 20480, 3722), (54, 3888, 14336, 3722),
    (53, 4096, 10240, 3722), (49, 2560, 15360, 3722), (66, 2560, 16384, 3722), (66, 2192, 20480, 10), (83, 2192, 20480, 10), (84, 2192, 20480, 3722),
    # ... and beside tile kernels with four K blocks per barrier
    (91, 2560, 3584, 10), (91, 2560, 3456, 3722), (91, 2560, 4096, 3722), (100, 2048, 1024, 3722), (91, 2048, 1536, 3731),
    # one group, more rounds than one, too many columns
    (16, 1280, 8192, 37), (32, 4096, 4096, 37), (48, 4096, 4096, 37), (48, 6144, 4096, 37), (60, 4160, 4096, 37),
])
def test_scaled_mm_row_groups_rule(M, N, K, kernel):
    """The rows of the weight stream in groups: 3700 + 10 (rows / 16) + columns / 16 of a workgroup, 37 in one."""
    from vllm_amd._lib import lib
    assert lib.vllm_amd_scaled_mm_kernel(M, N, K, 0) == kernel


@pytest.mark.parametrize("M,N,K,kernel", [
    (4096, 4096, 4096, 2), (3072, 6144, 4096, 39), (2048, 6144, 4096, 39), (512, 7168, 8192, 38), (128, 6144, 4096, 7),
    (1024, 10240, 8192, 39), (1536, 6144, 4096, 39), (288, 6144, 4096, 7), (384, 6144, 2048, 38), (1700, 1280, 8192, 38),
    (303, 1696, 6400, 9), (241, 2560, 5120, 7),                 # up to 288 tiles of 64 x 32 stay
    (2852, 11960, 256, 39), (2873, 10896, 384, 39),             # the narrow wide tile where the costs do not reach
    (467, 23432, 384, 3), (419, 16728, 384, 39), (977, 11720, 512, 39), (453, 16672, 512, 39), (674, 16088, 768, 39),   # a full third round of short K loops, a nearly empty one, K 768
    (66, 27848, 384, 38), (66, 28240, 256, 3),                  # K groups
    (1065, 13264, 10368, 3), (6553, 2320, 7424, 3), (8474, 1896, 12672, 39), (1572, 9480, 640, 3),   # tall outputs
])
def test_scaled_mm_tile_rule(M, N, K, kernel):
    """The tile above M 64: the table, and the cost of whole rounds where that overrules it."""
    from vllm_amd._lib import lib
    assert lib.vllm_amd_scaled_mm_kernel(M, N, K, 0) == kernel


def test_scaled_mm_two_slices_rule():
    """Two K slices (1000 + tile) instead of the weight stream where there is a workspace, not instead of small groups of rows."""
    from vllm_amd._lib import lib
    k = lib.vllm_amd_scaled_mm_kernel
    assert k(48, 4096, 14336, 1) == 1010 and k(48, 4096, 14336, 0) == 37 and k(32, 4096, 14336, 1) == 37
    assert k(40, 1248, 15360, 1) == 3711 and k(44, 2192, 14336, 1) == 3712 and k(60, 2560, 14336, 1) == 1010 and k(60, 2560, 14336, 0) == 3722
    assert k(100, 512, 12288, 1) == 3711 and k(0, 512, 1024, 1) == k(8, 512, 128, 1) == k(8, 516, 1024, 1) == 0


PAIRS, SHARES, BY_END, LONGEST = 1, 2, 4, 8


def _order(group, heads, blocks, chunks=1, over=0, cached=0, head=128, seqs=None, decodes=0, window=0, max_len=8192):
    from vllm_amd._lib import lib
    return lib.vllm_amd_prefill_order(head, group, heads, chunks + decodes if seqs is None else seqs, blocks, chunks, over, cached, decodes, window, max_len)


def test_prefill_order_shares():
    """1, 2 or 4 kv heads: shares per XCD in more than one round of row blocks or of a single chunk, not in one of several, and not under a
    window of less than 512 and a fifth of the keys."""
    assert _order(8, 1, 256) == PAIRS and _order(8, 1, 257) == SHARES and _order(4, 4, 64) == PAIRS and _order(4, 4, 65) == SHARES
    for one in (dict(head=256), dict(group=12), dict(window=4000), dict(decodes=20)):       # what keeps a round from being paired
        args = {"group": 8, "heads": 2, "blocks": 128, "chunks": 2, **one}
        assert _order(**args) & SHARES == 0 and _order(**{**args, "blocks": 129}) & SHARES == SHARES, one
        assert _order(**{**args, "chunks": 1}) == (0 if "window" in one else SHARES), one
    assert _order(8, 1, 400, window=512) == SHARES and _order(8, 1, 400, window=511) == 0
    assert _order(8, 1, 400, window=300, max_len=1500) == SHARES and _order(8, 1, 400, window=300, max_len=1501) == 0
    assert _order(8, 8, 400) == 0 and _order(8, 3, 400) == 0
    assert _order(8, 1, 400, chunks=3, over=1) == SHARES | BY_END and _order(8, 1, 400, chunks=3, over=2) == 0


def test_prefill_order_by_last_keys():
    """Several chunks in the order of their last keys: by the query tokens that share a key on an XCD, 32 x tokens per row block / chunks."""
    for group, two_rounds, more in ((4, 16, 3), (8, 8, 1), (2, 16, 6), (1, 16, 12), (16, 4, 0)):
        heads = 8 if group > 1 else 32
        for blocks, most in ((512 // heads, two_rounds), (512 // heads + 1, more), (2048 // heads, more), (2048 // heads + 1, 0)):
            for chunks in range(2, 20):
                assert _order(group, heads, blocks, chunks=chunks) == (BY_END if chunks <= most else 0), (group, blocks, chunks)
    assert _order(4, 8, 64, chunks=3, cached=3) == BY_END and _order(4, 8, 65, chunks=3, cached=1) == 0           # over a context
    assert _order(4, 8, 64, chunks=4, over=1) == BY_END and _order(4, 8, 64, chunks=4, over=2) == LONGEST
    assert _order(4, 8, 64, chunks=4, over=2, decodes=1) == 0 and _order(12, 8, 64, chunks=2) == 0                # a group that does not divide 128
    assert _order(2, 8, 600, chunks=30, head=256) == BY_END and _order(4, 8, 64, chunks=2, seqs=65) == 0
    assert _order(4, 8, 32, chunks=4) == PAIRS


def test_shard_helpers():
    from vllm_amd.distributed import shard_kv_heads, shard_range
    assert shard_range(8192, 8, 3) == (3072, 4096)
    assert shard_kv_heads(64, 8, 8, 5) == ((40, 48), (5, 6))
    assert shard_kv_heads(32, 8, 2, 1) == ((16, 32), (4, 8))
    with pytest.raises(ValueError):
        shard_kv_heads(32, 8, 3, 0)


def _free_port():
    s = socket.socket(); s.bind(("127.0.0.1", 0)); p = s.getsockname()[1]; s.close(); return p


def _tp_worker(rank, world, port, q):
    import torch.distributed as dist
    import sys
    here = os.path.dirname(os.path.abspath(__file__))
    sys.path[:0] = [os.path.dirname(here), here]
    from oracle import oracle as O
    from vllm_amd.distributed import shard_kv_heads, shard_range, tensor_model_parallel_all_reduce
    os.environ["MASTER_ADDR"] = "127.0.0.1"
    os.environ["MASTER_PORT"] = str(port)
    dist.init_process_group("gloo", rank=rank, world_size=world)
    try:
        # ---- attention: every rank owns KVH/world kv heads, no collective inside ----
        H, KVH, D, BS = 8, 2, 64, 16
        c = make_attn_case(3, H, KVH, D, BS, torch.bfloat16, "fp8", [5, 200, 530], seed=1, kv_scale=0.5)
        (h0, h1), (k0, k1) = shard_kv_heads(H, KVH, world, rank)
        qs = c["q"][:, h0:h1].contiguous()
        kcs, vcs = c["kc"][:, k0:k1].contiguous(), c["vc"][:, k0:k1].contiguous()
        out_s = torch.empty_like(qs)
        O.paged_attention_v1(out_s, qs, kcs, vcs, k1 - k0, c["scale"], c["bt"], c["sl"], BS,
                             c["max_len"], None, "fp8", 0.5, 0.5)
        gathered = [torch.empty_like(out_s) for _ in range(world)]
        dist.all_gather(gathered, out_s)
        full = torch.empty_like(c["q"])
        O.paged_attention_v1(full, c["q"], c["kc"], c["vc"], KVH, c["scale"], c["bt"], c["sl"], BS,
                             c["max_len"], None, "fp8", 0.5, 0.5)
        ok_attn = torch.equal(torch.cat(gathered, dim=1), full)   # sharding is exact
        # ---- row-parallel fp8 linear: quantise the K-shard per token on this rank, GEMM,
        #      then ONE sum all-reduce (linear.py:1385-1389) ----
        g = torch.Generator().manual_seed(7)
        M, K, N = 5, 256, 48
        x = torch.randn((M, K), generator=g).to(torch.bfloat16)
        w = torch.randn((N, K), generator=g).to(torch.bfloat16)
        ka, kb = shard_range(K, world, rank)
        xq, xs = O.scaled_fp8_quant(x[:, ka:kb].contiguous(), use_per_token_if_dynamic=True)
        wq, ws = O.scaled_fp8_quant(w[:, ka:kb].contiguous(), use_per_token_if_dynamic=True)
        part = O.scaled_mm(xq, wq.t(), xs, ws, torch.bfloat16).float()
        total = tensor_model_parallel_all_reduce(part, dist)
        ref = x.float() @ w.float().t()
        err = (total - ref).abs().max().item() / ref.abs().max().item()
        if rank == 0:
            q.put((ok_attn, err, part.data_ptr() != total.data_ptr()))
    finally:
        dist.destroy_process_group()


def test_tp2_gloo_sharded_attention_and_row_parallel():
    ctx = mp.get_context("spawn")
    q = ctx.Queue()
    port = _free_port()
    procs = [ctx.Process(target=_tp_worker, args=(r, 2, port, q)) for r in range(2)]
    for p in procs:
        p.start()
    ok_attn, err, out_of_place = q.get(timeout=120)
    for p in procs:
        p.join(timeout=60)
        assert p.exitcode == 0
    assert ok_attn, "KV-head-sharded attention must equal the unsharded result exactly"
    assert err < 0.06, err            # two fp8 quantisations (~2^-4 relative each, averaged over K)
    assert out_of_place


def test_v1_backend_host_logic():
    """TritonAttentionBackend / MetadataBuilder / Impl constructor: the reference's contract
    (vllm/v1/attention/backends/triton_attn.py:58-265) without a GPU."""
    import types
    from vllm_amd.v1.attention.backends import (TritonAttentionBackend, TritonAttentionImpl,
                                                TritonAttentionMetadata,
                                                TritonAttentionMetadataBuilder)
    B = TritonAttentionBackend
    assert B.get_name() == "TRITON_ATTN_VLLM_V1" and B.accept_output_buffer
    assert B.get_impl_cls() is TritonAttentionImpl and B.get_metadata_cls() is TritonAttentionMetadata
    assert B.get_builder_cls() is TritonAttentionMetadataBuilder
    assert B.get_kv_cache_shape(10, 16, 8, 128) == (2, 10, 16, 8, 128)
    with pytest.raises(ValueError, match="multiple of 16"):
        B.get_kv_cache_shape(10, 8, 8, 128)
    assert B.use_cascade_attention() is False
    assert B.get_kv_cache_stride_order() == (0, 1, 3, 2, 4)   # head-major memory by default
    assert torch.bfloat16 in B.get_supported_dtypes() and 128 in B.get_supported_head_sizes()
    assert B.get_supported_head_sizes() == [32, 64, 96, 128, 160, 192, 224, 256]   # triton_attn.py:147-148
    with pytest.raises(ValueError, match="Head size 80 is not supported by TritonAttention"):
        B.validate_head_size(80)

    common = types.SimpleNamespace(
        num_actual_tokens=7, max_query_len=5, query_start_loc=torch.tensor([0, 5, 6, 7], dtype=torch.int32),
        seq_lens=torch.tensor([9, 30, 2], dtype=torch.int32), seq_lens_cpu=torch.tensor([9, 30, 2], dtype=torch.int32),
        block_table_tensor=torch.zeros((3, 2), dtype=torch.int32), slot_mapping=torch.arange(7))
    cfg = types.SimpleNamespace(
        model_config=types.SimpleNamespace(get_num_attention_heads=lambda pc: 32 // pc.tp,
                                           get_num_kv_heads=lambda pc: 8 // pc.tp, get_head_size=lambda: 128),
        parallel_config=types.SimpleNamespace(tp=2))
    b = TritonAttentionMetadataBuilder(types.SimpleNamespace(block_size=16), cfg, torch.device("cpu"))
    assert b.block_size == 16
    md = b.build(0, common)
    assert (md.num_actual_tokens, md.max_query_len, md.max_seq_len) == (7, 5, 30)
    assert md.use_cascade is False and md.cu_prefix_query_lens is None and md.suffix_kv_lens is None
    assert md.block_table is common.block_table_tensor and md.slot_mapping is common.slot_mapping
    md = b.build(4, common)   # a common prefix is flagged (the impl rejects cascade); no cascade tensors
    assert md.use_cascade and md.common_prefix_len == 4 and md.prefix_kv_lens is None
    md = b.build_for_cudagraph_capture(common)
    assert md.seq_lens.tolist() == [1, 1, 1] and b.can_run_in_cudagraph(common)

    impl = TritonAttentionImpl(32, 128, 0.25, 8, [0.5] * 32, 1024, "fp8", 30.0)
    assert impl.sliding_window == (1023, 0) and impl.logits_soft_cap == 30.0 and impl.num_queries_per_kv == 4
    assert impl.alibi_slopes.dtype == torch.float32 and impl.fp8_dtype == torch.float8_e4m3fn
    impl = TritonAttentionImpl(32, 64, 0.25, 8, None, None, "auto")
    assert impl.sliding_window == (-1, -1) and impl.logits_soft_cap == 0 and impl.alibi_slopes is None
    assert impl.fused_output_quant_supported(torch.float8_e4m3fn, True, (-1, -1))


def test_bench_self_launch_two_ranks_gloo():
    """`python bench.py --gpus 2` with no launcher spawns its own ranks (127.0.0.1 rendezvous) and
    fails loudly when the world does not match: rehearsed on the CPU with gloo."""
    import json
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    env = {k: v for k, v in os.environ.items() if k not in ("WORLD_SIZE", "RANK", "LOCAL_RANK")}
    r = subprocess.run([sys.executable, os.path.join(root, "bench.py"), "--gpus", "2",
                        "--dry-run-backend", "gloo"], env=env, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-2000:]
    line = json.loads([l for l in r.stdout.splitlines() if l.startswith("{")][-1])
    assert line["n_gpus"] == 2 and line["sum"] == 2.0
    env2 = dict(env, WORLD_SIZE="2", RANK="0")
    r = subprocess.run([sys.executable, os.path.join(root, "bench.py"), "--gpus", "4",
                        "--dry-run-backend", "gloo"], env=env2, capture_output=True, text=True, timeout=60)
    assert r.returncode == 2 and "WORLD_SIZE=2" in r.stderr


def test_plugin_entry_point_metadata(tmp_path):
    """setup.py declares the `vllm.general_plugins` entry point the reference's plugin
    loader scans (vllm/plugins/__init__.py:19-81; packaging pattern of
    tests/plugins/vllm_add_dummy_platform/setup.py): build the metadata, discover the entry
    point through importlib.metadata as vLLM does, load and call it."""
    import importlib.metadata as md
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "setup.py", "-q", "egg_info", "--egg-base", str(tmp_path)],
                       cwd=root, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    dists = list(md.distributions(path=[str(tmp_path)]))
    assert len(dists) == 1 and dists[0].metadata["Name"] in ("vllm_amd", "vllm-amd")
    eps = [e for e in dists[0].entry_points if e.group == "vllm.general_plugins"]
    assert [e.name for e in eps] == ["vllm_amd"] and eps[0].value == "vllm_amd.plugin:register"
    register = eps[0].load()
    register()     # imports the op layer: the schemas are registered under the reference's names
    import torch
    for ns, op in (("_C", "paged_attention_v1"), ("_C", "cutlass_scaled_mm"),
                   ("_C_cache_ops", "reshape_and_cache"), ("_rocm_C", "paged_attention")):
        assert hasattr(getattr(torch.ops, ns), op)


def test_block_table_host_inputs_match_reference_arithmetic():
    """BlockTable.compute_slot_mapping with the numpy inputs the reference's model runner passes
    (block_table.py:84-99): host path, slot_mapping_np / slot_mapping_cpu filled, no device op."""
    import numpy as np
    from vllm_amd.worker import BlockTable
    bt = BlockTable(16, 4, 8, 64, False, torch.device("cpu"))
    bt.add_row([5, 9, 2], 0)
    bt.add_row([7, 1], 2)
    req = np.array([0, 0, 0, 2, 2], dtype=np.int32)
    pos = np.array([0, 17, 40, 3, 31], dtype=np.int64)
    bt.compute_slot_mapping(req, pos)
    want = np.array([5 * 16, 9 * 16 + 1, 2 * 16 + 8, 7 * 16 + 3, 1 * 16 + 15])
    assert (bt.slot_mapping_np[:5] == want).all() and (bt.slot_mapping_cpu[:5].numpy() == want).all()
    bt.commit_slot_mapping(5)
    assert (bt.slot_mapping[:5].numpy() == want).all()


def test_fp8_linear_static_zero_dim_scale_is_not_sliced(monkeypatch):
    """Static activation quantisation hands a 0-dim input_scale through (w8a8_utils.py:370-377);
    slicing it would raise IndexError."""
    from vllm_amd import quantization as Q
    seen = {}

    def fake_mm(a, b, sa, sb, out_dtype, bias=None):
        seen["sa"] = sa
        return torch.zeros((a.shape[0], b.shape[1]), dtype=out_dtype)

    monkeypatch.setattr(Q.ops, "cutlass_scaled_mm", fake_mm)
    op = Q.Fp8LinearOp(act_quant_static=True)
    monkeypatch.setattr(op, "quant_fp8", lambda x, s, ub: (x.to(torch.float8_e4m3fn), s))
    scale = torch.tensor(0.5)          # 0-dim, as Parameter(input_scale.max())
    out = op.apply(torch.zeros((3, 32), dtype=torch.bfloat16), torch.zeros((32, 16), dtype=torch.float8_e4m3fn),
                   torch.ones(16, 1), input_scale=scale)
    assert out.shape == (3, 16) and seen["sa"] is scale


def test_prefill_key_segments_plan():
    """What the prefill launches answer about their split (host arithmetic): long contexts of few tokens are cut, many rows over
    few keys, fresh prompts and decode-like calls are not, and the scratch of a mixed batch is bounded."""
    from vllm_amd._lib import lib
    uni, ctx = lib.vllm_amd_unified_attention_segments, lib.vllm_amd_context_attention_fwd_segments
    assert uni(1, 32, 8, 128, 512, 8000, 512, 0) > 1 and ctx(1, 32, 8, 128, 512, 8000, 512, 0, 0, 0) > 1
    assert uni(1, 64, 8, 128, 512, 1024, 512, 0) == 1 and ctx(1, 64, 8, 128, 512, 1024, 512, 0, 0, 0) == 1
    assert uni(1, 32, 8, 128, 300, 300, 300, 0) == 1 and uni(1, 32, 8, 128, 512, 8000, 512, 1) == 1
    assert ctx(1, 32, 8, 128, 512, 8000, 512, 0, 128, 0) == 1
    for tokens, heads, d in ((2064, 32, 128), (4096, 64, 256), (600, 8, 64), (64, 32, 128)):
        for n in (uni(tokens - 63, heads, 8, d, 64, 131072, tokens, 0), ctx(tokens - 63, heads, 8, d, 64, 131072, tokens, 0, 0, 1)):
            assert 1 <= n <= 32 and (n == 1 or tokens * heads * n * (d + 2) * 4 <= 256 << 20)
    assert uni(2001, 32, 8, 128, 64, 131072, 2064, 0) > 1
