"""GPU parity of the HIP paged-attention kernels (through the C-ABI) against the CPU oracle
(float64 restatement of nanoserve/kernels/paged_attention_triton.py:19-131). Tolerance per output
element: half an ulp of the output type (none for float32) + K * u * cond, cond = S * dev + Vabs the
oracle's condition term (the largest |q|.|k| score scale times the weighted spread of the values,
plus the weighted |v|), u = 2^-24 for float32 and 2^-16 for the 16-bit types, K = 8 resp. 0.25
(tests/pa_cases.py)."""
import numpy as np
import pytest
import torch

from conftest import pkg
from pa_cases import ARITH_K, UNIT, assert_close_to_oracle, make_case, oracle_args, to_device
from oracle import paged_attention_oracle as PA

pytestmark = pytest.mark.gpu
A = pkg("paged_attention")


def run(case, device, **kw):
    c = to_device(case, device)
    print(f"paged attention: q {tuple(case['query'].shape)} {case['query'].dtype} seqs {case['seq_lens'].tolist()} "
          f"q_lens {case['query_lens'].tolist()}", flush=True)
    out = A.paged_attention_hip(c["query"], c["k_cache"], c["v_cache"], c["block_tables"], c["seq_lens"],
                                c["query_start_loc"], c["query_lens"], c["scale"], c["block_size"], **kw)
    torch.cuda.synchronize()
    return out


def check(case, device, **kw):
    out = run(case, device, **kw)
    ref = PA.paged_attention(**oracle_args(case), terms=True)
    assert_close_to_oracle(out, ref, case["query"].dtype)
    return out


def test_decode_llama32_3b_split_partitions(device):
    # 8 decode rows, lengths around block edges and long enough to be split and merged
    case = make_case(10, [1, 15, 16, 17, 100, 513, 1500, 4000], [1] * 8)
    check(case, device)


def test_decode_batch_64_ctx_2048(device):
    # the benchmark's shape: 64 decode rows of 2048 positions, Llama-3.2-3B heads, bf16
    case = make_case(11, [2048] * 64, [1] * 64, spare_blocks=0, spare_cols=0)
    check(case, device)


def test_chunked_prefill_mix(device):
    # full prefill (causal), decode, chunked prefill, an empty sequence, a short full prefill
    case = make_case(12, [37, 64, 300, 20, 9], [37, 1, 45, 0, 9])
    check(case, device)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("hq,hkv,d", [(8, 8, 128), (16, 8, 64), (32, 8, 128), (32, 4, 64), (24, 8, 64), (64, 8, 128)])
def test_head_layouts_and_dtypes(device, dtype, hq, hkv, d):
    case = make_case(13 + hq + d, [70, 1, 260, 33], [1, 1, 30, 33], hq=hq, hkv=hkv, d=d, block_size=16,
                     dtype=dtype)
    check(case, device)


@pytest.mark.parametrize("block_size", [1, 7, 8, 12, 32])
def test_block_sizes(device, block_size):
    case = make_case(20 + block_size, [45, 130, 7], [1, 3, 7], block_size=block_size)
    check(case, device)


def test_strided_query_view_of_fused_qkv(device):
    # query as the view into the fused QKV output that Attention.forward passes
    case = make_case(30, [50, 200], [50, 1], qkv_view=True)
    assert not case["query"].is_contiguous()
    check(case, device)


def test_zero_visible_keys_gives_zeros(device):
    # a sequence of length 0 holding one query token (malformed batch): the reference's l == 0 guard
    case = make_case(31, [0, 20], [1, 1])
    out = check(case, device)
    assert torch.count_nonzero(out[0].float()).item() == 0


def test_long_rows_through_merge_and_repeat_bit_exact(device):
    case = make_case(32, [8192, 3], [1, 1], hq=32, hkv=8, d=128)
    a = check(case, device)
    b = run(case, device)
    assert torch.equal(a, b)


def test_status_flags_bad_block_and_short_max_seq_len(device):
    case = make_case(33, [40, 40], [1, 1])
    nb = case["k_cache"].shape[0]
    bad = {k: (v.clone() if isinstance(v, torch.Tensor) else v) for k, v in case.items()}
    bad["block_tables"][0, 1] = nb + 7  # out of the cache: the kernel skips those keys and flags it
    status = torch.zeros(1, dtype=torch.int32, device=device)
    out = run(bad, device, status=status)
    assert status.item() & A.STATUS_BAD_BLOCK
    ref, cond = PA.paged_attention(**oracle_args(case), terms=True)
    # the other sequence is untouched by the bad entry
    assert_close_to_oracle(out[1:], (ref[1:], cond[1:]), case["query"].dtype)
    status.zero_()
    run(case, device, status=status)
    assert status.item() == 0
    # a max_seq_len below a sequence's length: flagged when the grid cannot cover that sequence
    # (400 positions need 7 partitions of 64, the grid sized for 16 positions holds one)
    long_case = make_case(36, [400, 40], [1, 1])
    run(long_case, device, status=status, max_seq_len=16)
    assert status.item() & A.STATUS_SEQ_TOO_LONG


def test_empty_batch_and_argument_errors(device):
    case = make_case(34, [5], [0])
    out = run(case, device)
    assert out.shape[0] == 0
    c = to_device(make_case(35, [5], [1]), device)
    with pytest.raises(A.PagedAttentionError, match="block_size"):
        A.paged_attention_hip(c["query"], c["k_cache"], c["v_cache"], c["block_tables"], c["seq_lens"],
                              c["query_start_loc"], c["query_lens"], c["scale"], 8)


def test_split_rows_leave_the_counters_at_zero(device):
    # split rows are merged by their last partition's workgroup through arrival counters; each call
    # must leave them at zero, so repeated calls of different shapes on one counters buffer (and a
    # reused workspace holding an earlier call's partials) stay exact
    counters = torch.zeros(4096, dtype=torch.int32, device=device)
    ws = torch.full((32 << 20,), 0x7F, dtype=torch.uint8, device=device)  # largest need: 15.9 MB
    for seed, lens in ((37, [3000, 700, 5000]), (38, [64] * 70 + [9000]), (39, [2500] * 3)):
        case = make_case(seed, lens, [1] * len(lens))
        q = case["query"]
        assert A.workspace_bytes(q.shape[0], q.shape[1], case["k_cache"].shape[2], q.shape[2], max(lens)) > 0
        ref = PA.paged_attention(**oracle_args(case), terms=True)
        outs = []
        for _ in range(2):
            out = run(case, device, workspace=ws, counters=counters)
            assert_close_to_oracle(out, ref, q.dtype)
            outs.append(out)
        assert torch.equal(outs[0], outs[1])
        assert torch.count_nonzero(counters).item() == 0


def test_more_partitions_than_the_lds_weight_table(device):
    # one KV head and one long row: 1094 partitions of 64 positions, more than the merging
    # workgroup's LDS weight table (1024 entries) holds, so the one-pass rescaled merge runs
    case = make_case(40, [70000], [1], hq=8, hkv=1, d=128)
    assert A.workspace_bytes(1, 8, 1, 128, 70000) == 1 * 8 * 1094 * (128 + 2) * 4
    check(case, device)


@pytest.mark.parametrize("ctx,parts", [(16384, 256), (16385, 257), (40000, 625), (65536, 1024), (65600, 1025)])
@pytest.mark.parametrize("hq,d,dtype", [(8, 128, torch.bfloat16), (4, 64, torch.float16)])
def test_one_long_row_of_few_kv_heads(device, ctx, parts, hq, d, dtype):
    # a row of one KV head merges hundreds of partitions: through the LDS weight table up to 1024 of
    # them, whatever the number of heads it is shared by, and past it by the one-pass loop
    case = make_case(900 + parts, [ctx], [1], hq=hq, hkv=1, d=d, dtype=dtype)
    assert A.workspace_bytes(1, hq, 1, d, ctx) == hq * parts * (d + 2) * 4
    a = check(case, device, max_query_len=1)
    assert torch.equal(a, run(case, device, max_query_len=1))


def test_side_stream_and_output_stride(device):
    """A call on a side stream (its temporaries and counters made on that stream) equals the
    call on the current stream bit for bit; an output whose head_dim stride is not 1 is refused
    (the kernel writes out[token, head, d] with a unit stride along d)."""
    case = make_case(21, [1500, 7, 300], [1, 1, 20])
    want = run(case, device)
    side = torch.cuda.Stream(device=device)
    c = to_device(case, device)
    torch.cuda.synchronize()
    got = A.paged_attention_hip(c["query"], c["k_cache"], c["v_cache"], c["block_tables"], c["seq_lens"],
                                c["query_start_loc"], c["query_lens"], c["scale"], c["block_size"], stream=side)
    side.synchronize()
    assert torch.equal(got, want)
    raw = A.paged_attention_hip(c["query"], c["k_cache"], c["v_cache"], c["block_tables"], c["seq_lens"],
                                c["query_start_loc"], c["query_lens"], c["scale"], c["block_size"],
                                stream=side.cuda_stream)
    side.synchronize()
    assert torch.equal(raw, want)
    # a raw handle of 0 is the null stream, torch's default stream: the call is ordered after the
    # default stream's unsynchronized work (the caches written just before it)
    torch.cuda.synchronize()
    with torch.cuda.stream(torch.cuda.default_stream(device)):
        kc, vc = c["k_cache"].clone(), c["v_cache"].clone()
        null = A.paged_attention_hip(c["query"], kc, vc, c["block_tables"], c["seq_lens"], c["query_start_loc"],
                                     c["query_lens"], c["scale"], c["block_size"], stream=0)
    torch.cuda.default_stream(device).synchronize()
    assert torch.equal(null, want)
    q = c["query"]
    bad = torch.empty((q.shape[0], q.shape[1], q.shape[2] * 2), dtype=q.dtype, device=device)[:, :, ::2]
    with pytest.raises(A.PagedAttentionError, match="unit head_dim stride"):
        A.paged_attention_hip(q, c["k_cache"], c["v_cache"], c["block_tables"], c["seq_lens"],
                              c["query_start_loc"], c["query_lens"], c["scale"], c["block_size"], out=bad)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hq,hkv,d", [(24, 8, 128), (32, 8, 128), (8, 8, 64), (16, 8, 64), (64, 8, 128)])
def test_prefill_tiles_head_layouts(device, dtype, hq, hkv, d):
    # sequences of several query tokens go by MFMA query tile (128 // G tokens each): a chunk in the
    # middle of a long sequence, a full prefill, chunks shorter than a tile, and decode rows beside them
    case = make_case(50 + hq + d, [700, 300, 190, 1, 90, 45], [200, 300, 3, 1, 17, 1], hq=hq, hkv=hkv, d=d,
                     dtype=dtype)
    check(case, device)


def test_prefill_chunk_512_over_4096_positions(device):
    # the reference's chunked_prefill_size (config.py:53): a 512-token chunk at the end of a 4096-position
    # sequence, split over KV partitions merged by the last to arrive, and a second chunk of another sequence
    case = make_case(60, [4096, 1500], [512, 512])
    check(case, device)


@pytest.mark.parametrize("block_size", [1, 7, 16, 32])
def test_prefill_tiles_block_sizes(device, block_size):
    case = make_case(70 + block_size, [130, 77], [64, 77], block_size=block_size)
    check(case, device)


@pytest.mark.parametrize("d,block_size", [(128, 2), (128, 4), (128, 12), (128, 128), (64, 4), (64, 8), (64, 24)])
def test_prefill_row_addresses_by_block_size(device, d, block_size):
    # block sizes on both sides of the rule for scalar row addresses (a power of two of at least
    # 512 / d positions), lengths that end inside a block
    case = make_case(71 + block_size + d, [701, 77], [64, 77], d=d, block_size=block_size)
    check(case, device)


def test_prefill_tiles_repeat_bit_exact_and_strided_query(device):
    case = make_case(80, [900, 64], [300, 64], qkv_view=True)
    a = check(case, device)
    b = run(case, device)
    assert torch.equal(a, b)


def test_prefill_bad_tile_is_flagged(device):
    # a tile reaching past its sequence's query tokens is refused by the kernel (status bit), nothing
    # out of bounds is touched, and the other tiles and tokens are exact
    import ctypes

    case = make_case(90, [100, 40], [40, 1])
    c = to_device(case, device)
    q = c["query"]
    out = torch.full_like(q, 7.0)
    tiles = torch.tensor([[0, 0, 21], [0, 21, 19], [0, 30, 21]], dtype=torch.int32, device=device)
    tokens = torch.tensor([40], dtype=torch.int32, device=device)
    status = torch.zeros(1, dtype=torch.int32, device=device)
    lib = A.load()
    bt = c["block_tables"]
    a = A.NsPagedAttnArgs(
        q.data_ptr(), c["k_cache"].data_ptr(), c["v_cache"].data_ptr(), out.data_ptr(), bt.data_ptr(),
        c["seq_lens"].data_ptr(), c["query_start_loc"].data_ptr(), c["query_lens"].data_ptr(), status.data_ptr(),
        None, 0, None, q.stride(0), q.stride(1), c["k_cache"].stride(0), c["k_cache"].stride(1),
        c["k_cache"].stride(2), c["v_cache"].stride(0), c["v_cache"].stride(1), c["v_cache"].stride(2),
        out.stride(0), out.stride(1), bt.stride(0), q.shape[0], 2, 24, 8, 128, 16, c["k_cache"].shape[0], bt.shape[1],
        100, A.NS_PA_DTYPE_BF16, c["scale"])
    a.decode_tokens, a.n_decode_tokens = tokens.data_ptr(), 1
    a.prefill_tiles, a.n_prefill_tiles = tiles.data_ptr(), 3
    nb, nc = ctypes.c_uint64(0), ctypes.c_uint64(0)
    assert lib.ns_paged_attention_call_workspace(ctypes.byref(a), ctypes.byref(nb), ctypes.byref(nc)) == 0
    ws = torch.empty(max(int(nb.value), 1), dtype=torch.uint8, device=device)
    cnt = torch.zeros(max(int(nc.value), 1), dtype=torch.int32, device=device)
    a.workspace, a.workspace_bytes, a.counters = ws.data_ptr(), int(nb.value), cnt.data_ptr()
    assert lib.ns_paged_attention(ctypes.byref(a), None) == 0
    torch.cuda.synchronize()
    assert status.item() & A.STATUS_BAD_TILE
    ref = PA.paged_attention(**oracle_args(case), terms=True)
    assert_close_to_oracle(out, ref, q.dtype)   # the two valid tiles cover tokens 0..39, the list token 40
    assert torch.count_nonzero(cnt).item() == 0


def test_plan_reused_across_layers_and_refused_for_another_layout(device):
    # one host plan per step serves every layer's call (two caches here): same outputs as the
    # calls that plan for themselves, and a plan of another layout is refused
    case = make_case(95, [1200, 333, 64, 9], [400, 333, 1, 1])
    other = make_case(96, [1200, 333, 64, 9], [400, 333, 1, 1])
    c, o = to_device(case, device), to_device(other, device)
    plan = A.PagedAttentionPlan(c["seq_lens"], c["query_start_loc"], c["query_lens"], 24, 8, device)
    assert plan.tiles is not None and plan.tokens[1] == 2
    outs = []
    for x in (c, o):
        args = (x["query"], x["k_cache"], x["v_cache"], x["block_tables"], x["seq_lens"], x["query_start_loc"],
                x["query_lens"], x["scale"], x["block_size"])
        with_plan = A.paged_attention_hip(*args, plan=plan)
        without = A.paged_attention_hip(*args)
        torch.cuda.synchronize()
        assert torch.equal(with_plan, without)
        outs.append(with_plan)
    for case_, out in zip((case, other), outs):
        assert_close_to_oracle(out, PA.paged_attention(**oracle_args(case_), terms=True), torch.bfloat16)
    bad = A.PagedAttentionPlan(c["seq_lens"], c["query_start_loc"], c["query_lens"], 32, 8, device)
    with pytest.raises(A.PagedAttentionError, match="another batch layout"):
        A.paged_attention_hip(c["query"], c["k_cache"], c["v_cache"], c["block_tables"], c["seq_lens"],
                              c["query_start_loc"], c["query_lens"], c["scale"], c["block_size"], plan=bad)


@pytest.mark.parametrize("d", [128, 64])
def test_prefill_tile_merged_from_many_segments(device, d):
    # one tile over 9000 positions is cut between many workgroups, one over 4000 between fewer; the last
    # to arrive merges the segments one after the other
    case = make_case(97 + d, [9000, 4000], [20, 30], d=d)
    check(case, device)


@pytest.mark.parametrize("seqs,qlens,scale,bad", [
    ([3000, 65, 70, 64, 63], [500, 65, 2, 64, 3], 1.0, False),        # tiles cut mid-way, others whole beside them
    ([20000], [2], 1.0, False),                                       # a tile shared by many workgroups
    ([40, 1, 33, 2] * 70, [20, 1, 33, 2] * 70, 1.0, False),           # more tiles than threads, shares of several tiles
    ([1300, 257], [130, 257], -0.5, False),                           # a negative score scale
    ([1300, 257], [130, 257], 0.0, False),                            # and none
    ([1300, 500], [130, 200], 1.0, True),                             # blocks outside the cache in a cut tile
])
def test_prefill_shared_steps(device, seqs, qlens, scale, bad):
    # the steps of all tiles are shared evenly by the workgroups, whatever the tiles' lengths
    case = make_case(len(seqs) + seqs[0], seqs, qlens)
    case["scale"] *= scale
    if bad:
        case["block_tables"][0, 3:9:2] = 10 ** 6
        case["block_tables"][1, 20] = -3
    # an output whose rows are not 8-byte aligned, next to the plain one
    c = to_device(case, device)
    q = c["query"]
    wide = torch.empty((q.shape[0], q.shape[1], q.shape[2] + 1), dtype=q.dtype, device=device)
    a = run(case, device)
    b = run(case, device, out=wide[:, :, 1:])
    assert torch.equal(a, b)
    if bad:   # the per-token kernel skips the same keys
        ref = run(case, device, max_query_len=1).double()
        assert ((a.double() - ref).abs() <= 1e-4 + 2.0 ** -7 * ref.abs()).all()
    else:
        assert_close_to_oracle(a, PA.paged_attention(**oracle_args(case), terms=True), q.dtype)


@pytest.mark.parametrize("d,g,dtype,block_size", [(128, 1, torch.bfloat16, 16), (128, 3, torch.float16, 4),
                                                  (128, 8, torch.bfloat16, 2), (64, 2, torch.float16, 8),
                                                  (64, 4, torch.bfloat16, 7), (64, 8, torch.float16, 4)])
def test_decode_step_edges(device, d, g, dtype, block_size):
    # lengths around a wave's step (16 positions of 128 dims, 32 of 64), the four waves' share and the
    # partitions; block sizes on both sides of the rule for scalar row addresses
    lens = [1, 2, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 255, 257, 1023, 1025, 2500]
    case = make_case(600 + d + g, lens, [1] * len(lens), hq=2 * g, hkv=2, d=d, dtype=dtype, block_size=block_size)
    a = check(case, device, max_query_len=1)
    assert torch.equal(a, run(case, device, max_query_len=1))


@pytest.mark.parametrize("num_seqs", [1, 63, 64, 65, 129, 4097])
def test_decode_token_search(device, num_seqs):
    # the sequence of a query token is found 64 entries at a time; empty sequences share their start
    lens = [1 + (7 * i) % 19 for i in range(num_seqs)]
    qlens = [0 if i % 5 == 3 else 1 for i in range(num_seqs)]
    case = make_case(700 + num_seqs, lens, qlens, hq=2, hkv=1, d=64, block_size=8)
    check(case, device, max_query_len=1)


def test_decode_invalid_blocks_skip_their_keys(device):
    # garbage (NaN) in rows that no sequence holds must not reach the outputs
    case = make_case(800, [300, 40, 2000], [1, 1, 1])
    free = torch.ones(case["k_cache"].shape[0], dtype=torch.bool)
    for s, n in enumerate([300, 40, 2000]):
        free[case["block_tables"][s, :-(-n // 16)].long()] = False
        last = int(case["block_tables"][s, (n - 1) // 16])
        if n % 16:
            case["v_cache"][last, n % 16:] = float("nan")
            case["k_cache"][last, n % 16:] = float("nan")
    case["k_cache"][free] = float("nan")
    case["v_cache"][free] = float("nan")
    out = run(case, device, max_query_len=1)
    clean = {k: (torch.nan_to_num(v) if k.endswith("cache") else v) for k, v in case.items()}
    assert_close_to_oracle(out, PA.paged_attention(**oracle_args(clean), terms=True), case["query"].dtype)
    bad = {k: (v.clone() if isinstance(v, torch.Tensor) else v) for k, v in clean.items()}
    bad["block_tables"][0, 3] = -1
    bad["block_tables"][2, 5:9] = 10 ** 6
    a = run(bad, device, max_query_len=1)
    f32 = {k: (v.float() if isinstance(v, torch.Tensor) and v.is_floating_point() else v) for k, v in bad.items()}
    ref = run(f32, device, max_query_len=1).double()
    assert ((a.double() - ref).abs() <= 1e-4 + 2.0 ** -7 * ref.abs()).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_long_decode_row_beside_cut_tiles(device, dtype):
    # 130 listed tokens of 8 KV heads at max_seq_len 1000 fit one partition each and need no workspace,
    # the tile beside them is cut and does.  A decode row longer than max_seq_len allows is flagged, its
    # output undefined; nothing of it reaches the tile's partials, and all other rows are exact
    seqs, qlens = [990] + [40] * 129 + [1500], [30] + [1] * 130
    case = make_case(810, seqs, qlens, hq=8, hkv=8, d=64, dtype=dtype)
    assert A.workspace_bytes(130, 8, 8, 64, 1000) == 0
    status = torch.zeros(1, dtype=torch.int32, device=device)
    out = run(case, device, max_seq_len=1000, status=status)
    assert status.item() == A.STATUS_SEQ_TOO_LONG
    ref, cond = PA.paged_attention(**oracle_args(case), terms=True)
    assert_close_to_oracle(out[:-1], (ref[:-1], cond[:-1]), dtype)


@pytest.mark.parametrize("g,d,dtype", [(3, 128, torch.bfloat16), (8, 128, torch.float16), (4, 64, torch.bfloat16),
                                       (1, 64, torch.float16), (1, 128, torch.float32)])
def test_decode_values_that_are_not_finite(device, g, d, dtype):
    # infinities, NaN and values near the type's largest in visible rows, in whole and in split rows: each
    # reaches its own output element as in float arithmetic (weight times infinity is infinity), no other
    lens = [1, 40, 300, 700, 2500]
    case = make_case(820 + d + g, lens, [1] * 5, hq=2 * g, hkv=2, d=d, dtype=dtype)
    v, bt = case["v_cache"], case["block_tables"]

    def put(s, t, head, dim, x):
        v[int(bt[s, t // 16]), t % 16, head, dim] = x

    for s, n in enumerate(lens):
        put(s, n - 1, 0, 3, float("inf"))
        put(s, n // 2, 1, 5, float("-inf"))
        put(s, n // 3, 0, 8, float("nan"))
        put(s, n - 1, 1, 11, torch.finfo(dtype).max)   # the largest value, at a weight of at most 1
    for s, n in enumerate(lens[1:], 1):
        put(s, 0, 1, 17, float("inf"))                 # both infinities: NaN
        put(s, n - 2, 1, 17, float("-inf"))
    out = run(case, device, max_query_len=1)
    with np.errstate(invalid="ignore"):   # the condition term of an infinite output is NaN, and not used
        ref, cond = PA.paged_attention(**oracle_args(case), terms=True)
    got, odd = out.double().cpu().numpy(), ~np.isfinite(ref)
    assert odd.any() and np.array_equal(got[odd], ref[odd], equal_nan=True)
    fine = torch.from_numpy(np.where(odd, 0.0, got))
    assert_close_to_oracle(fine, (np.where(odd, 0.0, ref), np.where(odd, 0.0, cond)), dtype)


def sink_case(seed, seq_lens, query_lens, below, sinks, hq, hkv, d, dtype):
    """Keys of the positions ``sinks`` outweigh all others by about 2 ** below and their values are 0 (an
    attention sink), so that an output is the sum of the others' small weights; their values are about 256."""
    case = make_case(seed, seq_lens, query_lens, hq=hq, hkv=hkv, d=d, dtype=dtype)
    rng = torch.Generator().manual_seed(seed)
    k, v, bt = case["k_cache"], case["v_cache"], case["block_tables"]
    case["query"].fill_(1.0)
    k.copy_(torch.randn(k.shape, generator=rng) * 0.3)
    v.copy_((torch.rand(v.shape, generator=rng) + 0.5) * 256)
    for s, n in enumerate(seq_lens):
        for t in sinks:
            if t < n:
                k[int(bt[s, t // 16]), t % 16] = below * np.log(2.0) / np.sqrt(d)
                v[int(bt[s, t // 16]), t % 16] = 0.0
    return case


@pytest.mark.parametrize("below", [10, 18, 22, 24.5, 27, 31, 35])
@pytest.mark.parametrize("d,dtype", [(64, torch.float16), (128, torch.float16), (128, torch.bfloat16)])
def test_decode_small_weights_beside_large_ones(device, below, d, dtype):
    # in whole rows (partitions of 1024 positions) every wave has a sink, in split ones the first has
    lens = [1024, 700, 64, 17] * 32
    check(sink_case(830, lens, [1] * 128, below, (0, 16, 32, 48, 64, 96), 8, 8, d, dtype), device, max_query_len=1)
    check(sink_case(831, [3000, 200], [1, 1], below, (0,), 6, 2, d, dtype), device, max_query_len=1)


@pytest.mark.parametrize("below", [10, 18, 22, 24.5, 27, 31])
@pytest.mark.parametrize("d,dtype", [(64, torch.float16), (128, torch.float16), (128, torch.bfloat16)])
def test_prefill_small_weights_beside_large_ones(device, below, d, dtype):
    # a sink at the start of sequences whose tiles are cut and whole.  Beside the usual bound, float16's
    # parts of a weight end 2^-38 below the largest (absolute error of each)
    case = sink_case(840, [5000, 700, 300, 60], [40, 32, 90, 60], below, (0,), 8, 2, d, dtype)
    ref, cond = PA.paged_attention(**oracle_args(case), terms=True)
    if dtype == torch.float16:
        places = PA.query_places(case["seq_lens"], case["query_start_loc"], case["query_lens"])
        n = np.array([kv_len for _, kv_len, _ in places], dtype=np.float64)[:, None, None]
        cond = cond + n * 2.0 ** -38 * 384 / (ARITH_K[dtype] * UNIT[dtype])   # 384: the values' largest
    assert_close_to_oracle(run(case, device), (ref, cond), dtype)
