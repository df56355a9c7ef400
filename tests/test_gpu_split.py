"""GPU parity of the split decode (pa_fp8_decode_split: every (sequence, kv
head) over up to S workgroups, merged by the last one) and of the team decode
(pa_fp8_decode_team: equal runs of the batch per workgroup).  Edges of its ranges:
contexts around a chunk, a share and a split, empty sequences, 1 to 16 query
columns, both kernels' wave counts, windows, the flat page list with sequences
that have no pages; and of the workspaces that the launchers give them."""

from __future__ import annotations

import ctypes

import pytest
import torch

import flydsl_amd.pa_decode as pd
from flydsl_amd import _lib, pa_decode_ps_launch
from tests._cases import make_case, torch_oracle
from tests.test_gpu_parity import assert_parity, to_dev

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

EDGES = [0, 1, 31, 32, 33, 511, 512, 513, 1024, 1025, 5000]
SHAPES = {
    "gqa1_edges": dict(batch=len(EDGES), num_query_heads=3, num_kv_heads=3, ctx=EDGES),
    "gqa4_pt": dict(batch=4, num_query_heads=8, num_kv_heads=2, ctx=[1, 700, 2049, 8191], per_token=True),
    "gqa5_page64": dict(batch=3, num_query_heads=10, num_kv_heads=2, block_size=64, ctx=[64, 65, 3000]),
    "ql2_gqa8_pt": dict(batch=3, query_length=2, num_query_heads=16, num_kv_heads=2, ctx=[2, 517, 4100], per_token=True),
    "ql3_gqa5": dict(batch=3, query_length=3, num_query_heads=5, num_kv_heads=1, ctx=[3, 96, 2600]),
    "window": dict(batch=4, ctx=[5, 300, 1500, 6000], sliding_window=1000),
    "pairs_beyond_cus": dict(batch=140, num_query_heads=8, num_kv_heads=2, ctx_range=(1, 1100)),
}


def split(case, S, out_dtype=torch.bfloat16, team=False):
    out = torch.empty(case["query"].shape, dtype=out_dtype, device=DEV)
    a = pd._stream_args(out, case["query"], case["key_cache"], case["value_cache"], case["context_lengths"],
                        case["block_tables"], None, case["softmax_scale"], case["key_scale"], case["value_scale"],
                        case["key_scale"].dim() > 1, True, "bf16", pd._get_output_dtype_code(out),
                        case["sliding_window"])
    a.num_workers = S
    pairs = case["key_cache"].shape[1] * case["context_lengths"].shape[0]
    # slots full of NaN: a merge that reads one its launch did not write shows
    slots = torch.full((max(16, pairs * S * 8704),), 0xFF, dtype=torch.uint8, device=DEV)
    counters = torch.zeros(pairs, dtype=torch.int32, device=DEV)
    if team:
        slots = torch.full((_lib.team_slot_bytes(S),), 0xFF, dtype=torch.uint8, device=DEV)
    else:
        assert _lib.split_slot_bytes(case["context_lengths"].shape[0], case["key_cache"].shape[1], S) <= slots.numel()
    entry = _lib.load().pa_fp8_decode_team if team else _lib.load().pa_fp8_decode_split
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    outs = []
    for _ in range(2):
        _lib.check(entry(ctypes.byref(a), slots.data_ptr(), slots.numel(), counters.data_ptr(), counters.numel(), s),
                   "split")
        torch.cuda.synchronize()
        assert int(counters.abs().sum()) == 0
        outs.append(out.clone())
    assert torch.equal(outs[0], outs[1])
    return outs[0]


@pytest.mark.parametrize("S", [1, 2, 3, 8, 33])
@pytest.mark.parametrize("name", sorted(SHAPES))
def test_split_matches_oracle(name, S):
    case = make_case(seed=len(name) + S, **SHAPES[name])
    ctx = case["context_lengths"]
    ref = torch_oracle(dict(case, context_lengths=ctx.clamp(min=1)), float_out=False)
    for b in torch.nonzero(ctx == 0).flatten().tolist():
        ref[b] = 0
    assert_parity(split(to_dev(case), S, torch.float32 if S == 3 else torch.bfloat16), ref, f"{name}/S={S}")


@pytest.mark.parametrize("workgroups", [1, 5, 64, 256])
@pytest.mark.parametrize("name", sorted(set(SHAPES) - {"window"}))
def test_team_matches_oracle(name, workgroups):
    case = make_case(seed=len(name) + workgroups, **SHAPES[name])
    ctx = case["context_lengths"]
    ref = torch_oracle(dict(case, context_lengths=ctx.clamp(min=1)), float_out=False)
    for b in torch.nonzero(ctx == 0).flatten().tolist():
        ref[b] = 0
    assert_parity(split(to_dev(case), workgroups, torch.float16 if workgroups == 5 else torch.bfloat16, team=True), ref,
                  f"{name}/{workgroups}")


def test_launcher_shares_one_workspace_per_stream():
    """Calls on a stream reuse its workspace, calls on two unordered streams
    do not share one, and a prepared call has its own."""
    case = to_dev(make_case(batch=2, ctx=[3000, 9000], num_query_heads=16, seed=5))
    ref = torch_oracle({k: (v.cpu() if isinstance(v, torch.Tensor) else v) for k, v in case.items()}, float_out=False)
    args = (case["query"], case["key_cache"], case["value_cache"], case["context_lengths"], None, None,
            case["softmax_scale"], case["key_scale"], case["value_scale"])
    streams = [torch.cuda.Stream() for _ in range(2)]
    outs = [torch.empty_like(case["query"]) for _ in range(8)]
    torch.cuda.synchronize()
    for i, out in enumerate(outs):
        pa_decode_ps_launch(out, *args, block_tables=case["block_tables"], stream=streams[i % 2])
    torch.cuda.synchronize()
    for out in outs:
        assert_parity(out, ref, "two streams")
    spaces = [pd._split_workspace(0, s, 4, 16, True) for s in streams]
    assert spaces[0] is not spaces[1]
    assert spaces[0] is pd._split_workspace(0, streams[0], 4, 16, True)
    assert pd._split_workspace(0, streams[0], 4, 16, False) is not spaces[0]
    assert len(pd._workspaces) <= pd._WORKSPACES_KEPT


def launcher(case, S, team, counters, pages=None, indptr=None):
    """launch(out, stream) of one call with a workspace of its own (``pages``,
    ``indptr``: a flat page list in the place of the block table)."""
    a = pd._stream_args(case["query"], case["query"], case["key_cache"], case["value_cache"], case["context_lengths"],
                        case["block_tables"] if pages is None else pages, indptr, case["softmax_scale"],
                        case["key_scale"], case["value_scale"], case["key_scale"].dim() > 1, True, "bf16",
                        _lib.DTYPE_BF16, case["sliding_window"])
    a.num_workers = S
    nbytes = _lib.team_slot_bytes(S) if team else _lib.split_slot_bytes(a.num_seqs, a.num_kv_heads, S)
    slots = torch.full((max(16, nbytes),), 0xFF, dtype=torch.uint8, device=DEV)
    entry = _lib.load().pa_fp8_decode_team if team else _lib.load().pa_fp8_decode_split

    def launch(out, stream):
        a.output = out.data_ptr()
        _lib.check(entry(ctypes.byref(a), slots.data_ptr(), slots.numel(), counters.data_ptr(), counters.numel(),
                         ctypes.c_void_p(stream.cuda_stream)), "decode")
    return launch


@pytest.mark.parametrize("kernel,workers", [("split", 1), ("split", 8), ("team", 5), ("team", 256)])
@pytest.mark.parametrize("block_size,per_token", [(16, True), (128, False), (1024, True)])
def test_flat_page_list(kernel, workers, block_size, per_token):
    """Pages of all sequences end to end, two sequences without any (one of
    them with a length all the same): those rows are zero."""
    ctx = [700, 0, 3000, 1, 500, 6000, 33]
    case = make_case(batch=7, num_query_heads=24, num_kv_heads=2, block_size=block_size, ctx=ctx, per_token=per_token,
                     seed=workers)
    ref = torch_oracle(dict(case, context_lengths=case["context_lengths"].clamp(min=1)), float_out=False)
    none = (1, 4)
    for b in none:
        ref[b] = 0
    case = to_dev(case)
    rows = [case["block_tables"][b, : 0 if b in none else -(-c // block_size)] for b, c in enumerate(ctx)]
    pages = torch.cat(rows)
    indptr = torch.tensor([0] + [len(r) for r in rows]).cumsum(0).to(torch.int32).to(DEV)
    counters = torch.zeros(14, dtype=torch.int32, device=DEV)
    out = torch.empty_like(case["query"])
    launcher(case, workers, kernel == "team", counters, pages, indptr)(out, torch.cuda.current_stream())
    assert bool((counters == 0).all())
    assert_parity(out, ref, f"{kernel}/{workers}/{block_size}")


@pytest.mark.parametrize("workgroups", [1, 5, 64, 256])
@pytest.mark.parametrize("ql", [1, 2])
def test_team_window(ql, workgroups):
    case = make_case(batch=7, query_length=ql, num_query_heads=16, num_kv_heads=2, ctx=[5, 300, 1500, 6000, 1001, 2033, 64],
                     sliding_window=1000, seed=workgroups)
    ref = torch_oracle(case, float_out=False)
    assert_parity(split(to_dev(case), workgroups, team=True), ref, f"window/{ql}/{workgroups}")


@pytest.mark.parametrize("gqa", [4, 16])
def test_native_workspaces_of_overlapping_streams(gqa):
    """Calls on the current stream of two unordered streams, and on a stream
    that torch does not own, by the native path (no ``stream``)."""
    case = to_dev(make_case(batch=2, ctx=[3000, 9000], num_query_heads=2 * gqa, seed=5))
    ref = torch_oracle({k: (v.cpu() if isinstance(v, torch.Tensor) else v) for k, v in case.items()}, float_out=False)
    args = (case["query"], case["key_cache"], case["value_cache"], case["context_lengths"], None, None,
            case["softmax_scale"], case["key_scale"], case["value_scale"])
    own = torch.cuda.Stream()
    streams = [torch.cuda.Stream(), torch.cuda.Stream(), torch.cuda.ExternalStream(own.cuda_stream)]
    outs = [torch.empty_like(case["query"]) for _ in range(30)]
    torch.cuda.synchronize()
    for i, out in enumerate(outs):
        with torch.cuda.stream(streams[i % 3]):
            pa_decode_ps_launch(out, *args, block_tables=case["block_tables"])
    torch.cuda.synchronize()
    for out in outs:
        assert torch.equal(out, outs[0])
    assert_parity(outs[0], ref, "three streams")
    kept = [pd._workspaces[0, s.stream_id] for s in streams[:2]]
    assert kept[0] is not kept[1] and (0, streams[2].stream_id) not in pd._workspaces
    assert all(int(w.counters.abs().sum()) == 0 for w in kept)


@pytest.mark.parametrize("name", ["split", "team"])
def test_prepared_calls_replay_from_a_graph(name):
    """A prepared call's launches, captured: every replay gives the eager
    call's bits, with eager decodes on the stream in between."""
    shape = {"split": dict(batch=2, ctx=[3000, 9000], num_query_heads=16),
             "team": dict(batch=150, num_query_heads=64, num_kv_heads=8, ctx=[20000] + [30] * 149)}[name]
    case = to_dev(make_case(seed=6, **shape))
    args = (case["query"], case["key_cache"], case["value_cache"], case["context_lengths"], None, None,
            case["softmax_scale"], case["key_scale"], case["value_scale"])
    out, eager = torch.empty_like(case["query"]), torch.empty_like(case["query"])
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    call = pd.prepare_pa_decode(out, *args, block_tables=case["block_tables"], stream=s)
    assert [n for n, _ in call.kernels()] == [f"pa_fp8_decode_{name}"]
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=s):
        call.launch()
        call.launch()
    for _ in range(4):
        out.zero_()
        graph.replay()
        pa_decode_ps_launch(eager, *args, block_tables=case["block_tables"])
        torch.cuda.synchronize()
        assert torch.equal(out, eager)


RAGGED = dict(batch=6, num_query_heads=16, num_kv_heads=2, ctx=[9000, 17, 3000, 0, 700, 5000])


@pytest.mark.parametrize("team", [False, True])
def test_overlapping_launches_leave_the_workspace_sound(team):
    """Launches of one workspace that overlap may be wrong; one after them is
    right and finds every counter zero."""
    case = to_dev(make_case(seed=8, **RAGGED))
    counters = torch.zeros(12, dtype=torch.int32, device=DEV)
    launch = launcher(case, 64 if team else 8, team, counters)
    want = torch.empty_like(case["query"])
    launch(want, torch.cuda.current_stream())
    streams = [torch.cuda.Stream() for _ in range(2)]
    outs = [torch.empty_like(want) for _ in range(2)]
    torch.cuda.synchronize()
    for _ in range(50):
        for out, s in zip(outs, streams):
            launch(out, s)
    torch.cuda.synchronize()
    assert bool((counters == 0).all())
    launch(outs[0], torch.cuda.current_stream())
    assert torch.equal(outs[0], want)


def test_split_counts():
    assert pd._split_count(8, 2, 256) == 1 and pd._split_count(8, 16, 256) == 1  # short: one workgroup per pair
    assert pd._split_count(8, 256, 256) == 16 and pd._split_count(128, 256, 256) == 2
    assert pd._split_count(512, 128, 256) == 1 and pd._split_count(56, 824, 256) == 4
    assert pd._split_count(32, 4096, 256) == 8  # one round of workgroups
    # uneven pairs that are large parts of a CU's work: equal runs, unless few
    assert pd._split_count(212, 312, 256) == 0 and pd._split_count(200, 256, 256) == 0
    assert pd._split_count(200, 256, 256, True) == 1 and pd._split_count(200, 128, 256) == 1
    assert pd._split_count(64, 975, 256) == 4
    assert pd._split_count(1024, 1024, 256) == 0  # many long pairs: equal runs over the batch
    # where the longest sequence's share would set the time: both sides of the lines
    for pairs, chunks, columns, s in ((96, 256, 4, 2), (96, 257, 4, 0), (64, 1024, 4, 4), (64, 1025, 4, 0), (33, 3136, 4, 7),
                                      (33, 3137, 4, 0), (136, 96, 4, 1), (136, 97, 4, 0), (160, 128, 4, 1),
                                      (256, 129, 4, 0), (257, 64, 4, 1), (257, 65, 4, 0), (448, 128, 4, 1),
                                      (136, 128, 5, 1), (272, 129, 16, 0), (96, 320, 16, 2), (96, 321, 16, 0),
                                      (64, 4096, 16, 4), (64, 4097, 16, 0), (1, 16384, 4, 64)):
        assert pd._split_count(pairs, chunks, 256, False, columns) == s, (pairs, chunks, columns)
    # a flat page list gives the batch's total: its mean counts
    plan = lambda tokens: pd._plan("flat", 64, 2, 0, 8, 128, 128, None, tokens, False, False, False, True, False, 0)
    assert plan(64 * 512)[0] == "split" and plan(64 * 8192)[0] == "team"
