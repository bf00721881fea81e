"""A decode step captured once as a HIP graph and replayed: the append of one row per sequence, the
whole-context attention (decode kernel + merge launch) and the selected-token attention in halved
whole-selection units (whose workgroups meet on the library's counters). Every replay runs on new
inputs written into the captured buffers, with eager work and a device synchronisation between
replays, and is compared with the same calls made eagerly: bit for bit, since every kernel here is
deterministic. The library's entry points only enqueue kernels, so nothing else may appear in the
graph (no memset nodes, no copies)."""
import ctypes as C
import math

import numpy as np
import pytest
import torch

import kv_testing as kt
import mlakv_ffi as ffi

pytestmark = pytest.mark.gpu

LATENT, ROPE = kt.LATENT, kt.ROPE
SCALE = 1.0 / math.sqrt(192.0)


def _calls(lib, cache, state, stream):
    """The step: append, whole-context attention, selected-token attention; on `stream`."""
    heads, row = state["heads"], (LATENT + ROPE) * 2
    q, table, lens = state["q"], state["table"], state["lens"]
    ffi.check(lib.mlakvAppend(C.byref(cache.view), 0, 1, state["new_latent"].data_ptr(), state["new_latent"].stride(0) * 2,
                              state["new_latent"].stride(1) * 2, state["new_rope"].data_ptr(), state["new_rope"].stride(0) * 2,
                              state["new_rope"].stride(1) * 2, state["slots"].data_ptr(), state["slots"].numel(), stream))
    ffi.check(lib.mlakvAttnDecode(C.byref(state["plan"]), C.byref(cache.view), 0, q.data_ptr(), heads * row, row,
                                  q.data_ptr() + LATENT * 2, heads * row, row, table.data_ptr(), table.shape[1], lens.data_ptr(),
                                  float(SCALE), state["out"].data_ptr(), heads * LATENT * 2, LATENT * 2, state["lse"].data_ptr(),
                                  state["workspace"].data_ptr(), int(state["plan"].workspace_bytes), stream))
    ffi.check(lib.mlakvAttnDecodeSparse(C.byref(state["sparse_plan"]), C.byref(cache.view), 0, q.data_ptr(), heads * row, row,
                                        q.data_ptr() + LATENT * 2, heads * row, row, table.data_ptr(), table.shape[1],
                                        lens.data_ptr(), state["selection"].data_ptr(), state["selection"].stride(0), float(SCALE),
                                        state["sparse_out"].data_ptr(), heads * LATENT * 2, LATENT * 2, state["sparse_lse"].data_ptr(),
                                        state["sparse_workspace"].data_ptr(), int(state["sparse_plan"].workspace_bytes), stream))


def test_a_captured_decode_step_replays_like_eager_calls():
    lib = ffi.load()
    bs, heads, k = 64, 64, 512
    ctxs = [1500, 700, 2047, 64, 1, 900, 1300, 513]
    batch = len(ctxs)
    blocks = sum(-(-(n + 8) // bs) for n in ctxs) + 4
    pool = kt.build_tables([n + 8 for n in ctxs], bs, blocks, seed=11)   # room for the rows the replays append
    table = pool.table()
    cache = kt.PagedCache(1, blocks, bs)
    total = sum(ctxs)
    kt.append(cache, kt.randn_bf16((1, total, LATENT), seed=12).cuda(), kt.randn_bf16((1, total, ROPE), seed=13).cuda(),
              kt.dev_i32(kt.slots_for(table, ctxs, bs)))
    torch.cuda.synchronize()
    twin = kt.PagedCache(1, blocks, bs)        # the eager calls get a cache of their own with the same bytes
    twin.latent.copy_(cache.latent)
    twin.rope.copy_(cache.rope)

    def make_state():
        plan = kt.make_plan(batch, heads, 2048 + 8, bs, False)
        sparse_plan = kt.make_plan(batch, heads, k, bs, False, selection=True)
        assert sparse_plan.selection_units == ffi.ATTN_UNITS_HEAD_BLOCK_HALVES
        return {"heads": heads, "plan": plan, "sparse_plan": sparse_plan,
                "q": torch.zeros(batch, heads, LATENT + ROPE, dtype=torch.bfloat16, device="cuda"),
                "table": kt.dev_i32(table), "lens": torch.zeros(batch, dtype=torch.int32, device="cuda"),
                "slots": torch.zeros(batch, dtype=torch.int32, device="cuda"),
                "new_latent": torch.zeros(1, batch, LATENT, dtype=torch.bfloat16, device="cuda"),
                "new_rope": torch.zeros(1, batch, ROPE, dtype=torch.bfloat16, device="cuda"),
                "selection": torch.full((batch, k), -1, dtype=torch.int32, device="cuda"),
                "out": torch.zeros(batch, heads, LATENT, dtype=torch.bfloat16, device="cuda"),
                "lse": torch.zeros(batch, heads, dtype=torch.float32, device="cuda"),
                "sparse_out": torch.zeros(batch, heads, LATENT, dtype=torch.bfloat16, device="cuda"),
                "sparse_lse": torch.zeros(batch, heads, dtype=torch.float32, device="cuda"),
                "workspace": torch.empty(int(plan.workspace_bytes), dtype=torch.uint8, device="cuda"),
                "sparse_workspace": torch.empty(int(sparse_plan.workspace_bytes), dtype=torch.uint8, device="cuda")}

    def set_inputs(state, step):
        """Step `step`: every sequence gets one more row; new query, new selection."""
        lens = [n + step + 1 for n in ctxs]
        rng = np.random.default_rng(100 + step)
        selection = np.full((batch, k), -1, dtype=np.int32)
        for s, n in enumerate(lens):
            take = min(n, k)
            selection[s, :take] = rng.permutation(n)[:take]
        slots = [int(table[s, (n - 1) // bs]) * bs + (n - 1) % bs for s, n in enumerate(lens)]
        state["q"].copy_(kt.randn_bf16((batch, heads, LATENT + ROPE), seed=200 + step).cuda())
        state["new_latent"].copy_(kt.randn_bf16((1, batch, LATENT), seed=300 + step).cuda())
        state["new_rope"].copy_(kt.randn_bf16((1, batch, ROPE), seed=400 + step).cuda())
        state["lens"].copy_(kt.dev_i32(lens))
        state["slots"].copy_(kt.dev_i32(slots))
        state["selection"].copy_(kt.dev_i32(selection))
        for name in ("out", "sparse_out"):
            state[name].fill_(float("nan"))
        return lens, selection

    captured, eager = make_state(), make_state()
    side = torch.cuda.Stream()
    # Everything the library sets up on first use (kernel attributes, the counters' address) happens in
    # eager calls before the capture.
    set_inputs(eager, 0)
    _calls(lib, twin, eager, kt.stream_ptr())
    torch.cuda.synchronize()
    twin.latent.copy_(cache.latent)
    twin.rope.copy_(cache.rope)

    set_inputs(captured, 0)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        _calls(lib, cache, captured, C.c_void_p(torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    cache.latent.copy_(twin.latent)       # (the capture itself runs nothing; keep the two caches equal whatever it did)
    cache.rope.copy_(twin.rope)

    for step in range(5):
        lens, selection = set_inputs(captured, step)
        set_inputs(eager, step)
        graph.replay()
        _calls(lib, twin, eager, kt.stream_ptr())
        torch.cuda.synchronize()
        assert torch.equal(cache.latent, twin.latent) and torch.equal(cache.rope, twin.rope), step
        for name in ("out", "lse", "sparse_out", "sparse_lse"):
            assert torch.equal(captured[name], eager[name]), (step, name)
        if step in (0, 4):                 # and the eager calls are right
            expected, _ = kt.oracle_attention(twin, 0, eager["q"], table, lens, SCALE)
            got = eager["out"].float().cpu().numpy()
            assert np.abs(got - expected).max() <= 2e-2 * np.abs(expected).max()
            expected, _ = kt.oracle_attention(twin, 0, eager["q"], table, lens, SCALE, sparse_indices=selection)
            got = eager["sparse_out"].float().cpu().numpy()
            assert np.abs(got - expected).max() <= 2e-2 * np.abs(expected).max()
        # eager work of the program's own between replays
        torch.zeros(1 << 20, device="cuda").sum().item()


def test_recorded_steps_side_by_side_share_no_counters():
    """Two recorded steps of more layers than the library ever had regions handed out in turn, each with a workspace of
    its own, replayed on two streams without an order between them: every launch in them is of workgroups that meet on
    counters (units of 16 heads shared by four and by five to eight, whole contexts and selections, and the merge inside the launch).
    Every replay gives the bits of the same calls made one after the other."""
    lib, bs, heads, layers = ffi.load(), 64, 64, 20
    ctxs = [1700, 1100, 33, 1500, 1, 1024]
    batch = len(ctxs)
    blocks = sum(-(-n // bs) for n in ctxs) + 2
    table = kt.build_tables(ctxs, bs, blocks, seed=421, max_blocks=28).table()
    cache = kt.PagedCache(1, blocks, bs)
    kt.append(cache, kt.randn_bf16((1, sum(ctxs), LATENT), seed=422).cuda(), kt.randn_bf16((1, sum(ctxs), ROPE), seed=423).cuda(),
              kt.dev_i32(kt.slots_for(table, ctxs, bs)))
    rng = np.random.default_rng(424)
    table_d, lens = kt.dev_i32(table), [kt.dev_i32(ctxs), kt.dev_i32([min(n, 700) for n in ctxs])]
    selections = {}
    for k in (700, 1100):
        chosen = np.full((batch, k), -1, dtype=np.int32)
        for s, n in enumerate(ctxs):
            chosen[s, :min(n, k)] = rng.permutation(n)[:k]
        selections[k] = kt.dev_i32(chosen)
    plans = [kt.make_plan(batch, heads, 1700, bs, False), kt.make_plan(batch, heads, 700, bs, False),
             kt.make_plan(batch, heads, 1700, bs, False, merge_mode=ffi.ATTN_MERGE_IN_LAUNCH, merge_spin_us=-1)]
    sparse_plans = {k: kt.make_plan(batch, heads, k, bs, False, selection=True) for k in selections}
    assert [plan.reserved for plan in sparse_plans.values()] == [3, 5]
    row = (LATENT + ROPE) * 2

    class Step:
        def __init__(self, seed):
            self.q = kt.randn_bf16((layers, batch, heads, LATENT + ROPE), seed=seed).cuda()
            self.out = torch.zeros(layers, 5, batch, heads, LATENT, dtype=torch.bfloat16, device="cuda")
            size = max(int(p.workspace_bytes) for p in plans + list(sparse_plans.values()))
            self.workspace = torch.empty(size, dtype=torch.uint8, device="cuda")

        def calls(self):
            stream = kt.stream_ptr()
            for layer in range(layers):
                q = self.q[layer].data_ptr()
                head = (C.byref(cache.view), 0, q, heads * row, row, q + LATENT * 2, heads * row, row, table_d.data_ptr(), table_d.shape[1])

                def tail(n):
                    return (SCALE, self.out[layer, n].data_ptr(), heads * LATENT * 2, LATENT * 2, None, self.workspace.data_ptr(),
                            self.workspace.numel(), stream)

                for n, plan in enumerate(plans):
                    ffi.check(lib.mlakvAttnDecode(C.byref(plan), *head, lens[n % 2].data_ptr(), *tail(n)))
                for n, (k, chosen) in enumerate(selections.items()):
                    ffi.check(lib.mlakvAttnDecodeSparse(C.byref(sparse_plans[k]), *head, lens[0].data_ptr(), chosen.data_ptr(), k, *tail(3 + n)))

    steps = [Step(425), Step(426)]
    want, graphs, streams = [], [], [torch.cuda.Stream(), torch.cuda.Stream()]
    for step in steps:
        step.calls()
        torch.cuda.synchronize()
        want.append(step.out.clone())
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            step.calls()
        graphs.append(graph)
    assert torch.isfinite(want[0].float()).all()
    assert not torch.equal(want[0][:, 0], want[0][:, 2])  # (the same contexts in shared units and in the split)
    for _ in range(6):
        for step in steps:
            step.out.fill_(float("nan"))
        torch.cuda.synchronize()
        for graph, stream in zip(graphs, streams):
            with torch.cuda.stream(stream):
                graph.replay()
                graph.replay()
        torch.cuda.synchronize()
        for step, expected in zip(steps, want):
            assert torch.equal(step.out, expected)
