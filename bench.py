#!/usr/bin/env python3
"""Benchmark of the paged MLA KV-cache hot path on one MI355X.

A step is one pass of the hot path over one batch of synthetic input, for the workload the
headline metric is quoted on:
    43 layers, batch 32, contexts uniform in [128, 2048], block 64, seeded-shuffled free list,
    bf16 rows of 576 elements (512 latent + 64 rope); per step: host block-pool bookkeeping,
    metadata upload, append of one row per sequence per layer, gather of every sequence's
    full context into contiguous [sum ctx, 576] rows per layer.
`value` is algorithmic bytes per step / wall time per step with all inputs resident in HBM.
The decode-attention configuration (configs[2]: batch 32, 64 heads, context 2048) is timed in
the same run and reported under "attention" (us per launch and fraction of the HBM roofline);
launches rotate over 8 layer slices (604 MB) so the 256 MB Infinity Cache cannot hold the KV.

Prints ONE JSON line. Everything goes through the C ABI (include/mlakv.h); the CPU oracle is
used only for the cpu_baseline leg.
"""
import argparse
import ctypes as C
import gc
import json
import math
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(ROOT, "ascend-moe-engine_amd", "python"))
sys.path.insert(0, os.path.join(ROOT, "oracle"))

# HBM bytes per algorithmic byte of the gather kernel, from two rocprofv3 --pmc runs of this file
# (FETCH_SIZE scaled by 2.000, WRITE_SIZE by 1.000, the factors a plain 1 GiB copy gives; figures in
# profiles/bench_hbm_counters.md): (1556.12 + 1555.98) MB measured for the dispatch of 31,411 rows x
# 43 layers against 3112.04 MB algorithmic.
GATHER_TRAFFIC_PER_ALGORITHMIC_BYTE = 1.0000
HBM_PEAK_GBPS = 8000.0      # MI355X HBM3E, published
MFMA_BF16_PEAK_TFLOPS = 2500.0
LATENT, ROPE, ROW = 512, 64, 576
ROW_BYTES = ROW * 2
CONTEXT_SEED = 20251125
# Context draws of the headline workload (numpy default_rng(seed).integers(128, 2049, 32)): the first
# has the distribution's own mean (1088.0 against (128 + 2048) / 2 = 1088); the others are the three
# seeds from CONTEXT_SEED on, whatever their means are (1231, 1136, 981). The reported value is the
# lowest of the four runs.
HEADLINE_SEEDS = (20251176, 20251125, 20251126, 20251127)
# HBM bytes per algorithmic byte of the attention launches (decode + merge kernel), from the
# rocprofv3 --pmc runs of this file summarised in profiles/bench_hbm_counters.md (FETCH_SIZE
# x2.000, WRITE_SIZE x1.000 as for the gather): the excess is the partials of sequences split
# over several workgroups, written once and read once.
_TRAFFIC_SOURCE = ("rocprofv3 --pmc FETCH_SIZE x2.000 + WRITE_SIZE x1.000 per decode + merge dispatch pair of this command, "
                   "applied as a ratio to the algorithmic bytes of the timed launches")
ATTENTION_TRAFFIC = {
    "attention": {"ratio": 1.429, "source": _TRAFFIC_SOURCE},        # 114.27 MB against 79.96 MB
    "attention_fp8": {"ratio": 1.254, "source": _TRAFFIC_SOURCE},    # 221.43 MB against 176.52 MB
    "attention_long": {"ratio": 1.060, "source": _TRAFFIC_SOURCE},   # 952.84 MB against 898.64 MB
    "attention_sparse": {"ratio": 1.320, "source": _TRAFFIC_SOURCE}, # 30.90 MB against 23.41 MB (one dispatch: halved whole-selection units)
    "attention_short": {"ratio": 1.018, "source": _TRAFFIC_SOURCE},  # 14.14 MB against 13.89 MB (one dispatch, no partials)
    "attention_sparse_fp8": {"ratio": 1.613, "source": _TRAFFIC_SOURCE}, # 22.65 MB against 14.04 MB
    "indexer": {"ratio": 1.096, "source": _TRAFFIC_SOURCE},          # 38.30 MB against 34.96 MB
}
# Host orchestration of the reference's own 43-layer decode step (its mock build: every operator
# launch is a no-op), measured in the build container on 8 cores: 128 steps, 132,480 launches,
# 48.9 ms.
REFERENCE_HOST_PLUMBING_MS_PER_STEP = 0.38


def sustained_us(torch, fn, min_iters, warm_ms=250.0, timed_ms=100.0):
    """Average microseconds per fn(i) launch once the device has settled: launches get faster for
    some 100 ms of sustained load (the long attention shape measured 284 us per launch over 2
    launches, 254 over 32, 227 over 512; most likely clock and power management), so the launches
    run back to back for `warm_ms` before the timed ones, which then cover at least `timed_ms`."""
    def run(n):
        start, stop = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        start.record()
        for i in range(n):
            fn(i)
        stop.record()
        torch.cuda.synchronize()
        return start.elapsed_time(stop) * 1e3 / n
    rough = run(16)
    run(max(16, int(warm_ms * 1e3 / rough)))
    return run(max(min_iters, int(timed_ms * 1e3 / rough)))


def parse_args():
    p = argparse.ArgumentParser()
    p.add_argument("--gpus", type=int, default=1)
    p.add_argument("--steps", type=int, default=60)
    p.add_argument("--warmup", type=int, default=60)
    p.add_argument("--no-cpu-baseline", action="store_true")
    p.add_argument("--no-attention", action="store_true")
    p.add_argument("--side-only", action="store_true", help="development aid: time only the FP8 append/gather and compaction kernels")
    p.add_argument("--attention-only", action="store_true", help="development aid: time only the attention configurations")
    p.add_argument("--config5-only", action="store_true", help="development aid: run only the continuous-batching loop of configs[4]")
    p.add_argument("--config5-pool-gb", type=float, default=200.0, help="KV pool of the configs[4] loop, in GB (clamped to free memory)")
    p.add_argument("--attn-merge-spin-us", type=int, default=0,
                   help="development aid: bound of the in-launch merge's wait (0: the plan's default, -1: never wait)")
    p.add_argument("--attn-units", choices=["auto", "split", "head-block", "halves"], default="auto",
                   help="development aid: how the selected-token attention cuts its work (MLAKV_ATTN_UNITS_*)")
    p.add_argument("--attn-merge", choices=["auto", "in", "second"], default="auto",
                   help="development aid: how the attention launches merge their partials (default: the planner's choice)")
    p.add_argument("--attn-chunk-tiles", type=int, default=0, help="development aid: fixed tiles per work unit of the attention launches")
    p.add_argument("--attn-work-groups", type=int, default=0, help="development aid: workgroups per head group of the attention launches")
    p.add_argument("--attn-host-lens", action="store_true",
                   help="development aid: pass the lengths from the host (mlakvAttnDecodeHostLens) where the batch allows")
    p.add_argument("--split-out", action="store_true", help="gather into separate latent/rope planes instead of 576-wide rows")
    return p.parse_args()


def stream_ptr(torch):
    return C.c_void_p(torch.cuda.current_stream().cuda_stream)


def bench_append_gather(args, torch, np, ffi, seed):
    gc.collect()
    lib = ffi.load()
    layers, batch, bs = 43, 32, 64
    rng = np.random.default_rng(seed)
    ctxs = [int(v) for v in rng.integers(128, 2049, size=batch)]
    total_steps = args.warmup + args.steps
    max_ctx = 2048 + max(128, -(-total_steps // bs) * bs)  # every sequence grows by one token per step
    pool_blocks = sum(-(-(c + total_steps) // bs) for c in ctxs) + 32
    arena = ffi.Arena(ffi.BACKEND_HIP)
    cache = ffi.KvCache(arena, num_layers=layers, block_size=bs, max_context_len=max_ctx, max_batch=batch,
                        pool_blocks=pool_blocks, seed=seed, shuffle=1)
    arena.commit()
    cache.bind()
    arena.seal()
    view = cache.view()
    for s, n in enumerate(ctxs):
        cache.add_sequence(s, n)
    gen = torch.Generator(device="cuda").manual_seed(1)
    # prefill the pool with N(0,1) rows so the gather reads real data
    total = sum(ctxs)
    table = cache.host_block_table()
    slots = np.concatenate([table[s, np.arange(n) // bs].astype(np.int64) * bs + np.arange(n) % bs
                            for s, n in enumerate(ctxs)]).astype(np.int32)
    slots_dev = torch.as_tensor(slots, device="cuda")
    for layer in range(layers):
        lat = torch.randn(total, LATENT, generator=gen, device="cuda").to(torch.bfloat16)
        rop = torch.randn(total, ROPE, generator=gen, device="cuda").to(torch.bfloat16)
        ffi.check(lib.mlakvAppend(C.byref(view), layer, 1, lat.data_ptr(), 0, LATENT * 2, rop.data_ptr(), 0, ROPE * 2,
                                  slots_dev.data_ptr(), total, stream_ptr(torch)))
        torch.cuda.synchronize()
    step_latent = torch.randn(layers, batch, LATENT, generator=gen, device="cuda").to(torch.bfloat16)
    step_rope = torch.randn(layers, batch, ROPE, generator=gen, device="cuda").to(torch.bfloat16)
    rows_cap = total + batch * total_steps
    if args.split_out:
        out_latent = torch.empty(layers, rows_cap, LATENT, dtype=torch.bfloat16, device="cuda")
        out_rope = torch.empty(layers, rows_cap, ROPE, dtype=torch.bfloat16, device="cuda")
        dst = (out_latent.data_ptr(), rows_cap * LATENT * 2, LATENT * 2, out_rope.data_ptr(), rows_cap * ROPE * 2, ROPE * 2)
    else:
        out = torch.empty(layers, rows_cap, ROW, dtype=torch.bfloat16, device="cuda")
        dst = (out.data_ptr(), rows_cap * ROW_BYTES, ROW_BYTES, out.data_ptr() + LATENT * 2, rows_cap * ROW_BYTES, ROW_BYTES)
    allocations_before = arena.device_allocations
    # The gather of every timed step stamps its own start and end into a pair of HIP events
    # (mlakvGatherTimed): events recorded around it would each put a marker packet into the queue,
    # which cost the step 4 to 5 us.
    hip = HipEvents()
    gather_events = [(hip.create(), hip.create()) for _ in range(args.steps)]
    timed_steps = []

    def step(timed):
        cache.append_token_all()
        # the step's metadata and its 32 x 43 rows in one launch
        cache.upload_step_and_append(0, layers, step_latent.data_ptr(), batch * LATENT * 2, LATENT * 2, step_rope.data_ptr(),
                                     batch * ROPE * 2, ROPE * 2, stream_ptr(torch))
        gather_args = (C.byref(view), 0, layers, cache.device_block_table, cache.num_blocks, cache.device_seq_lens,
                       cache.device_cu_seq_lens, batch, max_ctx, dst[0], dst[1], dst[2], dst[3], dst[4], dst[5], stream_ptr(torch))
        if timed:
            pair = gather_events[len(timed_steps)]
            timed_steps.append(pair)
            ffi.check(lib.mlakvGatherTimed(*gather_args, pair[0], pair[1]))
        else:
            ffi.check(lib.mlakvGather(*gather_args))

    for _ in range(args.warmup):
        step(False)
    torch.cuda.synchronize()
    rows_per_step = []
    t0 = time.perf_counter()
    for i in range(args.steps):
        step(True)
        rows_per_step.append(total + batch * (args.warmup + i + 1))
    torch.cuda.synchronize()
    elapsed = time.perf_counter() - t0
    assert arena.device_allocations == allocations_before, "a step allocated device memory"

    blocks_per_step = []
    lens = cache.host_seq_lens()
    # algorithmic bytes: append 2*R*row + 4*R; gather 2*sum(ctx)*row + 4*sum(ceil(ctx/bs)), per layer
    def gather_bytes(rows, final_lens, back):
        nblk = sum(-(-(int(l) - back) // bs) for l in final_lens)
        return layers * (2 * rows * ROW_BYTES + 4 * nblk)
    append_bytes = layers * (2 * batch * ROW_BYTES + 4 * batch)
    g_bytes = [gather_bytes(rows_per_step[i], lens, args.steps - 1 - i) for i in range(args.steps)]
    total_bytes = sum(g_bytes) + append_bytes * args.steps
    gather_ms = [hip.elapsed_ms(a, b) for a, b in timed_steps]
    for a, b in gather_events:
        hip.destroy(a)
        hip.destroy(b)
    # the append launch on its own, after the timed region: the same rows to the same slots again,
    # 64 launches back to back between two events (one launch between two events times the events)
    def append_again():
        ffi.check(lib.mlakvAppend(C.byref(view), 0, layers, step_latent.data_ptr(), batch * LATENT * 2, LATENT * 2,
                                  step_rope.data_ptr(), batch * ROPE * 2, ROPE * 2, cache.device_slot_mapping, batch,
                                  stream_ptr(torch)))
    for _ in range(8):
        append_again()
    torch.cuda.synchronize()
    pair = (torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True))
    pair[0].record()
    for _ in range(64):
        append_again()
    pair[1].record()
    torch.cuda.synchronize()
    append_ms = [pair[0].elapsed_time(pair[1]) / 64]
    gather_gbps = sum(g_bytes) / (sum(gather_ms) * 1e-3) / 1e9
    result = {
        "value": total_bytes / elapsed / 1e9,
        "ms_per_step": elapsed / args.steps * 1e3,
        "gather_ms": sum(gather_ms) / len(gather_ms),
        "append_ms": sum(append_ms) / len(append_ms),
        "gather_gbps": gather_gbps,
        "append_gbps": append_bytes / (sum(append_ms) / len(append_ms) * 1e-3) / 1e9,
        "bytes_per_step": total_bytes / args.steps,
        "gather_bytes_per_launch": sum(g_bytes) / args.steps,
        "mean_ctx": sum(rows_per_step) / len(rows_per_step) / batch,
        "ctxs": ctxs, "pool_blocks": pool_blocks, "seed": seed, "initial_mean_ctx": sum(ctxs) / batch,
    }
    cache.close()
    arena.close()
    return result


class HipEvents:
    """HIP events through the runtime's C interface (the library torch has loaded), for the entry
    point that takes hipEvent_t handles."""

    def __init__(self):
        self.hip = C.CDLL("libamdhip64.so")
        self.hip.hipEventCreate.argtypes = [C.POINTER(C.c_void_p)]
        self.hip.hipEventDestroy.argtypes = [C.c_void_p]
        self.hip.hipEventElapsedTime.argtypes = [C.POINTER(C.c_float), C.c_void_p, C.c_void_p]

    def create(self):
        event = C.c_void_p()
        status = self.hip.hipEventCreate(C.byref(event))
        if status != 0:
            raise RuntimeError(f"hipEventCreate failed with {status}")
        return event

    def elapsed_ms(self, start, stop):
        ms = C.c_float()
        status = self.hip.hipEventElapsedTime(C.byref(ms), start, stop)
        if status != 0:
            raise RuntimeError(f"hipEventElapsedTime failed with {status}")
        return float(ms.value)

    def destroy(self, event):
        self.hip.hipEventDestroy(event)


def draw_contexts(np, kind, batch, seed):
    """Context lengths of the attention configurations, from a seeded numpy Generator (PCG64)."""
    rng = np.random.default_rng(seed)
    if kind == "uniform_512_8192":      # configs[3]
        return [int(v) for v in rng.integers(512, 8193, size=batch)]
    if kind == "lognormal_4096_cap_32768":  # configs[4]: median 4096, sigma 1.0
        return [int(min(32768, max(1, round(v)))) for v in np.exp(rng.normal(math.log(4096.0), 1.0, size=batch))]
    raise ValueError(kind)


def fill_cache(torch, np, ffi, lib, cache, view, ctxs, layers, bs, seed, outlier_fraction=0.0):
    """Every live slot of `layers` layer slices gets N(0,1) rows (optionally with outliers x20) through
    the append kernel (an FP8 cache quantizes on the way), in pieces of at most 128k rows."""
    table = cache.host_block_table()
    slots = np.concatenate([table[s, np.arange(n) // bs].astype(np.int64) * bs + np.arange(n) % bs
                            for s, n in enumerate(ctxs)]).astype(np.int32)
    slots_dev = torch.as_tensor(slots, device="cuda")
    gen = torch.Generator(device="cuda").manual_seed(seed)
    piece = 128 * 1024
    for layer in range(layers):
        for start in range(0, len(slots), piece):
            rows = min(piece, len(slots) - start)
            x = torch.randn(rows, ROW, generator=gen, device="cuda")
            if outlier_fraction > 0:
                x = torch.where(torch.rand(rows, ROW, generator=gen, device="cuda") < outlier_fraction, x * 20.0, x)
            x = x.to(torch.bfloat16)
            ffi.check(lib.mlakvAppend(C.byref(view), layer, 1, x.data_ptr(), 0, ROW_BYTES, x.data_ptr() + LATENT * 2, 0, ROW_BYTES,
                                      slots_dev.data_ptr() + 4 * start, rows, stream_ptr(torch)))
            torch.cuda.synchronize()


def bench_attention(args, torch, np, ffi, ctxs, fp8=False, heads=64, slices=8, iters=None, label=None, distribution=None,
                    outlier_fraction=0.0, mx_quant=False, sparse_k=None, traffic_ratio=None):
    gc.collect()
    lib = ffi.load()
    bs = 64
    batch = len(ctxs)
    max_ctx = max(ctxs)
    blocks = sum(-(-c // bs) for c in ctxs)
    pool_blocks = blocks + 8
    arena = ffi.Arena(ffi.BACKEND_HIP)
    cache = ffi.KvCache(arena, num_layers=slices, block_size=bs, max_context_len=max_ctx, max_batch=batch,
                        pool_blocks=pool_blocks, seed=7, shuffle=1, dtype=ffi.DTYPE_FP8_E4M3 if fp8 else ffi.DTYPE_BF16)
    plan = ffi.AttnPlan()
    merge_mode = {"auto": ffi.ATTN_MERGE_AUTO, "in": ffi.ATTN_MERGE_IN_LAUNCH, "second": ffi.ATTN_MERGE_SECOND_LAUNCH}[args.attn_merge]
    units = {"auto": ffi.ATTN_UNITS_AUTO, "split": ffi.ATTN_UNITS_SPLIT, "head-block": ffi.ATTN_UNITS_HEAD_BLOCK,
             "halves": ffi.ATTN_UNITS_HEAD_BLOCK_HALVES}[args.attn_units] if sparse_k or max_ctx <= ffi.ATTN_HEAD_BLOCK_TOKENS else 0
    if merge_mode != ffi.ATTN_MERGE_AUTO or args.attn_chunk_tiles or args.attn_work_groups or units:
        options = ffi.AttnPlanOptions(args.attn_chunk_tiles, args.attn_work_groups, merge_mode, args.attn_merge_spin_us, 1 if sparse_k else 0, units)
        ffi.check(lib.mlakvAttnPlanInitEx(batch, heads, sparse_k or max_ctx, bs, cache.config.dtype, C.byref(options), C.byref(plan)))
    elif sparse_k:
        ffi.check(lib.mlakvAttnSparsePlanInit(batch, heads, sparse_k, bs, cache.config.dtype, C.byref(plan)))
    else:
        ffi.check(lib.mlakvAttnPlanInit(batch, heads, max_ctx, bs, cache.config.dtype, C.byref(plan)))
    arena.note_workspace(int(plan.workspace_bytes))
    arena.commit()
    arena.commit_workspace()
    cache.bind()
    arena.seal()
    view = cache.view()
    for s, n in enumerate(ctxs):
        cache.add_sequence(s, n)
    cache.upload_step(stream_ptr(torch))
    fill_cache(torch, np, ffi, lib, cache, view, ctxs, slices, bs, seed=2, outlier_fraction=outlier_fraction)
    gen = torch.Generator(device="cuda").manual_seed(3)
    q = torch.randn(slices, batch, heads, ROW, generator=gen, device="cuda").to(torch.bfloat16)
    out = torch.empty(slices, batch, heads, LATENT, dtype=torch.bfloat16, device="cuda")

    selection = None
    if sparse_k:
        # every sequence attends to sparse_k distinct random positions of its context (what a
        # top-k selection looks like to the memory system), a fresh draw per layer slice
        rng = np.random.default_rng(5)
        selection = torch.as_tensor(np.stack([np.stack([rng.permutation(n)[:sparse_k] for n in ctxs])
                                              for _ in range(slices)]).astype(np.int32), device="cuda")

    def launch_sparse(i):
        k = i % slices
        ffi.check(lib.mlakvAttnDecodeSparse(C.byref(plan), C.byref(view), k, q[k].data_ptr(), heads * ROW_BYTES, ROW_BYTES,
                                            q[k].data_ptr() + LATENT * 2, heads * ROW_BYTES, ROW_BYTES,
                                            cache.device_block_table, cache.num_blocks, cache.device_seq_lens,
                                            selection[k].data_ptr(), sparse_k, 1.0 / math.sqrt(192.0), out[k].data_ptr(),
                                            heads * LATENT * 2, LATENT * 2, None, arena.workspace, arena.workspace_bytes,
                                            stream_ptr(torch)))

    host_lens = (C.c_int32 * batch)(*ctxs)

    def launch_host_lens(i):
        k = i % slices
        ffi.check(lib.mlakvAttnDecodeHostLens(C.byref(plan), C.byref(view), k, q[k].data_ptr(), heads * ROW_BYTES, ROW_BYTES,
                                              q[k].data_ptr() + LATENT * 2, heads * ROW_BYTES, ROW_BYTES,
                                              cache.device_block_table, cache.num_blocks, host_lens,
                                              1.0 / math.sqrt(192.0), out[k].data_ptr(), heads * LATENT * 2, LATENT * 2, None,
                                              arena.workspace, arena.workspace_bytes, stream_ptr(torch)))

    def launch(i):
        if sparse_k:
            return launch_sparse(i)
        if args.attn_host_lens and batch <= 64:
            return launch_host_lens(i)
        k = i % slices
        ffi.check(lib.mlakvAttnDecode(C.byref(plan), C.byref(view), k, q[k].data_ptr(), heads * ROW_BYTES, ROW_BYTES,
                                      q[k].data_ptr() + LATENT * 2, heads * ROW_BYTES, ROW_BYTES,
                                      cache.device_block_table, cache.num_blocks, cache.device_seq_lens,
                                      1.0 / math.sqrt(192.0), out[k].data_ptr(), heads * LATENT * 2, LATENT * 2, None,
                                      arena.workspace, arena.workspace_bytes, stream_ptr(torch)))

    iters = iters or max(args.steps * 8, 64)

    def timed_us(fn):
        return sustained_us(torch, fn, iters)

    us = timed_us(launch)
    # the same launches with the lengths known on the host (what the aclnn face does for the reference's call)
    us_host_lens = timed_us(launch_host_lens) if not sparse_k and batch <= 64 and not args.attn_host_lens else None
    mx = None
    if mx_quant:
        # the reference's next stage, block-32 MX quantisation of the output: fused into the
        # attention epilogue, against attention followed by the standalone operator
        codes = torch.empty(slices, batch, heads, LATENT, dtype=torch.uint8, device="cuda")
        scales = torch.empty(slices, batch, heads, LATENT // 32, dtype=torch.uint8, device="cuda")
        targets = [ffi.MxQuantOut(codes[k].data_ptr(), heads * LATENT, LATENT, scales[k].data_ptr(), heads * (LATENT // 32),
                                  LATENT // 32) for k in range(slices)]

        def fused(i):
            k = i % slices
            ffi.check(lib.mlakvAttnDecodeMxQuant(C.byref(plan), C.byref(view), k, q[k].data_ptr(), heads * ROW_BYTES, ROW_BYTES,
                                                 q[k].data_ptr() + LATENT * 2, heads * ROW_BYTES, ROW_BYTES,
                                                 cache.device_block_table, cache.num_blocks, cache.device_seq_lens,
                                                 1.0 / math.sqrt(192.0), None, 0, 0, C.byref(targets[k]), None,
                                                 arena.workspace, arena.workspace_bytes, stream_ptr(torch)))

        def unfused(i):
            k = i % slices
            launch(i)
            ffi.check(lib.mlakvDynamicMxQuant(out[k].data_ptr(), LATENT * 2, batch * heads, LATENT, codes[k].data_ptr(), LATENT,
                                              scales[k].data_ptr(), LATENT // 32, stream_ptr(torch)))

        mx = {"us_fused_epilogue": timed_us(fused), "us_attention_then_quant": timed_us(unfused)}
    kv_row = 580 if fp8 else ROW_BYTES
    attended = batch * sparse_k if sparse_k else sum(ctxs)
    algorithmic = attended * kv_row + batch * heads * ROW * 2 + batch * heads * LATENT * 2 + 4 * blocks
    if sparse_k:
        algorithmic += 4 * batch * sparse_k
    flops = 2.0 * heads * attended * (ROW + LATENT)
    lengths = (f"ctx {ctxs[0]}" if min(ctxs) == max(ctxs)
               else f"ctx {distribution} (min {min(ctxs)}, mean {sum(ctxs) / batch:.0f}, max {max(ctxs)})")
    result = {
        "us_per_step": us,
        "workload": f"{label}: 1 layer per launch, batch {batch}, {heads} heads, {lengths}, block 64, "
                    f"{'fp8 e4m3 + fp32 row scale' if fp8 else 'bf16'} KV"
                    + (", N(0,1) rows with 1% of the elements x20" if outlier_fraction else ", N(0,1) rows")
                    + f", shuffled table, {slices} rotating layer slices"
                    + (f", {sparse_k} selected tokens per sequence" if sparse_k else ""),
        "roofline": {"bound": "hbm", "achieved": algorithmic / (us * 1e-6) / 1e9, "peak": HBM_PEAK_GBPS, "unit": "GB/s",
                     "frac": algorithmic / (us * 1e-6) / 1e9 / HBM_PEAK_GBPS,
                     "traffic": algorithmic * traffic_ratio["ratio"] if traffic_ratio else None},
        "algorithmic_bytes": algorithmic,
        "mfma_tflops": flops / (us * 1e-6) / 1e12,
        "mfma_frac_of_bf16_peak": flops / (us * 1e-6) / 1e12 / MFMA_BF16_PEAK_TFLOPS,
        "work_groups": int(plan.work_groups), "max_units": int(plan.max_units),
        "merge": ("none (a unit holds a whole selection for 16 heads)" if plan.selection_units == ffi.ATTN_UNITS_HEAD_BLOCK
                  else "in launch, pairs (two workgroups per selection and 16 heads; the second to finish combines)"
                  if plan.selection_units == ffi.ATTN_UNITS_HEAD_BLOCK_HALVES
                  else "chosen per launch: units of 16 heads (no partials, or pairs combined in the launch) while the longest context "
                       "the launch can see is short, else the 64-head kernel with a second launch"
                  if not sparse_k and plan.selection_units == ffi.ATTN_UNITS_AUTO and max_ctx <= ffi.ATTN_HEAD_BLOCK_TOKENS
                  else "in launch" if plan.merge_mode == ffi.ATTN_MERGE_IN_LAUNCH else "second launch"),
        "workspace_bytes": int(plan.workspace_bytes), "timing": "250 ms of back-to-back launches untimed, then at least 100 ms of them timed",
    }
    if traffic_ratio:
        result["roofline"]["traffic_source"] = traffic_ratio["source"]
    if min(ctxs) != max(ctxs):
        result["context_seed"] = CONTEXT_SEED
        result["total_tokens"] = sum(ctxs)
    if mx is not None:
        result["mx_quant_output"] = mx
    if us_host_lens is not None:
        result["host_known_lengths"] = {"us_per_step": us_host_lens,
                                        "what": "mlakvAttnDecodeHostLens: the lengths ride in the kernels' argument block, no device array is read"}
    cache.close()
    arena.close()
    return result


def bench_indexer(args, torch, np, ffi, batch=32, ctx=8192, heads=64, k=512, bs=64, slices=4):
    """Lightning Indexer at the shape the selected-token attention is timed on: FP8 index keys
    (128 + 4 bytes per cached token) scored against one query token per sequence, top-k selected.
    HIP-event time of the operator (score kernel + selection kernel) over rotating key pools."""
    gc.collect()
    lib = ffi.load()
    blocks = batch * (ctx // bs)
    rng = np.random.default_rng(9)
    keys = [torch.randint(0, 0x58, (blocks * bs, 128), dtype=torch.uint8, device="cuda") for _ in range(slices)]
    scales = torch.rand(blocks * bs, device="cuda") * 0.04 + 0.01
    table = torch.as_tensor(rng.permutation(blocks).astype(np.int32).reshape(batch, ctx // bs), device="cuda")
    lens = torch.full((batch,), ctx, dtype=torch.int32, device="cuda")
    query = torch.randint(0, 0x58, (batch, heads, 128), dtype=torch.uint8, device="cuda")
    weights = torch.randn(batch, heads, device="cuda").to(torch.bfloat16)
    q_scale = torch.rand(batch, heads, device="cuda") * 0.04 + 0.01
    out = torch.empty(batch, k, dtype=torch.int32, device="cuda")
    workspace = torch.empty(int(lib.mlakvIndexerWorkspaceBytes(batch, ctx)), dtype=torch.uint8, device="cuda")
    views = [ffi.IndexKeyView(kp.data_ptr(), bs * 128, 128, scales.data_ptr(), bs, blocks, bs, 128, 0) for kp in keys]

    def launch(i):
        ffi.check(lib.mlakvLightningIndexer(C.byref(views[i % slices]), query.data_ptr(), heads * 128, 128, weights.data_ptr(),
                                            heads * 2, q_scale.data_ptr(), heads, heads, table.data_ptr(), ctx // bs, lens.data_ptr(),
                                            batch, ctx, k, out.data_ptr(), k, workspace.data_ptr(), workspace.numel(),
                                            stream_ptr(torch)))
    us = sustained_us(torch, launch, 64)
    algorithmic = batch * ctx * (128 + 4) + batch * heads * (128 + 2 + 4) + 4 * batch * (ctx // bs) + 4 * batch * k
    return {"us_per_step": us,
            "workload": f"batch {batch}, ctx {ctx}, {heads} index heads x 128, top-{k}, block {bs}, e4m3 keys + fp32 row scale, "
                        f"shuffled table, {slices} rotating key pools",
            "roofline": {"bound": "hbm", "achieved": algorithmic / (us * 1e-6) / 1e9, "peak": HBM_PEAK_GBPS, "unit": "GB/s",
                         "frac": algorithmic / (us * 1e-6) / 1e9 / HBM_PEAK_GBPS,
                         "traffic": algorithmic * ATTENTION_TRAFFIC["indexer"]["ratio"],
                         "traffic_source": ATTENTION_TRAFFIC["indexer"]["source"]},
            "algorithmic_bytes": algorithmic, "timing": "250 ms of back-to-back launches untimed, then at least 100 ms of them timed"}


def bench_side_kernels(args, torch, np, ffi):
    """The other data-movement kernels of the path at configs[3]/[4]-like sizes (8 layers to bound
    memory): FP8 quantize-on-append, FP8 dequantising gather, bf16 compaction copy. HIP-event
    time per launch against algorithmic bytes."""
    gc.collect()
    lib = ffi.load()
    bs, layers, batch, max_ctx = 64, 8, 64, 8192
    rng = np.random.default_rng(11)
    ctxs = [int(v) for v in rng.integers(512, 8193, size=batch)]
    total = sum(ctxs)
    blocks = sum(-(-c // bs) for c in ctxs)
    out = {}

    def timed(fn, reps=5):
        return sustained_us(torch, lambda i: fn(), reps, warm_ms=100.0, timed_ms=50.0) * 1e-3

    gen = torch.Generator(device="cuda").manual_seed(5)
    lat = torch.randn(layers, total, LATENT, generator=gen, device="cuda").to(torch.bfloat16)
    rop = torch.randn(layers, total, ROPE, generator=gen, device="cuda").to(torch.bfloat16)
    for fp8 in (True, False):
        arena = ffi.Arena(ffi.BACKEND_HIP)
        cache = ffi.KvCache(arena, num_layers=layers, block_size=bs, max_context_len=max_ctx, max_batch=batch,
                            pool_blocks=blocks + 16, seed=3, shuffle=1, dtype=ffi.DTYPE_FP8_E4M3 if fp8 else ffi.DTYPE_BF16)
        arena.commit()
        cache.bind()
        arena.seal()
        view = cache.view()
        for s, n in enumerate(ctxs):
            cache.add_sequence(s, n)
        cache.upload_step(stream_ptr(torch))
        table = cache.host_block_table()
        slots = torch.as_tensor(np.concatenate([table[s, np.arange(n) // bs].astype(np.int64) * bs + np.arange(n) % bs
                                                for s, n in enumerate(ctxs)]).astype(np.int32), device="cuda")

        def append():
            ffi.check(lib.mlakvAppend(C.byref(view), 0, layers, lat.data_ptr(), total * LATENT * 2, LATENT * 2, rop.data_ptr(),
                                      total * ROPE * 2, ROPE * 2, slots.data_ptr(), total, stream_ptr(torch)))
        ms = timed(append)
        if fp8:
            nbytes = layers * (total * (ROW_BYTES + 580) + 4 * total)
            out["append_fp8"] = {"ms": ms, "gbps": nbytes / (ms * 1e-3) / 1e9, "frac": nbytes / (ms * 1e-3) / 1e9 / HBM_PEAK_GBPS,
                                 "rows": total, "layers": layers}
            dst = torch.empty(layers, total, ROW, dtype=torch.bfloat16, device="cuda")

            def gather():
                ffi.check(lib.mlakvGather(C.byref(view), 0, layers, cache.device_block_table, cache.num_blocks,
                                          cache.device_seq_lens, cache.device_cu_seq_lens, batch, max_ctx, dst.data_ptr(),
                                          total * ROW_BYTES, ROW_BYTES, dst.data_ptr() + LATENT * 2, total * ROW_BYTES, ROW_BYTES,
                                          stream_ptr(torch)))
            ms = timed(gather)
            nbytes = layers * (total * (580 + ROW_BYTES) + 4 * blocks)
            out["gather_fp8"] = {"ms": ms, "gbps": nbytes / (ms * 1e-3) / 1e9, "frac": nbytes / (ms * 1e-3) / 1e9 / HBM_PEAK_GBPS,
                                 "rows": total, "layers": layers}
            del dst
        else:
            # fused latent RMSNorm + key RoPE + append of one layer over every row (prefill-sized launch)
            kv_a = torch.cat([lat[0], rop[0]], dim=1).contiguous()
            gamma = torch.ones(LATENT, dtype=torch.bfloat16, device="cuda")
            ang = torch.outer(torch.arange(max_ctx, dtype=torch.float32, device="cuda"),
                              10000.0 ** (-torch.arange(0, ROPE // 2, dtype=torch.float32, device="cuda") * 2 / ROPE))
            cos = torch.cat([ang.cos(), ang.cos()], dim=1).to(torch.bfloat16)
            sin = torch.cat([ang.sin(), ang.sin()], dim=1).to(torch.bfloat16)
            positions = torch.as_tensor(np.concatenate([np.arange(n) for n in ctxs]).astype(np.int32), device="cuda")

            def fused():
                ffi.check(lib.mlakvNormRopeAppend(C.byref(view), 0, kv_a.data_ptr(), ROW_BYTES, gamma.data_ptr(), 1e-6, cos.data_ptr(),
                                                  sin.data_ptr(), ROPE * 2, positions.data_ptr(), slots.data_ptr(), total, None, 0,
                                                  None, 0, None, 0, 0, 0, stream_ptr(torch)))
            ms = timed(fused)
            nbytes = total * (2 * ROW_BYTES + 8)
            out["norm_rope_append_bf16"] = {"ms": ms, "gbps": nbytes / (ms * 1e-3) / 1e9,
                                            "frac": nbytes / (ms * 1e-3) / 1e9 / HBM_PEAK_GBPS, "rows": total, "layers": 1}
            # the same with the query's rope slices (64 heads, 128 of every 1152 bytes) rotated in place
            q_tokens, heads = min(total, 32768), 64
            q = torch.randn(q_tokens, heads, ROW, device="cuda").to(torch.bfloat16)

            def fused_with_query():
                ffi.check(lib.mlakvNormRopeAppend(C.byref(view), 0, kv_a.data_ptr(), ROW_BYTES, gamma.data_ptr(), 1e-6, cos.data_ptr(),
                                                  sin.data_ptr(), ROPE * 2, positions.data_ptr(), slots.data_ptr(), q_tokens, None, 0,
                                                  None, 0, q.data_ptr() + LATENT * 2, heads * ROW_BYTES, ROW_BYTES, heads,
                                                  stream_ptr(torch)))
            ms = timed(fused_with_query)
            nbytes = q_tokens * (2 * ROW_BYTES + 8 + heads * 2 * ROPE * 2)
            out["norm_rope_append_query_rope_bf16"] = {"ms": ms, "gbps": nbytes / (ms * 1e-3) / 1e9,
                                                       "frac": nbytes / (ms * 1e-3) / 1e9 / HBM_PEAK_GBPS, "rows": q_tokens,
                                                       "heads": heads, "layers": 1}
            del q
            del kv_a
            # free every other sequence, then compact: the device copies each moved block in every layer
            for s in range(0, batch, 2):
                cache.free_sequence(s)
            torch.cuda.synchronize()
            # (the C call alone between the events: building a Python list of the moves inside the
            # bracket once triggered a 36 ms garbage collection that was then read as the library's time)
            start, stop = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            moves_out, moves_count = (C.c_int32 * (2 * cache.pool_blocks))(), C.c_int64()
            start.record()
            ffi.check(lib.mlakvKvCacheCompact(cache.handle, moves_out, C.byref(moves_count), stream_ptr(torch)))
            stop.record()
            torch.cuda.synchronize()
            whole_ms = start.elapsed_time(stop)
            moves = [(moves_out[2 * i], moves_out[2 * i + 1]) for i in range(moves_count.value)]
            # the copy kernel alone, replaying the same move list from device memory
            moves_dev = torch.as_tensor(np.asarray(moves, dtype=np.int32).reshape(-1), device="cuda")

            def copy():
                ffi.check(lib.mlakvCopyBlocks(C.byref(view), 0, layers, moves_dev.data_ptr(), len(moves), stream_ptr(torch)))
            ms = timed(copy)
            nbytes = 2 * len(moves) * bs * ROW_BYTES * layers
            out["compaction_bf16"] = {"ms": ms, "gbps": nbytes / (ms * 1e-3) / 1e9, "frac": nbytes / (ms * 1e-3) / 1e9 / HBM_PEAK_GBPS,
                                      "moved_blocks": len(moves), "layers": layers,
                                      "ms_with_host_plan_and_upload": whole_ms}
        cache.close()
        arena.close()
    return out


def bench_config5(args, torch, np, ffi, batch=128, heads=64, steps=6, warmup=2):
    """reservation pressure over all 43 layers. A pool of about 200 GB (clamped to what
    the device has free), 128 sequences with lognormal contexts, seeded finish times; a finished
    sequence frees its blocks and a new one (fresh lognormal context) takes its place from the
    recycled free list; after every step in which something finished the pool is compacted (the
    copy kernel moves the displaced blocks in all 43 layers). Every step appends one token per
    sequence and layer and runs the decode attention of all 43 layers."""
    gc.collect()
    lib = ffi.load()
    bs, layers = 64, 43
    block_bytes = bs * ROW_BYTES
    free_bytes, _ = torch.cuda.mem_get_info()
    pool_bytes = min(args.config5_pool_gb * 1e9, free_bytes - 24e9)
    pool_blocks = int(pool_bytes // (layers * block_bytes))
    rng = np.random.default_rng(CONTEXT_SEED + 5)

    def draw():
        return int(min(32768, max(1, round(float(np.exp(rng.normal(math.log(4096.0), 1.0)))))))

    ctxs = [draw() for _ in range(batch)]
    total_steps = steps + warmup
    max_ctx = 32768 + total_steps
    need_blocks = sum(-(-(c + total_steps) // bs) for c in ctxs)
    if pool_blocks < need_blocks + need_blocks // 4:
        return {"skipped": f"only {free_bytes / 1e9:.0f} GB free: a pool of {pool_blocks} blocks per layer is too small"}
    arena = ffi.Arena(ffi.BACKEND_HIP)
    cache = ffi.KvCache(arena, num_layers=layers, block_size=bs, max_context_len=max_ctx, max_batch=batch,
                        pool_blocks=pool_blocks, seed=CONTEXT_SEED, shuffle=1)
    plan = ffi.AttnPlan()
    ffi.check(lib.mlakvAttnPlanInit(batch, heads, max_ctx, bs, ffi.DTYPE_BF16, C.byref(plan)))
    arena.note_workspace(int(plan.workspace_bytes))
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    arena.commit()   # one allocation, zero-filled
    torch.cuda.synchronize()
    commit_seconds = time.perf_counter() - t0
    arena.commit_workspace()
    cache.bind()
    arena.seal()
    view = cache.view()
    # every slot of the pool gets N(0,1) rows, the same rows in every layer (one append call
    # writes a piece of slots into all 43 layers from one source): recycled blocks then hold data
    gen = torch.Generator(device="cuda").manual_seed(11)
    piece = 64 * 1024
    for start in range(0, pool_blocks * bs, piece):
        rows = min(piece, pool_blocks * bs - start)
        x = torch.randn(rows, ROW, generator=gen, device="cuda").to(torch.bfloat16)
        slots = torch.arange(start, start + rows, dtype=torch.int32, device="cuda")
        ffi.check(lib.mlakvAppend(C.byref(view), 0, layers, x.data_ptr(), 0, ROW_BYTES, x.data_ptr() + LATENT * 2, 0, ROW_BYTES,
                                  slots.data_ptr(), rows, stream_ptr(torch)))
        torch.cuda.synchronize()
    for s, n in enumerate(ctxs):
        cache.add_sequence(s, n)
    remaining = [int(v) for v in rng.integers(1, 2 * total_steps, size=batch)]  # steps until the sequence finishes
    qslices = 4
    q = torch.randn(qslices, batch, heads, ROW, generator=gen, device="cuda").to(torch.bfloat16)
    out = torch.empty(batch, heads, LATENT, dtype=torch.bfloat16, device="cuda")
    step_latent = torch.randn(layers, batch, LATENT, generator=gen, device="cuda").to(torch.bfloat16)
    step_rope = torch.randn(layers, batch, ROPE, generator=gen, device="cuda").to(torch.bfloat16)
    allocations_before = arena.device_allocations
    records = []
    for step in range(total_steps):
        finished = [s for s in range(batch) if remaining[s] == 0]
        for s in finished:
            cache.free_sequence(s)
        for s in finished:
            cache.add_sequence(s, draw())
            remaining[s] = int(rng.integers(1, 2 * total_steps))
        ev = [torch.cuda.Event(enable_timing=True) for _ in range(4)]
        ev[0].record()
        moved = len(cache.compact(stream_ptr(torch))) if finished else 0
        ev[1].record()
        cache.append_token_all()
        cache.upload_step(stream_ptr(torch))
        ffi.check(lib.mlakvAppend(C.byref(view), 0, layers, step_latent.data_ptr(), batch * LATENT * 2, LATENT * 2,
                                  step_rope.data_ptr(), batch * ROPE * 2, ROPE * 2, cache.device_slot_mapping, batch,
                                  stream_ptr(torch)))
        ev[2].record()
        for layer in range(layers):
            k = layer % qslices
            ffi.check(lib.mlakvAttnDecode(C.byref(plan), C.byref(view), layer, q[k].data_ptr(), heads * ROW_BYTES, ROW_BYTES,
                                          q[k].data_ptr() + LATENT * 2, heads * ROW_BYTES, ROW_BYTES, cache.device_block_table,
                                          cache.num_blocks, cache.device_seq_lens, 1.0 / math.sqrt(192.0), out.data_ptr(),
                                          heads * LATENT * 2, LATENT * 2, None, arena.workspace, arena.workspace_bytes,
                                          stream_ptr(torch)))
        ev[3].record()
        torch.cuda.synchronize()
        lens = [int(v) for v in cache.host_seq_lens()]
        tokens = sum(lens)
        attention_bytes = layers * (tokens * ROW_BYTES + batch * heads * (ROW + LATENT) * 2 + 4 * sum(-(-n // bs) for n in lens))
        records.append({"finished": len(finished), "moved_blocks": moved, "tokens": tokens,
                        "compaction_ms": ev[0].elapsed_time(ev[1]), "append_ms": ev[1].elapsed_time(ev[2]),
                        "attention_ms": ev[2].elapsed_time(ev[3]), "step_ms": ev[0].elapsed_time(ev[3]),
                        "attention_bytes": attention_bytes, "compaction_bytes": 2 * moved * block_bytes * layers,
                        "append_bytes": layers * batch * (2 * ROW_BYTES + 4)})
        for s in range(batch):
            remaining[s] -= 1
    assert arena.device_allocations == allocations_before, "a step allocated device memory"
    timed = records[warmup:]
    step_ms = sum(r["step_ms"] for r in timed) / len(timed)
    attention_ms = sum(r["attention_ms"] for r in timed) / len(timed)
    attention_bytes = sum(r["attention_bytes"] for r in timed) / len(timed)
    all_bytes = sum(r["attention_bytes"] + r["compaction_bytes"] + r["append_bytes"] for r in timed) / len(timed)
    compactions = [r for r in timed if r["moved_blocks"] > 0]
    stats = cache.stats()
    result = {
        "workload": f"configs[4]: {layers} layers, batch {batch}, ctx lognormal (median 4096, sigma 1.0, cap 32768), block 64, bf16, "
                    f"pool {pool_blocks} blocks per layer = {pool_blocks * layers * block_bytes / 1e9:.1f} GB, seeded finish times, "
                    "recycled blocks, compaction after every step that finished a sequence, decode attention of every layer each step",
        "seed": CONTEXT_SEED + 5, "steps": steps, "warmup": warmup,
        "ms_per_step": step_ms, "attention_ms_per_step": attention_ms, "attention_us_per_layer": attention_ms * 1e3 / layers,
        "gbps": all_bytes / (step_ms * 1e-3) / 1e9,
        "roofline": {"bound": "hbm", "achieved": attention_bytes / (attention_ms * 1e-3) / 1e9, "peak": HBM_PEAK_GBPS, "unit": "GB/s",
                     "frac": attention_bytes / (attention_ms * 1e-3) / 1e9 / HBM_PEAK_GBPS,
                     "traffic": attention_bytes * ATTENTION_TRAFFIC["attention_long"]["ratio"],
                     "traffic_source": "the ratio measured for the attention_long launches (same kernel, same context distribution)",
                     "what": "the 43 attention launches of a step, algorithmic bytes over HIP-event time"},
        "mean_tokens": sum(r["tokens"] for r in timed) / len(timed),
        "finished_sequences": sum(r["finished"] for r in timed),
        "compaction": {"steps_with_compaction": len(compactions),
                       "moved_blocks": sum(r["moved_blocks"] for r in compactions),
                       "bytes": sum(r["compaction_bytes"] for r in compactions),
                       "ms": sum(r["compaction_ms"] for r in compactions),
                       "gbps": (sum(r["compaction_bytes"] for r in compactions) / (sum(r["compaction_ms"] for r in compactions) * 1e-3) / 1e9
                                if compactions else None),
                       "note": "ms covers the host-side plan, the move-list upload and the copy kernel"},
        "arena_commit_seconds": commit_seconds, "arena_bytes": arena.total_bytes,
        "kv_cache_utilization": stats.kv_cache_utilization,
    }
    cache.close()
    arena.close()
    return result


def _threads():
    """One thread per core this process may use, at most 16 (a one-GPU box's CPU share)."""
    try:
        return max(1, min(16, len(os.sched_getaffinity(0))))
    except AttributeError:
        return max(1, min(16, os.cpu_count() or 1))


def cpu_baseline(np, ag):
    """The CPU oracle (a port: the reference has no CPU numerics for this path) on a bounded sample
    of the same workload: the append+gather step of all 43 layers, on one core and with one thread
    per core (layers are independent; the C routines run outside the interpreter lock)."""
    from concurrent.futures import ThreadPoolExecutor

    import oracle_ffi as orc
    bs, batch = 64, len(ag["ctxs"])
    sample_layers = 43
    ctxs = [c + 1 for c in ag["ctxs"]]
    pool = orc.Pool(ag["pool_blocks"], bs, batch, 40, seed=ag["seed"], shuffle=True)
    for s, n in enumerate(ctxs):
        pool.add_sequence(s, n)
    table = pool.table()
    rng = np.random.default_rng(3)
    plane0 = rng.integers(0, 255, size=ag["pool_blocks"] * bs * ROW_BYTES, dtype=np.uint8)
    planes = [plane0.copy() for _ in range(sample_layers)]  # distinct memory per layer, same bytes
    rows = rng.integers(0, 255, size=(sample_layers, batch * ROW_BYTES), dtype=np.uint8)
    slots = np.array([int(table[s, (n - 1) // bs]) * bs + (n - 1) % bs for s, n in enumerate(ctxs)], dtype=np.int32)

    def one_layer(layer):
        orc.append_rows(planes[layer], bs * ROW_BYTES, ROW_BYTES, bs, rows[layer], ROW_BYTES, ROW_BYTES, slots)
        orc.gather_rows(planes[layer], bs * ROW_BYTES, ROW_BYTES, bs, table, ctxs, ROW_BYTES)

    def median_seconds(step, reps):
        times = []
        for _ in range(reps + 1):
            t0 = time.perf_counter()
            step()
            times.append(time.perf_counter() - t0)
        times = sorted(times[1:])
        return times[len(times) // 2]

    nbytes = sample_layers * (2 * sum(ctxs) * ROW_BYTES + 2 * batch * ROW_BYTES)
    single = median_seconds(lambda: [one_layer(layer) for layer in range(sample_layers)], 8)
    threads = _threads()
    with ThreadPoolExecutor(max_workers=threads) as workers:
        multi = median_seconds(lambda: list(workers.map(one_layer, range(sample_layers))), 8)
    return {"value": nbytes / single / 1e9, "unit": "GB/s", "cores": 1, "kind": "port",
            "sample": f"append+gather of {sample_layers} of 43 layers of the same workload (fused 576-element rows), "
                      f"median of 8 runs after one warm-up, host cores visible: {os.cpu_count()}",
            "all_cores": {"value": nbytes / multi / 1e9, "unit": "GB/s", "cores": threads,
                          "sample": "the same step, layers spread over one thread per core"},
            "reference_host_plumbing": {"ms_per_step": REFERENCE_HOST_PLUMBING_MS_PER_STEP,
                                        "what": "host orchestration of the reference's own 43-layer decode step in its mock build "
                                                "(operator launches are no-ops; no KV byte moves), 8 cores of the build container; "
                                                "the reference has no CPU numerics for this path to time"}}


def cpu_attention_baseline(np):
    """Config-3 attention by the CPU oracle (fp32 accumulate): every one of the 32 sequences, on one
    core and with one thread per core (sequences are independent)."""
    from concurrent.futures import ThreadPoolExecutor

    import oracle_ffi as orc
    bs, heads, ctx, batch = 64, 64, 2048, 32
    rng = np.random.default_rng(4)
    blocks = ctx // bs
    orc.bf16_to_f32(np.zeros(1, np.uint16))  # warm the library
    latent_plane = (rng.standard_normal(blocks * bs * LATENT).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)
    rope_plane = (rng.standard_normal(blocks * bs * ROPE).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)
    q_lat = (rng.standard_normal((1, heads, LATENT)).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)
    q_rope = (rng.standard_normal((1, heads, ROPE)).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)
    table = np.arange(blocks, dtype=np.int32).reshape(1, blocks)

    def one_sequence(_):
        orc.mla_decode(q_lat, q_rope, latent_plane, rope_plane, bs, table, [ctx], 1 / math.sqrt(192.0), accum_f32=True)

    t0 = time.perf_counter()
    for b in range(batch):
        one_sequence(b)
    single = time.perf_counter() - t0
    threads = _threads()
    with ThreadPoolExecutor(max_workers=threads) as workers:
        t0 = time.perf_counter()
        list(workers.map(one_sequence, range(batch)))
        multi = time.perf_counter() - t0
    return {"value": single * 1e6, "unit": "us/step", "cores": 1, "kind": "port",
            "sample": "all 32 sequences (64 heads, ctx 2048, fp32 accumulate), one after the other",
            "all_cores": {"value": multi * 1e6, "unit": "us/step", "cores": threads,
                          "sample": "the same 32 sequences spread over one thread per core"}}


def attention_suite(args, torch, np, ffi):
    """The attention configurations: configs[2] (the target shape), configs[3] (FP8 KV, ragged
    contexts with outliers), configs[4]'s decode step for one layer (lognormal contexts), the
    selected-token decode and the indexer that feeds it."""
    out = {}
    out["attention"] = bench_attention(args, torch, np, ffi, [2048] * 32, mx_quant=True, label="configs[2]",
                                       traffic_ratio=ATTENTION_TRAFFIC["attention"])
    out["attention_fp8"] = bench_attention(
        args, torch, np, ffi, draw_contexts(np, "uniform_512_8192", 64, CONTEXT_SEED), fp8=True, iters=64, label="configs[3]",
        distribution="uniform in [512, 8192]", outlier_fraction=0.01,
        traffic_ratio=ATTENTION_TRAFFIC["attention_fp8"])
    out["attention_long"] = bench_attention(
        args, torch, np, ffi, draw_contexts(np, "lognormal_4096_cap_32768", 128, CONTEXT_SEED), slices=2, iters=16,
        label="configs[4] decode attention of one layer", distribution="lognormal (median 4096, sigma 1.0, cap 32768)",
        traffic_ratio=ATTENTION_TRAFFIC["attention_long"])
    # short whole contexts: the launch takes the units of the selected-token attention (every position of the sequence)
    out["attention_short"] = bench_attention(args, torch, np, ffi, [256] * 32, slices=8, label="whole contexts of 256 tokens",
                                             traffic_ratio=ATTENTION_TRAFFIC["attention_short"])
    out["attention_sparse"] = bench_attention(args, torch, np, ffi, [8192] * 32, slices=4, sparse_k=512,
                                              label="selected-token decode (index_topk 512 of 8192)",
                                              traffic_ratio=ATTENTION_TRAFFIC["attention_sparse"])
    out["attention_sparse_fp8"] = bench_attention(args, torch, np, ffi, [8192] * 32, slices=4, sparse_k=512, fp8=True,
                                                  label="selected-token decode over an FP8 cache (index_topk 512 of 8192)",
                                                  traffic_ratio=ATTENTION_TRAFFIC["attention_sparse_fp8"])
    out["indexer"] = bench_indexer(args, torch, np, ffi)
    # The pair as a decode step would run it (indexer, then attention over its selection), against
    # the bytes the pair has to move: B * ctx * 132 of index keys and scales, B * k * 1152 of selected rows.
    pair_us = out["indexer"]["us_per_step"] + out["attention_sparse"]["us_per_step"]
    pair_bytes = 32 * 8192 * 132 + 32 * 512 * ROW_BYTES
    out["indexer_then_attention_sparse"] = {
        "us_per_step": pair_us, "algorithmic_bytes": pair_bytes,
        "roofline": {"bound": "hbm", "achieved": pair_bytes / (pair_us * 1e-6) / 1e9, "peak": HBM_PEAK_GBPS, "unit": "GB/s",
                     "frac": pair_bytes / (pair_us * 1e-6) / 1e9 / HBM_PEAK_GBPS,
                     "traffic": out["indexer"]["roofline"]["traffic"] + out["attention_sparse"]["roofline"]["traffic"],
                     "traffic_source": "the sum of the two records' figures"},
        "what": "sum of the two launches above (each timed back to back on its own), batch 32, ctx 8192, top-512",
    }
    return out


def main():
    args = parse_args()
    if args.gpus != 1:
        sys.stderr.write("bench.py measures one GPU: this path has no multi-GPU leg (sequences shard with no exchange); "
                         "run with --gpus 1\n")
        return 2
    import numpy as np
    import torch

    import mlakv_ffi as ffi
    if not torch.cuda.is_available():
        sys.stderr.write("bench.py needs a GPU: the HIP library has no CPU fallback\n")
        return 3
    torch.cuda.set_device(0)
    # The interpreter's cycle collector stays out of the timed regions (a full collection takes
    # tens of milliseconds with torch loaded and falls wherever an allocation count happens to
    # cross its threshold); it runs between the sections instead.
    gc.disable()
    # A plain 1 GiB device copy of known size: the reference point that scales rocprofv3's
    # FETCH_SIZE / WRITE_SIZE readings for the kernels below.
    calib_src = torch.ones(1 << 30, dtype=torch.uint8, device="cuda")
    calib_dst = torch.empty_like(calib_src)
    calib_dst.copy_(calib_src)
    torch.cuda.synchronize()
    # The same copy, timed: what a device-to-device copy of the runtime reaches on this GPU, the
    # measured ceiling the roofline fractions (quoted against the published 8 TB/s) can be read
    # against. 2 GiB move per copy; the fastest of five.
    copy_ms = []
    for _ in range(5):
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        start.record()
        calib_dst.copy_(calib_src)
        end.record()
        end.synchronize()
        copy_ms.append(start.elapsed_time(end))
    copy_ceiling_gbps = 2 * (1 << 30) / (min(copy_ms) * 1e-3) / 1e9
    del calib_src, calib_dst
    if args.side_only:
        print(json.dumps({"side_kernels": bench_side_kernels(args, torch, np, ffi)}))
        return 0
    if args.attention_only:
        print(json.dumps(attention_suite(args, torch, np, ffi)))
        return 0
    if args.config5_only:
        print(json.dumps({"config5": bench_config5(args, torch, np, ffi)}))
        return 0
    draws = [bench_append_gather(args, torch, np, ffi, seed) for seed in HEADLINE_SEEDS]
    ag = min(draws, key=lambda d: d["value"])   # the slowest draw is the one reported
    line = {
        "metric": "paged-KV append+gather GB/s; MLA decode attn us/step (% HBM roofline)",
        "value": ag["value"], "unit": "GB/s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": ag["ms_per_step"], "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
        "dtype": "bf16", "data": "synthetic",
        "config": {"workload": "configs[1]: paged append+gather, 43 layers, batch 32, ctx uniform [128,2048] "
                               f"(mean {ag['mean_ctx']:.0f} in the timed steps), block 64, seeded-shuffled free list, bf16 rows "
                               "of 576 elements, 1 row appended per sequence per layer then full-context gather into "
                               + ("separate latent/rope planes" if args.split_out else "contiguous 576-element rows"),
                   "bytes_per_step": ag["bytes_per_step"], "frac_of_hbm_peak": ag["value"] / HBM_PEAK_GBPS,
                   "context_seed": ag["seed"],
                   "context_draws": [{"seed": d["seed"], "initial_mean_ctx": d["initial_mean_ctx"], "mean_ctx_timed": d["mean_ctx"],
                                      "value_gbps": d["value"], "frac_of_hbm_peak": d["value"] / HBM_PEAK_GBPS,
                                      "ms_per_step": d["ms_per_step"], "gather_kernel_frac": d["gather_gbps"] / HBM_PEAK_GBPS}
                                     for d in draws],
                   "value_is": "the lowest of the context draws listed (each: W warm-up steps, then K timed steps)"},
        "measured_copy_ceiling": {"gbps": copy_ceiling_gbps, "frac_of_hbm_peak": copy_ceiling_gbps / HBM_PEAK_GBPS,
                                  "how": "device-to-device copy of 1 GiB by the runtime (2 GiB moved), fastest of 5",
                                  "value_over_ceiling": ag["value"] / copy_ceiling_gbps,
                                  "gather_kernel_over_ceiling": ag["gather_gbps"] / copy_ceiling_gbps},
        "roofline": {"bound": "hbm", "achieved": ag["gather_gbps"], "peak": HBM_PEAK_GBPS, "unit": "GB/s",
                     "frac": ag["gather_gbps"] / HBM_PEAK_GBPS,
                     "traffic": ag["gather_bytes_per_launch"] * GATHER_TRAFFIC_PER_ALGORITHMIC_BYTE,
                     "traffic_source": "rocprofv3 --pmc FETCH_SIZE x2.000 + WRITE_SIZE x1.000 per gather dispatch of this "
                                       "command, applied as a ratio to the algorithmic bytes of the timed launches",
                     "kernel": "GatherBf16TileKernel",
                     "avg_launch_ms": ag["gather_ms"], "algorithmic_bytes_per_launch": ag["gather_bytes_per_launch"]},
        "append": {"avg_launch_ms": ag["append_ms"], "achieved_gbps": ag["append_gbps"],
                   "note": "interval between 64 back-to-back launches of the 32-row x 43-layer append (2.9 MB): "
                           "bound by the launch rate, the kernel itself runs about 4 us in the rocprofv3 trace"},
    }
    if not args.no_attention:
        line.update(attention_suite(args, torch, np, ffi))
        line["side_kernels"] = bench_side_kernels(args, torch, np, ffi)
        line["config5"] = bench_config5(args, torch, np, ffi)
    if not args.no_cpu_baseline:
        line["cpu_baseline"] = cpu_baseline(np, ag)
        if not args.no_attention:
            line["attention"]["cpu_baseline"] = cpu_attention_baseline(np)
    print(json.dumps(line))
    return 0


if __name__ == "__main__":
    sys.exit(main())
