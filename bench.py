"""Benchmark of the int8 attention path on one MI355X.

python bench.py [--gpus 1] [--steps K] [--warmup W] [--no-cpu] [--no-decode]
python bench.py --profile-pass   (a few launches of every timed kernel and of a plain
                                  copy of known size, for hardware-counter runs)

Headline (the JSON line's value): causal int8 prefill attention, batch 4, 32
heads, seq 8192, head_dim 128, per-head scales, values with 1% of the channels
scaled x8 as activation outliers -- TOPS of algorithmic work (4 * head_dim per
visible query-key pair) with the int8 inputs resident in HBM. One step is one
call of the prefill entry point over the whole batch.

Also reported in the same line: the other prefill workloads (1x32x2048x128 MHA,
1x8x4096x128 GQA 8:1), the int8-KV decode configurations (B64 32q/8kv L4096
contiguous; B128 8q/1kv ragged L in [512, 8192] over a 16-token paged cache) as
GB/s of algorithmic bytes against HBM peak, and the Reef engine's CPU path (its
own functions, compiled from its headers into oracle/_ref) timed on this host's
cores: a bounded sample of the headline workload, the whole 1x32x2048x128
prefill and the whole B64 L4096 decode step.
"""
from __future__ import annotations

import argparse
import ctypes as C
import json
import math
import os
import re
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "prefill int8 attn TOPS (% MFMA peak); decode KV GB/s (% HBM peak)"
PEAK_INT8_TOPS = 5000.0   # MI355X dense int8 matrix peak, TOP/s
PEAK_HBM_GBS = 8000.0     # MI355X HBM3E, GB/s
CPU_THREADS = 16          # host-core share of one GPU on the benchmark machines
PREFILL_WORKLOADS = ["prefill_1x1x128x64", "prefill_1x32x2048x128", "prefill_4x32x8192x128",
                     "prefill_1x8x4096x128_gqa"]


def parse():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=5)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-decode", action="store_true")
    ap.add_argument("--cpu-seconds", type=float, default=16.0,
                    help="approximate budget of the CPU-baseline sample")
    ap.add_argument("--prefill", default="prefill_4x32x8192x128",
                    choices=PREFILL_WORKLOADS,
                    help="headline prefill workload (4x32x8192x128 by default)")
    ap.add_argument("--prefill-other", default="prefill_1x32x2048x128,prefill_1x8x4096x128_gqa",
                    help="further prefill workloads reported beside the headline (comma list)")
    ap.add_argument("--decode", default="decode_b64_l4096,decode_paged_b128_ragged",
                    help="decode workloads to time (comma list of decode_b64_l4096, "
                         "decode_paged_b128_ragged)")
    ap.add_argument("--no-extra", action="store_true",
                    help="skip the W8A8 projection, integer-only head and KV-append lines")
    ap.add_argument("--profile-pass", action="store_true",
                    help="run COPY_LAUNCHES copies of COPY_BYTES, then 3 launches of each "
                         "kernel, and exit (for rocprofv3 --pmc runs)")
    return ap.parse_args()


def timed(torch, launch, steps, warmup):
    """Wall time per launch of exactly `steps` back-to-back launches between
    synchronizations, and the GPU time per launch from two HIP events recorded on
    the launch stream around the same region."""
    for _ in range(warmup):
        launch()
    torch.cuda.synchronize()
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    t0 = time.perf_counter()
    start.record()
    for _ in range(steps):
        launch()
    end.record()
    torch.cuda.synchronize()
    wall_ms = (time.perf_counter() - t0) * 1e3 / steps
    kern_ms = start.elapsed_time(end) / steps
    return wall_ms, kern_ms


def prefill_launcher(torch, reef, cfg, q, k, v, qs, ks, vs, out):
    """Direct C-ABI call with prebuilt arguments (no per-call Python setup)."""
    lib = reef.lib()
    B, Hq, S, D = q.shape
    gran = reef.PER_HEAD if cfg.granularity == 1 else reef.PER_TENSOR
    p = reef.AttentionParams(B, Hq, k.shape[1], S, S, D, 0, 0, cfg.softmax_scale, gran, gran, 0)
    st = lambda t: reef.Strides(t.stride(0), t.stride(1), t.stride(2))  # noqa: E731
    sq, sk, sv, so = st(q), st(k), st(v), st(out)
    args = (C.byref(p), C.c_void_p(q.data_ptr()), C.byref(sq), C.c_void_p(k.data_ptr()),
            C.byref(sk), C.c_void_p(v.data_ptr()), C.byref(sv), C.c_void_p(qs.data_ptr()),
            C.c_void_p(ks.data_ptr()), C.c_void_p(vs.data_ptr()), C.c_void_p(out.data_ptr()),
            C.byref(so))
    # The balanced schedule's workspace: zero-filled once, left zero-filled by every launch.
    ws = reef.prefill_workspace(p, q.device)
    args = args + (C.c_void_p(ws.data_ptr()), ws.numel())
    fn = lib.reef_attention_prefill_int8

    def launch():
        rc = fn(*args, C.c_void_p(torch.cuda.current_stream().cuda_stream))
        if rc != 0:
            raise RuntimeError(f"prefill status {rc}")
    return launch


def quant_launcher(torch, reef, cfg, tensors):
    """The quantization of q, k and v through the C ABI into preallocated outputs, one
    status word checked after the timed launches (the Python wrappers allocate and
    synchronize on their status word per call)."""
    lib = reef.lib()
    status = reef.StatusWord()
    stream = lambda: C.c_void_p(torch.cuda.current_stream().cuda_stream)  # noqa: E731
    calls = []
    for x in tensors:
        q = torch.empty(x.shape, dtype=torch.int8, device=x.device)
        if cfg.granularity == 1:
            B, H, S, D = x.shape
            s = torch.empty(H, dtype=torch.float32, device=x.device)
            st = reef.Strides(x.stride(0), x.stride(1), x.stride(2))
            args = (C.c_void_p(x.data_ptr()), B, H, S, D, C.byref(st), C.c_void_p(q.data_ptr()),
                    C.c_void_p(s.data_ptr()), status.ptr)
            calls.append((lib.reef_quantize_int8_per_head, args, (q, s, st)))
        else:
            s = torch.empty(1, dtype=torch.float32, device=x.device)
            args = (C.c_void_p(x.data_ptr()), x.numel(), C.c_void_p(q.data_ptr()),
                    C.c_void_p(s.data_ptr()), status.ptr)
            calls.append((lib.reef_quantize_int8_per_tensor, args, (q, s)))

    def launch():
        for fn, args, _ in calls:
            rc = fn(*args, stream())
            if rc != 0:
                raise RuntimeError(f"quantize status {rc}")
    launch.check = lambda: status.check("quantize")
    launch.calls = calls
    return launch


def quant_graph_ms(torch, launch, steps=20, warmup=3):
    """GPU time per quantization of q, k and v: the 9 short launches replayed as one
    captured HIP graph (launched one by one, the host's submission of each kernel
    takes longer than the kernel). Every replay's codes and scales are checked
    bit-for-bit against the eager launch first; if capture fails or a replay
    differs, the eager launches are timed instead."""
    launch()
    torch.cuda.synchronize()
    ref = [t.clone() for _, _, keep in launch.calls for t in keep[:2]]
    try:
        g = torch.cuda.CUDAGraph()
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            launch()  # warm the side stream
            torch.cuda.synchronize()
            with torch.cuda.graph(g, stream=s):
                launch()
        torch.cuda.synchronize()
        for _ in range(3):
            for _, _, keep in launch.calls:
                for t in keep[:2]:
                    t.zero_()
            g.replay()
            torch.cuda.synchronize()
            got = [t for _, _, keep in launch.calls for t in keep[:2]]
            if not all(torch.equal(a, b) for a, b in zip(ref, got)):
                raise RuntimeError("graph replay differs from the eager launches")
            launch()  # eager work between replays
            torch.cuda.synchronize()
    except Exception as e:  # noqa: BLE001
        print(f"# quantize graph timing unavailable ({e}); timing eager launches", file=sys.stderr)
        return timed(torch, launch, steps, warmup)[1], "eager launches"
    return timed(torch, g.replay, steps, warmup)[1], "one HIP graph of the launches"


def prefill_setup(torch, reef, W, name):
    """The inputs of prefill workload `name` drawn on the GPU and quantized by the
    library, the fp32 output buffer, and the launch the bench times (the tests of the
    benchmark workloads call this same launch)."""
    cfg = W.CONFIGS[name]
    qf, kf, vf = W.device_prefill_inputs(cfg)
    quantize = reef.quantize_per_head if cfg.granularity == 1 else reef.quantize_per_tensor
    q, qs = quantize(qf)
    k, ks = quantize(kf)
    v, vs = quantize(vf)
    out = torch.empty(q.shape, dtype=torch.float32, device="cuda")
    launch = prefill_launcher(torch, reef, cfg, q, k, v, qs, ks, vs, out)
    return cfg, (qf, kf, vf), (q, k, v, qs, ks, vs), out, launch


def prefill_kernels(torch, cfg):
    """The kernels the entry point's automatic schedule launches for `cfg` (per-tensor
    or per-head scales, a workspace): the packed schedule (a V-image pack, then the
    attention kernel) when head_dim is 128 and there is at least one pair of 256-row
    query tiles per compute unit; the balanced schedule with at most one 128-row
    query tile per compute unit whose heaviest has so many key tiles more than an equal
    share that cutting it pays (a smaller excess with a tile for almost every unit and a
    whole number of units per head); otherwise the split kernel at head_dim 128 and on such small grids, the one-item
    kernel at 64. Each is one launch; the packed kernel splits P into fp16
    hi + lo parts for the heads whose values need it, the others always."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    pairs = ((cfg.seq + 255) // 256 + 1) // 2 * cfg.batch * cfg.q_heads
    if cfg.head_dim == 128 and pairs >= cus:
        return "vt_pack_kernel + prefill_packed_kernel"
    tiles = (cfg.seq + 127) // 128
    items = tiles * cfg.batch * cfg.q_heads
    steps = [(min(128 * (t + 1), cfg.seq) + 63) // 64 for t in range(tiles)]
    share = max(8, sum(steps) * cfg.batch * cfg.q_heads // cus)
    even = 16 * items >= 15 * cus and cus % (cfg.batch * cfg.q_heads) == 0
    line = (11 if even else 20) if cfg.head_dim == 128 else (7 if even else 16)
    if items <= cus and max(steps) - share >= line:
        return "prefill_stream_kernel"
    return "prefill_split_kernel" if cfg.head_dim == 128 or items <= cus else "prefill_kernel"


def bench_prefill(torch, reef, W, name, steps, warmup, with_quant=True):
    cfg, (qf, kf, vf), (q, k, v, qs, ks, vs), out, launch = prefill_setup(torch, reef, W, name)
    quant = None
    if with_quant:
        ql = quant_launcher(torch, reef, cfg, (qf, kf, vf))
        quant_ms, quant_how = quant_graph_ms(torch, ql)
        ql.check()
        quant_bytes = ((q.numel() + k.numel() + v.numel()) * 5
                       + 4 * (qs.numel() + ks.numel() + vs.numel()))
        quant = {"kernels": "per-head quantize of q, k and v (per tensor: block maxima, "
                            "then scales and quantize)",
                 "timing": quant_how, "ms": round(quant_ms, 4),
                 "GB/s": round(quant_bytes / (quant_ms * 1e-3) / 1e9, 1)}
        del ql
    del qf, kf, vf
    wall_ms, kern_ms = timed(torch, launch, steps, warmup)
    if not torch.isfinite(out).all():
        raise RuntimeError("prefill produced non-finite output")
    del out
    return cfg, cfg.algorithmic_ops(), wall_ms, kern_ms, quant, (q, k, v, qs, ks, vs)


def decode_query(torch, reef, cfg, g):
    """The one-token queries [B, Hq, D] of a decode workload, N(0, 1), quantized with
    one scale per query head over the batch (PER_HEAD)."""
    B, Hq, D = cfg.batch, cfg.q_heads, cfg.head_dim
    qf = torch.randn((B, Hq, 1, D), generator=g, device="cuda")
    q, qsc = reef.quantize_per_head(qf)
    return q.view(B, Hq, D), qsc


def decode_contiguous_setup(torch, reef, W, num_splits=0):
    """The B64 32q/8kv L4096 decode workload on the GPU and the launch the bench
    times: returns (cfg, launch, tensors) with tensors = (q, q_scales, k, v_pages,
    k_scales, v_scales, out)."""
    cfg = W.CONFIGS["decode_b64_l4096"]
    g = torch.Generator(device="cuda")
    g.manual_seed(cfg.seed)
    B, Hq, Hkv, D, L = cfg.batch, cfg.q_heads, cfg.kv_heads, cfg.head_dim, cfg.context
    q, qsc = decode_query(torch, reef, cfg, g)
    kf = torch.randn((B, Hkv, L, D), generator=g, device="cuda")
    k, ksc = reef.quantize_rows(kf)
    del kf
    vf = torch.randn((B, Hkv, L, D), generator=g, device="cuda")
    vq, vsc = reef.quantize_rows(vf)
    del vf
    vp = reef.pack_v_pages(vq)
    del vq
    out = torch.empty((B, Hq, D), dtype=torch.float32, device="cuda")
    status = reef.StatusWord()
    p = reef._decode_params(q, L, Hkv, 0, 1 / math.sqrt(D), reef.PER_HEAD, num_splits)
    ws = reef.decode_workspace(p, q.device)

    def launch():
        reef.attention_decode(q, qsc, k, vp, ksc, vsc, None, softmax_scale=1 / math.sqrt(D),
                              q_granularity=reef.PER_HEAD, num_splits=num_splits, workspace=ws,
                              status=status, out=out)
    launch.check = lambda: status.check("decode")
    return cfg, launch, (q, qsc, k, vp, ksc, vsc, out)


def decode_contiguous(torch, reef, W, steps, warmup, num_splits=0):
    cfg, launch, _ = decode_contiguous_setup(torch, reef, W, num_splits)
    wall_ms, kern_ms = timed(torch, launch, steps, warmup)
    launch.check()
    return cfg, cfg.kv_bytes(), wall_ms, kern_ms


def decode_paged_setup(torch, reef, W, pools=3, num_splits=0):
    """The ragged paged B128 8q/1kv decode workload. The pages of one step (about
    150 MB) fit in the 256 MB last-level cache, so successive launches rotate over
    `pools` independent page pools. Returns (cfg, lens, launch, setups, (q,
    q_scales, out)); setups[i] = (k_pages, v_pages, k_scale_pages, v_scale_pages,
    block_table) of pool i, and launch(i) runs on pool i (launch() on the next)."""
    cfg = W.CONFIGS["decode_paged_b128_ragged"]
    B, Hq, Hkv, D = cfg.batch, cfg.q_heads, cfg.kv_heads, cfg.head_dim
    lens = cfg.lengths()
    npages = (lens + 15) // 16
    total = int(npages.sum())
    pool_pages = int(total * cfg.pool_slack) + 1
    max_blocks = cfg.context // 16
    g = torch.Generator(device="cuda")
    g.manual_seed(cfg.seed)
    q, qsc = decode_query(torch, reef, cfg, g)
    setups = []
    for i in range(pools):
        kf = torch.randn((pool_pages, Hkv, 16, D), generator=g, device="cuda")
        kp, ksp = reef.quantize_rows(kf)
        del kf
        vf = torch.randn((pool_pages, Hkv, 16, D), generator=g, device="cuda")
        vq, vsp = reef.quantize_rows(vf)
        del vf
        vp = reef.pack_v_pages(vq.reshape(pool_pages * Hkv * 16, D)).reshape(pool_pages, Hkv, D, 16)
        del vq
        order = np.argsort(W.lcg_states(cfg.seed + 7 + i, pool_pages), kind="stable")
        table = np.zeros((B, max_blocks), np.int32)
        at = 0
        for b in range(B):
            table[b, : npages[b]] = order[at: at + npages[b]]
            at += npages[b]
        setups.append((kp, vp, ksp, vsp, torch.from_numpy(table).cuda()))
    lens_t = torch.from_numpy(lens.astype(np.int32)).cuda()
    out = torch.empty((B, Hq, D), dtype=torch.float32, device="cuda")
    status = reef.StatusWord()
    p = reef._decode_params(q, max_blocks * 16, Hkv, 0, 1 / math.sqrt(D), reef.PER_HEAD,
                            num_splits)
    ws = reef.decode_workspace(p, q.device)
    it = [0]

    def launch(pool=None):
        if pool is None:
            pool = it[0] % pools
            it[0] += 1
        kp, vp, ksp, vsp, table = setups[pool]
        reef.attention_decode_paged(q, qsc, kp, vp, ksp, vsp, table, lens_t,
                                    softmax_scale=1 / math.sqrt(D), q_granularity=reef.PER_HEAD,
                                    num_splits=num_splits, workspace=ws, status=status, out=out)
    launch.check = lambda: status.check("decode paged")
    return cfg, lens, launch, setups, (q, qsc, out)


def decode_paged_ragged(torch, reef, W, steps, warmup, pools=3, num_splits=0):
    cfg, lens, launch, _, _ = decode_paged_setup(torch, reef, W, pools, num_splits)
    wall_ms, kern_ms = timed(torch, launch, steps, warmup)
    launch.check()
    return cfg, cfg.kv_bytes(lens), wall_ms, kern_ms


def bench_extras(torch, reef, W, steps):
    """The paths beside attention, each on a workload of the benchmark's shapes:
    the W8A8 projection of one tensor-parallel rank of a Llama-70B layer (4096
    tokens, 8192 -> (8 + 2 * 1) * 128 features), the integer-only head on the
    1x32x2048x128 causal prefill, and the KV-cache append of a 512-token prompt
    chunk for 64 sequences x 8 KV heads."""
    import ctypes as C
    lib = reef.lib()
    st = lambda: C.c_void_p(torch.cuda.current_stream().cuda_stream)  # noqa: E731
    P = lambda t: C.c_void_p(t.data_ptr())  # noqa: E731
    g = torch.Generator(device="cuda")
    g.manual_seed(11)
    out = {}
    # W8A8 projection
    M, K, N = 4096, 8192, 1280
    x = torch.randn((M, K), generator=g, device="cuda")
    w = torch.randint(-127, 128, (N, K), dtype=torch.int8, device="cuda", generator=g)
    ws = torch.rand(N, device="cuda", generator=g) * 0.01
    y = torch.empty((M, N), device="cuda")
    wsp = torch.empty(lib.reef_linear_w8a8_workspace_bytes(M, K) // 4 + 4, device="cuda")

    def lin():
        rc = lib.reef_linear_w8a8(P(x), M, K, K, P(w), P(ws), None, N, P(y), N, P(wsp),
                                  wsp.numel() * 4, None, st())
        if rc != 0:
            raise RuntimeError(f"linear status {rc}")
    _, lin_ms = timed(torch, lin, steps, 3)
    xq = torch.randint(-127, 128, (M, K), dtype=torch.int8, device="cuda", generator=g)
    xs = torch.rand(M, device="cuda", generator=g) * 0.01

    def gemm():
        rc = lib.reef_gemm_w8a8(P(xq), P(xs), M, K, P(w), P(ws), None, N, P(y), N, None, st())
        if rc != 0:
            raise RuntimeError(f"gemm status {rc}")
    _, gemm_ms = timed(torch, gemm, steps, 3)
    ops = 2 * M * N * K
    out["linear_w8a8"] = {"workload": f"{M} tokens x {K} -> {N} features",
                          "ms": round(lin_ms, 5), "TOPS": round(ops / (lin_ms * 1e-3) / 1e12, 1),
                          "gemm_only_ms": round(gemm_ms, 5),
                          "gemm_only_TOPS": round(ops / (gemm_ms * 1e-3) / 1e12, 1),
                          "frac_int8_peak": round(ops / (gemm_ms * 1e-3) / 1e12 / PEAK_INT8_TOPS, 4)}
    del x, w, y, wsp, xq
    # integer-only head, 1x32x2048x128 causal
    cfg = W.CONFIGS["prefill_1x32x2048x128"]
    qi = torch.randint(-127, 128, (1, 32, 2048, 128), dtype=torch.int8, device="cuda", generator=g)
    ki = torch.randint(-127, 128, (1, 32, 2048, 128), dtype=torch.int8, device="cuda", generator=g)
    vi = torch.randint(-127, 128, (1, 32, 2048, 128), dtype=torch.int8, device="cuda", generator=g)
    # a table of the exp_table() form, round(32768 * e^(-d / 16)); the timing does
    # not depend on its exact entries
    table = torch.from_numpy(
        np.rint(32768.0 * np.exp(-np.arange(256) / 16.0)).astype(np.uint16).view(np.int16)).cuda()
    p = reef.AttentionParams(1, 32, 32, 2048, 2048, 128, 0, 0, 1.0, 1, 1, 0)
    yi = torch.empty_like(qi)

    def ihead():
        rc = lib.reef_attention_int8_integer(C.byref(p), P(qi), None, P(ki), None, P(vi), None, 10,
                                             P(table), 8, P(yi), None, st())
        if rc != 0:
            raise RuntimeError(f"integer head status {rc}")
    _, ih_ms = timed(torch, ihead, max(5, steps // 4), 2)
    iops = cfg.algorithmic_ops()
    out["integer_head"] = {"workload": cfg.name + ", integer-only (int8.hpp)",
                           "ms": round(ih_ms, 5), "TOPS": round(iops / (ih_ms * 1e-3) / 1e12, 1),
                           "note": "three passes over the keys (max, sum, output)"}
    del qi, ki, vi, yi
    # KV append: a 512-token chunk for 64 sequences x 8 KV heads into an 8192-token cache
    B, H, T, D, L = 64, 8, 512, 128, 8192
    kf = torch.randn((B, H, T, D), device="cuda", generator=g)
    vf = torch.randn((B, H, T, D), device="cuda", generator=g)
    kc = torch.empty((B, H, L, D), dtype=torch.int8, device="cuda")
    vc = torch.empty((B, H, L // 16, D, 16), dtype=torch.int8, device="cuda")
    kcs = torch.empty((B, H, L), device="cuda")
    vcs = torch.empty((B, H, L), device="cuda")
    starts = torch.full((B,), 1024, dtype=torch.int32, device="cuda")
    ap = reef.KvAppendParams(B, H, D, T, L)
    sk = reef.Strides(*kf.stride()[:3])
    sv = reef.Strides(*vf.stride()[:3])

    def append():
        rc = lib.reef_kv_append_int8(C.byref(ap), P(kf), C.byref(sk), P(vf), C.byref(sv), P(starts),
                                     P(kc), P(vc), P(kcs), P(vcs), None, None, st())
        if rc != 0:
            raise RuntimeError(f"append status {rc}")
    _, ap_ms = timed(torch, append, steps, 3)
    ab = 2 * B * H * T * (4 * D + D + 4)
    out["kv_append"] = {"workload": f"{T}-token chunk, {B} sequences x {H} KV heads, d {D}",
                        "ms": round(ap_ms, 5), "GB/s": round(ab / (ap_ms * 1e-3) / 1e9, 1),
                        "frac_hbm": round(ab / (ap_ms * 1e-3) / 1e9 / PEAK_HBM_GBS, 4)}
    del kf, vf, kc, vc, kcs, vcs
    # prefill over the cache: a 512-token turn of one sequence, 8 q / 1 KV head, on a
    # paged cache that holds 4096 tokens (the turn's included)
    Hq, Hkv, S, KV = 8, 1, 512, 4096
    pool = KV // 16 + 64
    kp = torch.randint(-127, 128, (pool, Hkv, 16, D), dtype=torch.int8, device="cuda", generator=g)
    vp = torch.randint(-127, 128, (pool, Hkv, D, 16), dtype=torch.int8, device="cuda", generator=g)
    ksp = torch.rand((pool, Hkv, 16), device="cuda", generator=g) * 0.01 + 0.01
    vsp = torch.rand((pool, Hkv, 16), device="cuda", generator=g) * 0.01 + 0.01
    table = torch.randperm(pool, device="cuda", generator=g)[: KV // 16].to(torch.int32)[None]
    qc = torch.randint(-127, 128, (1, Hq, S, D), dtype=torch.int8, device="cuda", generator=g)
    qcs = torch.rand(Hq, device="cuda", generator=g) * 0.01 + 0.01
    cp = reef.AttentionParams(1, Hq, Hkv, S, KV, D, KV - S, 0, 1 / math.sqrt(D), reef.PER_HEAD,
                              reef.PER_TOKEN, 0)
    cws_n = lib.reef_attention_prefill_cache_workspace_bytes(C.byref(cp))
    cws = torch.zeros(cws_n, dtype=torch.uint8, device="cuda")
    yc = torch.empty((1, Hq, S, D), device="cuda")
    qst, yst = reef.Strides(*qc.stride()[:3]), reef.Strides(*yc.stride()[:3])

    def chunk():
        rc = lib.reef_attention_prefill_int8_cache(
            C.byref(cp), P(qc), C.byref(qst), P(qcs), P(kp), P(vp), P(ksp), P(vsp), 0, P(table),
            table.shape[1], pool, P(yc), C.byref(yst), P(cws), cws_n, None, st())
        if rc != 0:
            raise RuntimeError(f"prefill over the cache status {rc}")
    _, ch_ms = timed(torch, chunk, steps, 3)
    pairs = S * (KV - S) + S * (S + 1) // 2
    cops = 4 * D * pairs * Hq
    out["prefill_over_cache"] = {
        "workload": f"{S}-token turn over a {KV}-token paged cache, {Hq}q/{Hkv}kv, d {D}",
        "ms": round(ch_ms, 5), "TOPS": round(cops / (ch_ms * 1e-3) / 1e12, 1),
        "note": "gather of the cached pages + prefill with per-token K/V scales (hi + lo P)"}
    return out


COPY_BYTES = 1 << 30  # the calibration copy reads and writes this many bytes
COPY_LAUNCHES = 3


def copy_calibration(torch):
    """A plain elementwise copy (negation) of COPY_BYTES fp32 bytes: its FETCH_SIZE and
    WRITE_SIZE counters against the known bytes give the scale of those counters."""
    x = torch.ones(COPY_BYTES // 4, dtype=torch.float32, device="cuda")
    y = torch.empty_like(x)
    for _ in range(COPY_LAUNCHES):
        torch.neg(x, out=y)
    torch.cuda.synchronize()


def recorded_traffic(workload):
    """HBM bytes per prefill launch measured by the hardware counters and recorded
    in profiles/ (FETCH_SIZE + WRITE_SIZE, each scaled by the copy calibration)."""
    path = os.path.join(ROOT, "profiles", f"{workload}_hbm_traffic.md")
    try:
        with open(path) as f:
            text = f.read()
    except OSError:
        return None
    m = re.search(r"^traffic_bytes_per_launch:\s*(\d+)", text, re.M)
    return int(m.group(1)) if m else None


def host_cpu():
    """(CPU model name, logical CPUs this process may run on)."""
    model = ""
    try:
        with open("/proc/cpuinfo") as f:
            model = next((l.split(":", 1)[1].strip() for l in f if "model name" in l), "")
    except OSError:
        pass
    try:
        n = len(os.sched_getaffinity(0))
    except AttributeError:
        n = os.cpu_count() or 1
    return model, n


def causal_pairs(r0, rows):
    """Visible query-key pairs of query rows [r0, r0 + rows) of a causal head whose
    first query is key 0 (row i sees keys 0..i)."""
    return rows * (2 * r0 + rows + 1) // 2


def cpu_prefill_rows(oracle, kind, cfg, host, b, h, r0, rows):
    """Query rows [r0, r0 + rows) of head (b, h) through the CPU path (the engine
    computes every key of every row it is given and masks; the oracle skips the
    invisible ones). Returns the algorithmic ops of those rows."""
    q, k, v, qs, ks, vs = host
    S, D = cfg.seq, cfg.head_dim
    kvh = h // (cfg.q_heads // cfg.kv_heads)
    if kind == "reference":
        oracle.ref_attention_int8_head(q[b, h, r0:r0 + rows], k[b, kvh], v[b, kvh],
                                       np.full(rows, qs[h], np.float32),
                                       np.full(S, ks[kvh], np.float32),
                                       np.full(S, vs[kvh], np.float32), r0, 0, cfg.softmax_scale)
    else:
        p = oracle.Problem(1, 1, 1, rows, S, D, query_start=r0, softmax_scale=cfg.softmax_scale)
        oracle.attention_int8(p, q[b:b + 1, h:h + 1, r0:r0 + rows], k[b:b + 1, kvh:kvh + 1],
                              v[b:b + 1, kvh:kvh + 1], qs[h:h + 1], ks[kvh:kvh + 1],
                              vs[kvh:kvh + 1], threads=1)
    return 4 * D * causal_pairs(r0, rows)


def run_jobs(jobs, threads):
    """Runs the callables on `threads` threads (the CPU path is a C call that releases
    the interpreter lock); returns (sum of their results, wall seconds)."""
    from concurrent.futures import ThreadPoolExecutor
    t0 = time.perf_counter()
    if threads == 1:
        total = sum(j() for j in jobs)
    else:
        with ThreadPoolExecutor(threads) as ex:
            total = sum(ex.map(lambda j: j(), jobs))
    return total, time.perf_counter() - t0


def cpu_prefill_sample(oracle, kind, cfg, host, threads, budget_s):
    """A bounded sample of a prefill workload: first one thread on one slice of query
    rows, sized from a short probe to about a quarter of the budget; then `threads`
    slices at once, on different heads, at offsets spread evenly over the causal
    range, sized to about half of it. Returns the record of both."""
    S, H, B = cfg.seq, cfg.q_heads, cfg.batch
    probe_rows = min(S, 32)
    ops, t = run_jobs([lambda: cpu_prefill_rows(oracle, kind, cfg, host, 0, 0, S - probe_rows,
                                                probe_rows)], 1)
    per_row = t / probe_rows  # the engine's time per row does not depend on the row
    rows1 = int(max(1, min(S, budget_s * 0.25 / per_row)))
    ops1, t1 = run_jobs([lambda: cpu_prefill_rows(oracle, kind, cfg, host, 0, 0, S - rows1,
                                                  rows1)], 1)
    rows = int(max(1, min(S, budget_s * 0.5 / per_row)))
    jobs = []
    for i in range(threads):
        head = (i * 7) % (B * H)
        r0 = min(S - rows, (S * i) // threads)
        jobs.append(lambda b=head // H, h=head % H, r0=r0: cpu_prefill_rows(
            oracle, kind, cfg, host, b, h, r0, rows))
    opsn, tn = run_jobs(jobs, threads)
    value = opsn / tn / 1e12
    return {
        "value": value, "unit": "TOPS", "cores": threads, "kind": kind,
        "sample": f"{threads} slices of {rows} query rows (of {S}) of {cfg.name}, one per "
                  f"thread on {threads} threads, offsets spread over the causal range "
                  f"({tn:.1f} s); ops are the algorithmic ops of the rows done",
        "single_thread": {"value": ops1 / t1 / 1e12, "unit": "TOPS", "cores": 1,
                          "sample": f"the last {rows1} query rows of one head ({t1:.1f} s)"},
        "seconds_full_workload_extrapolated": tn * (S * B * H) / (rows * threads),
        "extrapolated_from": "the sample's wall time per row, scaled to every row of every "
                             "head at the same thread count",
    }


def cpu_prefill_full(oracle, kind, cfg, host, threads):
    """Every head of a prefill workload, one job per head on `threads` threads."""
    jobs = [lambda b=b, h=h: cpu_prefill_rows(oracle, kind, cfg, host, b, h, 0, cfg.seq)
            for b in range(cfg.batch) for h in range(cfg.q_heads)]
    ops, t = run_jobs(jobs, threads)
    return {"workload": cfg.name, "value": ops / t / 1e12, "unit": "TOPS", "seconds": t,
            "cores": threads, "kind": kind, "sample": "the whole workload"}


def cpu_decode_full(oracle, kind, cfg, host, threads):
    """Every (sequence, query head) of a contiguous decode step through the CPU path:
    one query row at position L - 1 over the L cached keys of its KV head, per-token
    K/V scales, one scale per query head. GB/s of the step's algorithmic bytes."""
    q, qsc, k, v, ksc, vsc = host
    B, Hq, Hkv, D, L = cfg.batch, cfg.q_heads, cfg.kv_heads, cfg.head_dim, cfg.context
    scale = 1.0 / math.sqrt(D)

    def job(b):
        for h in range(Hq):
            kvh = h // (Hq // Hkv)
            if kind == "reference":
                oracle.ref_attention_int8_head(q[b, h][None], k[b, kvh], v[b, kvh],
                                               np.full(1, qsc[h], np.float32), ksc[b, kvh],
                                               vsc[b, kvh], L - 1, 0, scale)
            else:
                p = oracle.Problem(1, 1, 1, 1, L, D, query_start=L - 1, softmax_scale=scale,
                                   q_granularity=oracle.GRAN_HEAD,
                                   kv_granularity=oracle.GRAN_TOKEN)
                oracle.attention_int8(p, q[b, h][None, None, None], k[b, kvh][None, None],
                                      v[b, kvh][None, None], qsc[h:h + 1], ksc[b, kvh],
                                      vsc[b, kvh], threads=1)
        return 0
    _, t = run_jobs([lambda b=b: job(b) for b in range(B)], threads)
    nbytes = cfg.kv_bytes()
    return {"workload": cfg.name, "value": nbytes / t / 1e9, "unit": "GB/s", "seconds": t,
            "cores": threads, "kind": kind, "sample": "the whole decode step"}


def cpu_decode_paged_full(oracle, kind, cfg, lens, host, threads):
    """Every (sequence, query head) of the ragged paged decode step through the CPU
    path, each sequence's pages gathered into token order first (outside the timed
    region): one query row at position L_b - 1 over its L_b cached keys, per-token
    K/V scales. GB/s of the step's algorithmic bytes."""
    q, qsc, kp, vp, ksp, vsp, table = host
    B, Hq, Hkv, D = cfg.batch, cfg.q_heads, cfg.kv_heads, cfg.head_dim
    scale = 1.0 / math.sqrt(D)
    seqs = []
    for b in range(B):
        L = int(lens[b])
        pages = table[b, : (L + 15) // 16]
        k = kp[pages].transpose(1, 0, 2, 3).reshape(Hkv, -1, D)[:, :L]
        v = vp[pages].transpose(1, 0, 3, 2).reshape(Hkv, -1, D)[:, :L]  # [P, Hkv, D, 16] pages
        ks = ksp[pages].transpose(1, 0, 2).reshape(Hkv, -1)[:, :L]
        vs = vsp[pages].transpose(1, 0, 2).reshape(Hkv, -1)[:, :L]
        seqs.append(tuple(np.ascontiguousarray(x) for x in (k, v, ks, vs)))

    def job(b):
        k, v, ks, vs = seqs[b]
        L = int(lens[b])
        for h in range(Hq):
            kvh = h // (Hq // Hkv)
            if kind == "reference":
                oracle.ref_attention_int8_head(q[b, h][None], k[kvh], v[kvh],
                                               np.full(1, qsc[h], np.float32), ks[kvh], vs[kvh],
                                               L - 1, 0, scale)
            else:
                p = oracle.Problem(1, 1, 1, 1, L, D, query_start=L - 1, softmax_scale=scale,
                                   q_granularity=oracle.GRAN_HEAD,
                                   kv_granularity=oracle.GRAN_TOKEN)
                oracle.attention_int8(p, q[b, h][None, None, None], k[kvh][None, None],
                                      v[kvh][None, None], qsc[h:h + 1], ks[kvh], vs[kvh],
                                      threads=1)
        return 0
    _, t = run_jobs([lambda b=b: job(b) for b in range(B)], threads)
    nbytes = cfg.kv_bytes(lens)
    return {"workload": cfg.name, "value": nbytes / t / 1e9, "unit": "GB/s", "seconds": t,
            "cores": threads, "kind": kind, "sample": "the whole decode step"}


def cpu_baselines(torch, reef, W, cfg, inputs, budget_s):
    """The CPU path on this host: a bounded sample of the headline prefill (the
    record's value), plus the whole 1x32x2048x128 prefill, a bounded sample of the
    1x8q/1kv x4096x128 prefill (extrapolated to the whole workload), the whole B64
    L4096 decode step and the whole ragged paged B128 decode step on the same
    threads."""
    import oracle
    kind = "reference" if oracle.ref_available() else "port"
    model, ncpu = host_cpu()
    threads = max(1, min(CPU_THREADS, ncpu))
    host = tuple(t.cpu().numpy() for t in inputs)
    rec = cpu_prefill_sample(oracle, kind, cfg, host, threads, budget_s)
    rec["host"] = {"cpu_model": model, "logical_cpus": ncpu, "threads_used": threads}
    full = []
    c2, _, t2, _, _ = prefill_setup(torch, reef, W, "prefill_1x32x2048x128")
    full.append(cpu_prefill_full(oracle, kind, c2, tuple(t.cpu().numpy() for t in t2), threads))
    del t2
    c3, _, (q, qsc, k, vp, ksc, vsc, _) = decode_contiguous_setup(torch, reef, W)
    B, Hkv, D, L = c3.batch, c3.kv_heads, c3.head_dim, c3.context
    v_tok = vp.view(B, Hkv, L // 16, D, 16).transpose(3, 4).reshape(B, Hkv, L, D)
    host3 = (q.cpu().numpy(), qsc.cpu().numpy(), k.cpu().numpy(), v_tok.cpu().numpy(),
             ksc.cpu().numpy(), vsc.cpu().numpy())
    del q, qsc, k, vp, ksc, vsc, v_tok
    torch.cuda.empty_cache()
    full.append(cpu_decode_full(oracle, kind, c3, host3, threads))
    del host3
    c5b, lens5, _, setups5, (q5, qsc5, _) = decode_paged_setup(torch, reef, W, pools=1)
    host5 = (q5.cpu().numpy(), qsc5.cpu().numpy()) + tuple(t.cpu().numpy() for t in setups5[0])
    del setups5, q5, qsc5
    torch.cuda.empty_cache()
    full.append(cpu_decode_paged_full(oracle, kind, c5b, lens5, host5, threads))
    del host5
    rec["full_runs"] = full
    c5a, _, t5, _, _ = prefill_setup(torch, reef, W, "prefill_1x8x4096x128_gqa")
    s5 = cpu_prefill_sample(oracle, kind, c5a, tuple(t.cpu().numpy() for t in t5), threads,
                            budget_s / 4)
    del t5
    ops5 = c5a.algorithmic_ops()
    rec["extrapolated_runs"] = [{
        "workload": c5a.name, "value": s5["value"], "unit": "TOPS", "cores": threads,
        "kind": kind, "sample": s5["sample"],
        "seconds_full_workload_extrapolated": ops5 / (s5["value"] * 1e12),
        "extrapolated_from": "the sample's rate in algorithmic ops, applied to the whole "
                             "workload's ops"}]
    return rec


def prefill_record(torch, cfg, ops, wall_ms, kern_ms):
    return {"workload": cfg.name, "kernels": prefill_kernels(torch, cfg),
            "ms_per_step": round(wall_ms, 5), "kernel_ms": round(kern_ms, 5),
            "TOPS": round(ops / (kern_ms * 1e-3) / 1e12, 2),
            "frac_int8_peak": round(ops / (kern_ms * 1e-3) / 1e12 / PEAK_INT8_TOPS, 4)}


def main():
    args = parse()
    if args.gpus != 1:
        print(f"bench.py measures one GPU: this build has no multi-GPU path "
              f"(asked for --gpus {args.gpus}).", file=sys.stderr)
        sys.exit(2)
    import torch

    import reef_amd as reef
    from reef_amd import workloads as W

    reef.lib()
    others = [n for n in args.prefill_other.split(",") if n and n != args.prefill]
    for n in others:
        if n not in PREFILL_WORKLOADS:
            raise SystemExit(f"unknown prefill workload {n}")
    if args.profile_pass:
        copy_calibration(torch)
        for n in [args.prefill] + others:
            bench_prefill(torch, reef, W, n, 3, 1, with_quant=n == args.prefill)
            torch.cuda.empty_cache()
        fns = {"decode_b64_l4096": decode_contiguous, "decode_paged_b128_ragged": decode_paged_ragged}
        for fn in (fns[n] for n in args.decode.split(",") if n):
            fn(torch, reef, W, 3, 1)
        if not args.no_extra:
            bench_extras(torch, reef, W, 3)
        print(json.dumps({"profile_pass": True, "copy_bytes": COPY_BYTES,
                          "copy_launches": COPY_LAUNCHES}), flush=True)
        return
    cfg, ops, wall_ms, kern_ms, quant, inputs = bench_prefill(
        torch, reef, W, args.prefill, args.steps, args.warmup)
    torch.cuda.empty_cache()
    value = ops / (wall_ms * 1e-3) / 1e12
    achieved = ops / (kern_ms * 1e-3) / 1e12
    outliers = (f", {cfg.outlier_fraction:.0%} of channels x{cfg.outlier_gain:g}"
                if cfg.outlier_fraction else "")
    rec = {
        "metric": METRIC,
        "value": round(value, 2),
        "unit": "TOPS",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(wall_ms, 5),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "int8",
        "data": "synthetic: N(0,1) fp32 drawn on the GPU from a fixed seed" + outliers +
                ", quantized per head to int8 by the library before timing",
        "config": {"workload": cfg.name, "batch": cfg.batch, "q_heads": cfg.q_heads,
                   "kv_heads": cfg.kv_heads, "seq_len": cfg.seq, "head_dim": cfg.head_dim,
                   "causal": True, "scales": "per-head"},
        "roofline": {"bound": "mfma", "achieved": round(achieved, 2), "peak": PEAK_INT8_TOPS,
                     "unit": "TFLOP/s", "frac": round(achieved / PEAK_INT8_TOPS, 4),
                     "traffic": recorded_traffic(args.prefill),
                     "traffic_source": f"profiles/{args.prefill}_hbm_traffic.md: rocprofv3 "
                                       "FETCH_SIZE and WRITE_SIZE per call in a separate "
                                       "profiling run of the same kernels, each scaled by "
                                       "what the counter reads for a plain copy of known "
                                       "size; not measured in this run",
                     "kernel": prefill_kernels(torch, cfg),
                     "kernel_ms": round(kern_ms, 5), "algorithmic_ops_per_launch": ops,
                     "timing": "HIP events on the launch stream around the timed launches; "
                               "kernel_ms covers every kernel of one entry-point call"},
        "quantize": quant,
    }
    other = []
    for n in others:
        ocfg, oops, ow, ok, _, _ = bench_prefill(torch, reef, W, n, args.steps, args.warmup,
                                                 with_quant=False)
        other.append(prefill_record(torch, ocfg, oops, ow, ok))
        torch.cuda.empty_cache()
    rec["prefill_other"] = other
    if not args.no_decode:
        dec = []
        fns = {"decode_b64_l4096": decode_contiguous, "decode_paged_b128_ragged": decode_paged_ragged}
        for fn in (fns[n] for n in args.decode.split(",") if n):
            dcfg, nbytes, dwall, dkern = fn(torch, reef, W, max(10, args.steps // 2), 5)
            gbs = nbytes / (dkern * 1e-3) / 1e9
            dec.append({"workload": dcfg.name, "bytes_per_step": nbytes,
                        "ms_per_step": round(dwall, 5), "kernel_ms": round(dkern, 5),
                        "GB/s": round(gbs, 1), "frac_hbm": round(gbs / PEAK_HBM_GBS, 4),
                        "GB/s_wall": round(nbytes / (dwall * 1e-3) / 1e9, 1)})
            torch.cuda.empty_cache()
        rec["decode"] = dec
    if not args.no_extra:
        rec["extra"] = bench_extras(torch, reef, W, max(10, args.steps // 2))
        torch.cuda.empty_cache()
    if not args.no_cpu:
        rec["cpu_baseline"] = cpu_baselines(torch, reef, W, cfg, inputs, args.cpu_seconds)
    else:
        rec["cpu_baseline"] = None
    print(json.dumps(rec), flush=True)


if __name__ == "__main__":
    main()
