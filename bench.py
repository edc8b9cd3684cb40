"""W4A4 linear-layer benchmark on one MI355X.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--workload prefill]

A step is one W4A4 linear over one batch of synthetic activations with the
weights pre-packed:  fused block-Hadamard rotate + per-token int4 quantize +
pack  ->  packed-int4 GEMM on the int8 matrix cores with the fp16 dequant
epilogue.  Default workload: M=2048 tokens, K=N=4096 (the prefill shape),
X ~ N(0,1) fp16 with 1% outlier channels x50, W ~ N(0,0.02), H_128 rotation.

Inputs are resident in HBM before timing starts; the activation batch cycles
through enough distinct buffers (> 256 MiB) that the Infinity Cache cannot
serve them.  Steps are replayed from HIP graphs holding up to 64 consecutive
steps each, timed with a host clock between two device synchronizations.  Per-kernel durations
come from HIP events recorded on the launch stream around runs of back-to-back
launches of that kernel alone.

Prints one JSON line (see README / the driver contract).  `value` is the
whole step's throughput in TOPS (2*M*N*K ops per step / step time);
`roofline` is the GEMM kernel against the dense int8 MFMA peak (against HBM
bandwidth for the skinny-M kernel, M <= 16); `kernels` also carries the
quantize kernel against HBM bandwidth; `cpu_baseline` is
the reference's fake-quant forward (core/linear.py:48-52) restated in torch
and timed on this host's CPU cores.
"""
from __future__ import annotations

import argparse
import json
import math
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "W4A4 GEMM TOPS & fused-quant GB/s vs MI355X roofline, M=2048 K=N=4096"
PEAK_INT8_TOPS = 5000.0      # MI355X dense int8 MFMA, published
PEAK_HBM_GBS = 8000.0        # MI355X HBM3E, published
MALL_BYTES = 256 << 20

WORKLOADS = {
    # name: (M, N, K, rotate_block)
    "prefill": (2048, 4096, 4096, 128),
    "mlp_up": (512, 11008, 4096, 128),
    "mlp_down": (512, 4096, 11008, 128),
    "70b_qo": (4096, 8192, 8192, 128),
    "70b_up": (4096, 28672, 8192, 128),
    "70b_down": (4096, 8192, 28672, 128),
    # small-batch MLP down projection (128 tokens): few 64x128 tiles over a
    # long K, split over workgroups through dscq_matmul_ws
    "down_b128": (128, 4096, 11008, 128),
    # SiLU-gated MLP block (Llama-7B shapes): x[M,K] -> gate|up GEMM [M, 2N] ->
    # silu*up + rotate + quantize -> down GEMM [M, K]
    "mlp": (512, 11008, 4096, 128),
    # decode: one fused launch (dscq_linear_decode) per step where it applies
    # (M * K / 128 <= 128), else quantize + the skinny-M GEMM; the packed weights
    # cycle through more than the Infinity Cache, so they stream from HBM
    "decode1": (1, 4096, 4096, 128),
    "decode4": (4, 4096, 4096, 128),
    "decode8": (8, 4096, 4096, 128),
    "decode16": (16, 4096, 4096, 128),
    "decode1_up": (1, 11008, 4096, 128),
    "decode4_up": (4, 11008, 4096, 128),
    "decode8_up": (8, 11008, 4096, 128),
    "decode16_up": (16, 11008, 4096, 128),
}


def parse():
    p = argparse.ArgumentParser()
    p.add_argument("--gpus", type=int, default=1)
    p.add_argument("--steps", type=int, default=200)
    p.add_argument("--warmup", type=int, default=20)
    p.add_argument("--workload", default="prefill", choices=sorted(WORKLOADS))
    p.add_argument("--kernel-iters", type=int, default=100)
    p.add_argument("--cpu-seconds", type=float, default=10.0,
                   help="budget of the CPU baseline sample")
    p.add_argument("--warm-seconds", type=float, default=2.0,
                   help="run the workload's steps back to back this long before timing anything "
                        "(from idle the GPU takes a few hundred milliseconds to reach its "
                        "steady clock)")
    p.add_argument("--gemm-kernel", choices=("auto", "wide", "pipe", "wide256", "wide128"),
                   default="auto",
                   help="dense GEMM kernel (dscq_set_gemm_kernel): the automatic choice, the "
                        "wide-tile kernel wherever it applies (with the automatic tile width, "
                        "or 256 x 256 / 256 x 128 tiles), or never the wide-tile kernel")
    p.add_argument("--no-cpu", action="store_true")
    p.add_argument("--no-graph", action="store_true")
    p.add_argument("--kernels-only", action="store_true",
                   help="launch only the quantize kernel, the GEMM and a 16 MiB device copy "
                        "(--kernel-iters each), for rocprofv3 --pmc passes")
    p.add_argument("--vendor-int8", action="store_true",
                   help="context only: time the vendor library's int8 GEMM (torch._int_mm, "
                        "hipBLASLt) and fp16 matmul at the prefill and 70B shapes")
    p.add_argument("--traffic", nargs=2, metavar=("FETCH_CSV", "WRITE_CSV"),
                   help="turn two rocprofv3 --pmc counter_collection.csv files of a "
                        "--kernels-only run (FETCH_SIZE, WRITE_SIZE) into HBM bytes per launch, "
                        "calibrated on the copy kernel; prints the JSON block kept under profiles/")
    p.add_argument("--counters", metavar="COUNTER_CSV",
                   help="summarize one rocprofv3 --pmc counter_collection.csv of a --kernels-only "
                        "run of --workload (SQ_VALU_MFMA_BUSY_CYCLES, SQ_BUSY_CYCLES, "
                        "SQ_INSTS_VALU, SQ_INSTS_MFMA, SQ_WAVES): MFMA busy fraction, shader "
                        "clock and VALU instructions per activation element, as JSON")
    return p.parse_args()


def synthetic(M, N, K, seed=0):
    import torch
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(M, K, generator=g)
    idx = torch.randperm(K, generator=torch.Generator().manual_seed(seed + 2))[:math.ceil(0.01 * K)]
    x[:, idx] *= 50
    w = torch.randn(N, K, generator=torch.Generator().manual_seed(seed + 1)) * 0.02
    return x.half(), w.half()


def time_kernel(launch, n, torch, dev):
    """Average device time of one launch: n back-to-back launches captured in a
    HIP graph and timed with HIP events around its replay on the current
    stream (the stream the kernels are launched on).  The graph removes the
    host launch gaps, so the figure matches a profiler's kernel durations."""
    s = torch.cuda.Stream(device=dev)
    s.wait_stream(torch.cuda.current_stream(dev))
    with torch.cuda.stream(s):
        launch(0)
    torch.cuda.current_stream(dev).wait_stream(s)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        for i in range(n):
            launch(i)
    g.replay()
    torch.cuda.synchronize()
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    start.record()
    g.replay()
    end.record()
    end.synchronize()
    return start.elapsed_time(end) / n * 1e-3  # seconds


def time_in_steps(kernels, n, torch, lead=512):
    """Average device duration of each kernel of a step, over n eager steps that
    run the kernels in the mix the timed steps run them in (a GEMM right after a
    quantize kernel) rather than a hundred launches of one kernel back to back,
    whose sustained power draw lowers the clock.  Each launch stamps its own
    start and end into a pair of HIP events on its stream (dscq_time_next_kernel:
    hipExtLaunchKernel), so the figure is the kernel's duration as a kernel trace
    reports it, without the event markers and dispatch gaps that events recorded
    around a call would add (~2 us per interval on this platform)."""
    from dscquant_amd import _lib
    L = _lib.lib()
    nk = len(kernels)
    evs = [[(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True))
            for _ in range(nk)] for _ in range(n)]
    for row in evs:  # torch creates the HIP events on their first record
        for start, end in row:
            start.record()
            end.record()
    torch.cuda.synchronize()
    # A lead of untimed steps keeps the GPU busy while the host queues the timed
    # ones, as in the graph-replayed steps.
    for i in range(lead):
        for fn in kernels:
            fn(i)
    for i in range(n):
        for k, fn in enumerate(kernels):
            start, end = evs[i][k]
            L.dscq_time_next_kernel(start.cuda_event, end.cuda_event)
            fn(i)
    torch.cuda.synchronize()
    return [sum(evs[i][k][0].elapsed_time(evs[i][k][1]) for i in range(n)) / n * 1e-3
            for k in range(nk)]


def warm_up(step, seconds, torch):
    """Runs step(0), step(1), ... back to back for about `seconds`.  From idle the
    GPU needs a few hundred milliseconds of sustained work to reach its steady
    clock: the first few hundred GEMM launches of a fresh process run up to ~20%
    slower than the ones after them."""
    if seconds <= 0:
        return
    t_end = time.perf_counter() + seconds
    i = 0
    while time.perf_counter() < t_end:
        for _ in range(32):
            step(i)
            i += 1
        torch.cuda.synchronize()


COPY_BYTES = 16 << 20


def probes(torch, dev):
    """Launchers of the measurement probes (include/dscq.h): a streaming kernel
    with a kernel's own byte shape, and the MFMAs of a GEMM with no memory
    traffic.  The ceilings reported beside the kernels they bound."""
    from dscquant_amd import _lib
    L = _lib.lib()
    sink = torch.empty(4096, dtype=torch.int32, device=dev)

    def stream(src, read_bytes, dst, write_bytes, pieces):
        rc = L.dscq_stream_probe(src.data_ptr(), read_bytes,
                                 (dst if dst is not None else sink).data_ptr(), write_bytes,
                                 pieces, _lib.stream(dev))
        assert rc == 0, L.dscq_last_error()

    def mfma(M, N, K):
        """The MFMA count of an M x N x K GEMM (2 M N K / 65536 per 32x32x32 MFMA)
        spread over 256 workgroups of 8 waves; None if it does not divide evenly."""
        total = M * N * K // 32768
        if (M * N * K) % 32768 or total % (2048 * 8):
            return None
        per_wave = total // 2048

        def launch(i):
            rc = L.dscq_mfma_probe(256, 8, per_wave, sink.data_ptr(), _lib.stream(dev))
            assert rc == 0, L.dscq_last_error()
        return launch
    return stream, mfma


def kernel_class(name):
    if "mfma_probe" in name:
        return "mfma_probe"
    if "stream_probe" in name:
        return "stream_probe"
    if "row_quant" in name:
        # template arguments <T, ROT, MODE, ...>: MODE 1 is the weight pre-pack
        args = name.split("row_quant_kernel<", 1)[-1].split(",")
        return "pack" if len(args) > 2 and args[2].strip() == "1" else "quantize"
    if "w4a4_gemm" in name or "w4a4_gemv" in name:  # pipe, wide, general kernels
        return "gemm"
    if "w4a4_decode" in name:
        return "decode"
    if "copy" in name.lower():
        return "copy"
    return None


GEMM_KERNELS = {"auto": 0, "wide": 1, "pipe": 2, "wide256": 3, "wide128": 4}


def gemm_kernel_name(M, N, K, choice, gated=False):
    """The kernel that the library says dscq_matmul_ws takes for an fp16 M x N x K GEMM
    (gated: dscq_matmul_silu_mul with N h columns) under a choice of GEMM_KERNELS; a
    square tile and 256 x 128 by one number."""
    from dscquant_amd import _lib
    L = _lib.lib()
    KP = -(-K // 64) * 64
    before = L.dscq_set_gemm_kernel(GEMM_KERNELS[choice])
    try:
        need = 0 if gated else L.dscq_matmul_workspace_bytes(M, N, KP, 0)
        name = L.dscq_matmul_kernel(M, N, KP, int(gated), 0, 0, None, None, 256, need)
    finally:
        L.dscq_set_gemm_kernel(before)
    return name.decode().replace("<256x256>", "<256>").replace("<256x128>", "<128>")


def gated_kernel_name(M, NH, K, choice):
    return gemm_kernel_name(M, NH, K, choice, gated=True)


def traffic_summary(fetch_csv, write_csv):
    """Mean FETCH_SIZE / WRITE_SIZE (KiB per dispatch) per kernel class, scaled by the
    ratio of bytes a 16 MiB device copy really moves to what the counter reports for it."""
    import csv
    means = {}
    for path, counter in ((fetch_csv, "FETCH_SIZE"), (write_csv, "WRITE_SIZE")):
        acc = {}
        for row in csv.DictReader(open(path)):
            cls = kernel_class(row["Kernel_Name"])
            if cls is None or row["Counter_Name"] != counter:
                continue
            acc.setdefault(cls, []).append(float(row["Counter_Value"]) * 1024.0)
        for cls, v in acc.items():
            if cls == "copy":  # the 16 MiB calibration copies, not small setup copies
                v = [x for x in v if x >= 0.5 * max(v)]
            means.setdefault(cls, {})[counter] = sum(v) / len(v)
    f_fetch = COPY_BYTES / means["copy"]["FETCH_SIZE"]
    f_write = COPY_BYTES / means["copy"]["WRITE_SIZE"]
    out = {"calibration": {"copy_bytes_each_way": COPY_BYTES,
                           "fetch_counter_bytes": round(means["copy"]["FETCH_SIZE"]),
                           "write_counter_bytes": round(means["copy"]["WRITE_SIZE"]),
                           "fetch_factor": round(f_fetch, 4), "write_factor": round(f_write, 4)}}
    for cls in ("quantize", "gemm", "decode"):
        if cls in means:
            fb = means[cls]["FETCH_SIZE"] * f_fetch
            wb = means[cls]["WRITE_SIZE"] * f_write
            out[cls] = {"fetch_bytes": round(fb), "write_bytes": round(wb),
                        "traffic": round(fb) + round(wb)}
    return out


def counter_summary(counter_csv, workload):
    """Per kernel class: mean counters per dispatch and what they give.

    SQ_BUSY_CYCLES is summed over the shader arrays (Array_Count in the agent info
    file beside the CSV), so per array it is the kernel's length in shader clocks:
      clock_ghz       = SQ_BUSY_CYCLES / arrays / dispatch duration
      mfma_busy_frac  = SQ_VALU_MFMA_BUSY_CYCLES / (SIMDs * SQ_BUSY_CYCLES / arrays),
                        the share of the kernel's cycles the MFMA pipes are busy
                        (32 busy cycles per v_mfma_i32_32x32x32_i8 on this chip)
      valu_per_element = (SQ_INSTS_VALU - SQ_INSTS_MFMA) * 64 / (M * K): VALU
                        instructions per activation element and lane (quantize).
    With the wave-state counters (summed over waves, same unit as SQ_WAVE_CYCLES):
      wait_frac       = SQ_WAIT_ANY / SQ_WAVE_CYCLES, the share of the waves' lifetime
                        spent in s_waitcnt / barriers (memory and LDS waits)
      wait_inst_frac  = SQ_WAIT_INST_ANY / SQ_WAVE_CYCLES, waiting to issue (dependencies)
      active_frac     = SQ_ACTIVE_INST_ANY / SQ_WAVE_CYCLES, issuing
      valu_busy_frac  = 4 * SQ_ACTIVE_INST_VALU / (SIMDs * kernel cycles), the share of
                        the kernel's cycles a SIMD issues VALU work (a wave64 VALU
                        instruction occupies the SIMD for 4 cycles).
    """
    import csv
    agent = os.path.join(os.path.dirname(counter_csv),
                         os.path.basename(counter_csv).replace("counter_collection", "agent_info"))
    gpu = [r for r in csv.DictReader(open(agent)) if r["Agent_Type"] == "GPU"][0]
    arrays, simds = int(gpu["Array_Count"]), int(gpu["Simd_Count"])
    acc, dur = {}, {}
    for row in csv.DictReader(open(counter_csv)):
        cls = kernel_class(row["Kernel_Name"])
        if cls not in ("quantize", "gemm", "decode", "mfma_probe", "stream_probe"):
            continue
        acc.setdefault(cls, {}).setdefault(row["Counter_Name"], []).append(
            float(row["Counter_Value"]))
        dur.setdefault(cls, {})[row["Dispatch_Id"]] = (
            int(row["End_Timestamp"]) - int(row["Start_Timestamp"]))
    M, N, K = WORKLOADS[workload][:3]
    out = {"workload": workload, "arrays": arrays, "simds": simds}
    for cls, counters in acc.items():
        mean = {n: sum(v) / len(v) for n, v in counters.items()}
        d_ns = sum(dur[cls].values()) / len(dur[cls])
        entry = {"dispatches": len(dur[cls]), "duration_ns": round(d_ns),
                 "counters": {n: round(v) for n, v in sorted(mean.items())}}
        busy = mean.get("SQ_BUSY_CYCLES")
        if busy:
            cycles = busy / arrays
            entry["kernel_cycles"] = round(cycles)
            entry["clock_ghz"] = round(cycles / d_ns, 3)
            if mean.get("SQ_VALU_MFMA_BUSY_CYCLES"):
                entry["mfma_busy_frac"] = round(mean["SQ_VALU_MFMA_BUSY_CYCLES"] / (simds * cycles), 4)
        waves = mean.get("SQ_WAVE_CYCLES")
        if waves:
            for key, name in (("wait_frac", "SQ_WAIT_ANY"), ("wait_inst_frac", "SQ_WAIT_INST_ANY"),
                              ("active_frac", "SQ_ACTIVE_INST_ANY")):
                if name in mean:
                    entry[key] = round(mean[name] / waves, 4)
        if busy and "SQ_ACTIVE_INST_VALU" in mean:
            entry["valu_busy_frac"] = round(4 * mean["SQ_ACTIVE_INST_VALU"] / (simds * busy / arrays), 4)
        if cls == "quantize" and "SQ_INSTS_VALU" in mean:
            entry["valu_per_element"] = round(
                (mean["SQ_INSTS_VALU"] - mean.get("SQ_INSTS_MFMA", 0.0)) * 64 / (M * K), 2)
        out[cls] = entry
    return out


def load_traffic(workload):
    """The traffic block committed for this workload, or None."""
    import re
    path = os.path.join(ROOT, "profiles", f"traffic_{workload}.md")
    if not os.path.exists(path):
        return None
    m = re.search(r"```json\n(.*?)\n```", open(path).read(), re.S)
    return json.loads(m.group(1)) if m else None


def cpu_model():
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def cpu_threads():
    """Threads for the CPU baseline: every core this process may use.  A GPU
    box's share of its host is set by OMP_NUM_THREADS and the CPU affinity
    mask, which can be fewer than os.cpu_count() reports for the whole host."""
    host = os.cpu_count() or 1
    try:
        allowed = len(os.sched_getaffinity(0))
    except (AttributeError, OSError):
        allowed = host
    limit = allowed
    env = os.environ.get("OMP_NUM_THREADS", "")
    if env.isdigit() and int(env) > 0:
        limit = min(limit, int(env))
    share = (f"all {host} host cores" if limit == host else
             f"this process's share: {limit} of {host} host cores "
             f"(affinity {allowed}, OMP_NUM_THREADS={env or 'unset'})")
    return limit, share


def cpu_baseline(M, N, K, budget_s):
    """The reference's CPU fake-quant forward on the same workload, median time:
    as the reference runs it (weight re-quantized on every call) and with the
    fake-quantized weight cached, each on half of the time budget."""
    import torch
    from oracle import fakequant
    threads, share = cpu_threads()
    torch.set_num_threads(threads)
    x, w = synthetic(M, N, K)

    def median_time(fn, budget):
        fn()  # warm-up
        times = []
        t_end = time.perf_counter() + budget
        while len(times) < 3 or (time.perf_counter() < t_end and len(times) < 30):
            t0 = time.perf_counter()
            fn()
            times.append(time.perf_counter() - t0)
        return sorted(times)[len(times) // 2], len(times)

    med, n = median_time(lambda: fakequant.forward(x, w, None), budget_s / 2)
    w_hat = fakequant.quantize_weight(w, 4)
    med_c, n_c = median_time(lambda: fakequant.forward(x, w, None, w_hat=w_hat), budget_s / 2)
    ops = 2.0 * M * N * K
    return {
        "value": round(ops / med / 1e12, 4),
        "unit": "TOPS",
        "cores": threads,
        "kind": "port",
        "sample": (f"torch-CPU fake-quant QuantLinear.forward (core/linear.py:48-52), "
                   f"weights re-quantized per call, M={M} N={N} K={K} fp16, "
                   f"median of {n} runs ({med * 1e3:.1f} ms/run) on {threads} threads of "
                   f"{cpu_model()} ({share})"),
        "weights_cached": {"value": round(ops / med_c / 1e12, 4), "unit": "TOPS",
                           "ms_per_run": round(med_c * 1e3, 2), "runs": n_c},
    }


def main():
    args = parse()
    if args.counters:
        print(json.dumps(counter_summary(args.counters, args.workload), indent=1))
        return
    if args.traffic:
        print(json.dumps(traffic_summary(*args.traffic), indent=1))
        return
    if args.vendor_int8:
        return vendor_int8(args.warm_seconds)
    if args.gpus != 1:
        print(f"bench.py measures one GPU; --gpus {args.gpus} is not supported "
              "(the W4A4 path runs on a single MI355X)", file=sys.stderr)
        sys.exit(2)

    import torch
    from dscquant_amd import _lib, w4a4

    _lib.lib().dscq_set_gemm_kernel(GEMM_KERNELS[args.gemm_kernel])
    if args.workload == "mlp":
        return main_mlp(args, torch, _lib, w4a4)
    if args.workload.startswith("decode"):
        return main_decode(args, torch, _lib, w4a4)

    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)
    _lib.require_gfx950(dev)
    M, N, K, rot = WORKLOADS[args.workload]
    MP, KP = (M + 7) // 8 * 8, (K + 63) // 64 * 64
    stream = _lib.stream(dev)

    x, w = synthetic(M, N, K)
    nbuf = max(2, math.ceil(2 * MALL_BYTES / (M * K * 2)))
    xs = [x.to(dev)]
    for i in range(1, nbuf):  # distinct contents, same distribution
        xs.append(xs[0].roll(i, dims=0).contiguous())
    packed_w, sw, sums = w4a4.pack_weight(w.to(dev), 1.0, rot)
    pa = torch.empty((MP, KP // 2), dtype=torch.uint8, device=dev)
    sx = torch.empty((MP,), dtype=torch.float32, device=dev)
    zx = torch.empty((MP,), dtype=torch.int32, device=dev)
    out = torch.empty((M, N), dtype=torch.float16, device=dev)
    torch.cuda.synchronize()

    L = _lib.lib()

    def quantize(xb):
        rc = L.dscq_quantize(xb.data_ptr(), _lib.F16, M, K, 1.0, 1, rot, pa.data_ptr(),
                             sx.data_ptr(), zx.data_ptr(), None, _lib.stream(dev))
        assert rc == 0, L.dscq_last_error()

    # scratch for the K split (0 bytes unless few tiles meet a long K), allocated
    # once, outside the timed region, as a caller of dscq_matmul_ws would
    nws = L.dscq_matmul_workspace_bytes(M, N, KP, 0)
    assert nws >= 0, L.dscq_last_error()
    ws = torch.empty((max(nws, 16),), dtype=torch.uint8, device=dev)

    def gemm():
        rc = L.dscq_matmul_ws(pa.data_ptr(), packed_w.data_ptr(), sx.data_ptr(), zx.data_ptr(),
                              sw.data_ptr(), sums.data_ptr(), None, M, N, KP, 1, 0, 0,
                              out.data_ptr(), None, ws.data_ptr(), nws, _lib.stream(dev))
        assert rc == 0, L.dscq_last_error()

    def step(i):
        quantize(xs[i % nbuf])
        gemm()

    if args.kernels_only:
        # copy sources cycle through more than the 256 MiB Infinity Cache
        srcs = [torch.ones(COPY_BYTES // 2, dtype=torch.float16, device=dev)
                for _ in range(2 * MALL_BYTES // COPY_BYTES + 2)]
        dst = torch.empty_like(srcs[0])
        for i in range(args.kernel_iters):
            quantize(xs[i % nbuf])
        for i in range(args.kernel_iters):
            gemm()
        for i in range(args.kernel_iters):
            dst.copy_(srcs[i % len(srcs)])
        stream_probe, mfma_probe = probes(torch, dev)
        qdst = torch.empty((MP, KP // 2), dtype=torch.uint8, device=dev)
        for i in range(args.kernel_iters):
            stream_probe(xs[i % nbuf], 2 * M * K, qdst, M * K // 2, 4)
        mfma_launch = mfma_probe(M, N, K)
        if mfma_launch:
            for i in range(args.kernel_iters):
                mfma_launch(i)
        torch.cuda.synchronize()
        print(f"kernels-only: {args.kernel_iters} launches each of quantize, gemm, "
              f"{COPY_BYTES >> 20} MiB copy, the quantize-shaped stream probe"
              f"{' and the MFMA probe' if mfma_launch else ''}", flush=True)
        return

    # ---- per-kernel device times (HIP events on the launch stream): inside
    # steps (the roofline figures) and, for reference, back to back
    warm_up(step, args.warm_seconds, torch)
    t_quant, t_gemm = time_in_steps([lambda i: quantize(xs[i % nbuf]), lambda i: gemm()],
                                    args.kernel_iters, torch)
    t_quant_iso = time_kernel(lambda i: quantize(xs[i % nbuf]), args.kernel_iters, torch, dev)
    quantize(xs[0])
    t_gemm_iso = time_kernel(lambda i: gemm(), args.kernel_iters, torch, dev)
    # Ceilings, each timed in the step in place of the kernel it bounds (like
    # the kernels' own in-step figures): a plain streaming kernel moving the
    # quantize's bytes (read x, write M K / 2) between GEMMs, and the GEMM's
    # MFMAs alone (None where the count does not spread evenly) after quantizes.
    stream_probe, mfma_probe = probes(torch, dev)
    qdst = torch.empty((MP, KP // 2), dtype=torch.uint8, device=dev)
    t_copy = None
    if (2 * M * K) % 64 == 0:
        t_copy = time_in_steps(
            [lambda i: stream_probe(xs[i % nbuf], 2 * M * K, qdst, M * K // 2, 4),
             lambda i: gemm()], args.kernel_iters, torch)[0]
    mfma_launch = mfma_probe(M, N, K)
    t_mfma = None
    if mfma_launch:
        t_mfma = time_in_steps([lambda i: quantize(xs[i % nbuf]), mfma_launch],
                               args.kernel_iters, torch)[1]

    # ---- whole steps.  Runs of up to GRAPH_STEPS consecutive steps are captured
    # into one HIP graph each, so the timed region is the GPU's own step time
    # rather than one host launch per kernel.
    GRAPH_STEPS = 64

    def plan(n):
        """Graphs (and their replay counts) that together run exactly n steps."""
        if args.no_graph or n == 0:
            return None
        s = torch.cuda.Stream(device=dev)
        s.wait_stream(torch.cuda.current_stream(dev))
        with torch.cuda.stream(s):
            for i in range(3):  # warm the captured path outside capture
                step(i)
        torch.cuda.current_stream(dev).wait_stream(s)
        torch.cuda.synchronize()
        out = []
        full, rest = divmod(n, GRAPH_STEPS)
        for count, reps in ((GRAPH_STEPS, full), (rest, 1)):
            if count == 0 or reps == 0:
                continue
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g):
                for i in range(count):
                    step(i)
            out.append((g, reps))
        torch.cuda.synchronize()
        return out

    def run(n, graphs):
        if graphs is None:
            for i in range(n):
                step(i)
        else:
            for g, reps in graphs:
                for _ in range(reps):
                    g.replay()

    warm = plan(args.warmup)
    timed = plan(args.steps)
    run(args.warmup, warm)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    run(args.steps, timed)
    torch.cuda.synchronize()
    elapsed = time.perf_counter() - t0
    ms_per_step = elapsed / args.steps * 1e3
    ops = 2.0 * M * N * K
    value = ops / (ms_per_step * 1e-3) / 1e12

    gemm_tops = ops / t_gemm / 1e12
    qbytes = 2 * M * K + M * K // 2 + 8 * M  # read x fp16, write int4 + scale + zero
    quant_gbs = qbytes / t_quant / 1e9
    # The skinny-M kernel (M <= 16) streams the packed weights once: HBM-bound.
    skinny = M <= 16
    gbytes = N * KP // 2 + MP * KP // 2 + 8 * (N + M) + 2 * M * N
    gemm_gbs = gbytes / t_gemm / 1e9
    if skinny:
        gemm_line = {"bound": "hbm", "achieved": round(gemm_gbs, 1), "peak": PEAK_HBM_GBS,
                     "unit": "GB/s", "frac": round(gemm_gbs / PEAK_HBM_GBS, 4),
                     "kernel": "w4a4_gemv_kernel", "avg_us": round(t_gemm * 1e6, 3),
                     "isolated_us": round(t_gemm_iso * 1e6, 3),
                     "bytes_per_launch": gbytes, "tops": round(gemm_tops, 2)}
    else:
        gemm_line = {"bound": "mfma", "achieved": round(gemm_tops, 2), "peak": PEAK_INT8_TOPS,
                     "unit": "TFLOP/s", "frac": round(gemm_tops / PEAK_INT8_TOPS, 4),
                     "kernel": gemm_kernel_name(M, N, K, args.gemm_kernel),
                     "avg_us": round(t_gemm * 1e6, 3),
                     "isolated_us": round(t_gemm_iso * 1e6, 3),
                     "ops_per_launch": ops, "algorithmic_bytes": M * K // 2 + N * K // 2 + 2 * M * N,
                     "mfma_only_us": None if t_mfma is None else round(t_mfma * 1e6, 3),
                     "mfma_only_frac": (None if t_mfma is None else
                                        round(ops / t_mfma / 1e12 / PEAK_INT8_TOPS, 4))}

    traffic = load_traffic(args.workload)
    cpu = None
    if not args.no_cpu:
        cpu = cpu_baseline(M, N, K, args.cpu_seconds)

    result = {
        "metric": METRIC,
        "value": round(value, 2),
        "unit": "TOPS",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms_per_step, 5),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "int4xint4->int32 (int8 MFMA), fp16 in/out",
        "data": "synthetic: X~N(0,1) fp16 with 1% outlier channels x50, W~N(0,0.02), seeded",
        "config": {"workload": f"{args.workload}: W4A4 linear M={M} K={K} N={N}, "
                               f"rotate_block={rot}, pre-packed weights, fp16 out",
                   "M": M, "N": N, "K": K, "rotate_block": rot, "gemm_kernel": args.gemm_kernel,
                   "input_buffers": nbuf, "steps_per_graph": None if args.no_graph else GRAPH_STEPS},
        "roofline": dict(gemm_line, traffic=(traffic["gemm"]["traffic"]
                                             if traffic and "gemm" in traffic else None)),
        "kernels": {
            "quantize": {"bound": "hbm", "achieved": round(quant_gbs, 1), "peak": PEAK_HBM_GBS,
                         "unit": "GB/s", "frac": round(quant_gbs / PEAK_HBM_GBS, 4),
                         "avg_us": round(t_quant * 1e6, 3),
                         "isolated_us": round(t_quant_iso * 1e6, 3), "bytes_per_launch": qbytes,
                         "copy_ceiling_us": None if t_copy is None else round(t_copy * 1e6, 3),
                         "copy_ceiling_frac": (None if t_copy is None else
                                               round(qbytes / t_copy / 1e9 / PEAK_HBM_GBS, 4)),
                         "traffic": (traffic["quantize"]["traffic"]
                                     if traffic and "quantize" in traffic else None)},
            "gemm": gemm_line,
        },
        "cpu_baseline": cpu,
    }
    print(json.dumps(result))


def run_graph_steps(args, torch, dev, step):
    """Whole-step timing: runs of up to 64 steps captured per HIP graph."""
    GRAPH_STEPS = 64
    s = torch.cuda.Stream(device=dev)
    s.wait_stream(torch.cuda.current_stream(dev))
    with torch.cuda.stream(s):
        for i in range(3):
            step(i)
    torch.cuda.current_stream(dev).wait_stream(s)
    torch.cuda.synchronize()

    def plan(n):
        out = []
        full, rest = divmod(n, GRAPH_STEPS)
        for count, reps in ((GRAPH_STEPS, full), (rest, 1)):
            if count and reps:
                g = torch.cuda.CUDAGraph()
                with torch.cuda.graph(g):
                    for i in range(count):
                        step(i)
                out.append((g, reps))
        torch.cuda.synchronize()
        return out

    def run(graphs):
        for g, reps in graphs:
            for _ in range(reps):
                g.replay()

    run(plan(args.warmup))
    timed = plan(args.steps)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    run(timed)
    torch.cuda.synchronize()
    return (time.perf_counter() - t0) / args.steps


def vendor_int8(warm_seconds=2.0):
    """The platform library's dense int8 GEMM (hipBLASLt through torch._int_mm: int8
    operands, int32 result, no int4 unpacking, no epilogue) and fp16 matmul, as a
    reference point for the W4A4 kernel.  B is K-contiguous (the layout the W4A4
    GEMM reads).  Not part of the default run."""
    import torch
    dev = torch.device("cuda:0")
    res = {}
    for M, N, K in ((2048, 4096, 4096), (4096, 8192, 8192)):
        a = torch.randint(-8, 8, (M, K), dtype=torch.int8, device=dev)
        b = torch.randint(-8, 8, (N, K), dtype=torch.int8, device=dev).t()  # [K, N], K-contiguous
        ah, bh = a.half(), b.half()
        for name, fn in (("int8 torch._int_mm", lambda: torch._int_mm(a, b)),
                         ("fp16 matmul", lambda: ah @ bh)):
            warm_up(lambda i: fn(), warm_seconds, torch)  # same warm-up as the W4A4 timings
            times = []
            for _ in range(5):
                s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                s.record()
                for _ in range(50):
                    fn()
                e.record()
                e.synchronize()
                times.append(s.elapsed_time(e) / 50 * 1e3)
            us = sorted(times)[2]
            res[f"{name} {M}x{N}x{K}"] = {"us": round(us, 2),
                                           "TOPS": round(2.0 * M * N * K / us / 1e6, 1)}
    print(json.dumps({"vendor_gemm": res}))


def main_decode(args, torch, _lib, w4a4):
    """Decode-shaped W4A4 linear (a few tokens), against HBM bandwidth.  Where
    the fused kernel applies (dscq_linear_decode: quantize + skinny product in
    one launch) a step is that launch; otherwise a step is quantize + the
    skinny-M GEMM.  The two-launch path is timed beside the fused one."""
    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)
    _lib.require_gfx950(dev)
    M, N, K, rot = WORKLOADS[args.workload]
    MP, KP = (M + 7) // 8 * 8, (K + 63) // 64 * 64
    L = _lib.lib()
    fused_ok = bool(L.dscq_linear_decode_supported(M, K))
    x, w = synthetic(M, N, K)
    wbytes = N * KP // 2
    nw = max(2, math.ceil(2 * MALL_BYTES / wbytes))
    packs = [w4a4.pack_weight(w.to(dev).roll(i, dims=0).contiguous(), 1.0, rot) for i in range(nw)]
    xs = [x.to(dev).roll(i, dims=1).contiguous() for i in range(8)]
    out = torch.empty((M, N), dtype=torch.float16, device=dev)
    pa = torch.empty((MP, KP // 2), dtype=torch.uint8, device=dev)
    sx = torch.empty((MP,), dtype=torch.float32, device=dev)
    zx = torch.empty((MP,), dtype=torch.int32, device=dev)
    torch.cuda.synchronize()

    def ok(rc):
        assert rc == 0, L.dscq_last_error()

    def fused(i):
        pw, sw, sums = packs[i % nw]
        ok(L.dscq_linear_decode(xs[i % 8].data_ptr(), _lib.F16, M, K, 1.0, rot, pw.data_ptr(),
                                sw.data_ptr(), sums.data_ptr(), None, N, 0, out.data_ptr(),
                                _lib.stream(dev)))

    def quantize(i):
        ok(L.dscq_quantize(xs[i % 8].data_ptr(), _lib.F16, M, K, 1.0, 1, rot, pa.data_ptr(),
                           sx.data_ptr(), zx.data_ptr(), None, _lib.stream(dev)))

    def gemv(i):
        pw, sw, sums = packs[i % nw]
        ok(L.dscq_matmul(pa.data_ptr(), pw.data_ptr(), sx.data_ptr(), zx.data_ptr(),
                         sw.data_ptr(), sums.data_ptr(), None, M, N, KP, 1, 0, 0,
                         out.data_ptr(), None, _lib.stream(dev)))

    def two_launch(i):
        quantize(i)
        gemv(i)

    step = fused if fused_ok else two_launch
    if args.kernels_only:
        srcs = [torch.ones(COPY_BYTES // 2, dtype=torch.float16, device=dev)
                for _ in range(2 * MALL_BYTES // COPY_BYTES + 2)]
        dst = torch.empty_like(srcs[0])
        for i in range(args.kernel_iters):
            step(i)
        for i in range(args.kernel_iters):
            dst.copy_(srcs[i % len(srcs)])
        stream_probe, _ = probes(torch, dev)
        for i in range(args.kernel_iters):
            stream_probe(packs[i % nw][0], wbytes, None, 0, 4)
        torch.cuda.synchronize()
        print(f"kernels-only: {args.kernel_iters} steps ("
              f"{'fused decode kernel' if fused_ok else 'quantize + skinny-M GEMM'}), "
              f"{COPY_BYTES >> 20} MiB copy", flush=True)
        return

    warm_up(step, args.warm_seconds, torch)
    t_two = time_kernel(two_launch, args.kernel_iters, torch, dev)
    t_quant, t_gemv = time_in_steps([quantize, gemv], args.kernel_iters, torch)
    t_fused = time_in_steps([fused], args.kernel_iters, torch)[0] if fused_ok else None
    t_fused_iso = time_kernel(fused, args.kernel_iters, torch, dev) if fused_ok else None
    t_step = run_graph_steps(args, torch, dev, step)
    ops = 2.0 * M * N * K
    traffic = load_traffic(args.workload) or {}
    # Ceiling: a bare read of the weight bytes the step streams (the best of
    # 2, 4 or 8 pieces per thread), back to back in a graph.
    stream_probe, _ = probes(torch, dev)
    t_read = min(time_kernel(lambda i, p=p: stream_probe(packs[i % nw][0], wbytes, None, 0, p),
                             args.kernel_iters, torch, dev) for p in (2, 4, 8))

    def hbm_line(kernel, dbytes, t, cls, t_iso=None):
        gbs = dbytes / t / 1e9
        line = {"bound": "hbm", "achieved": round(gbs, 1), "peak": PEAK_HBM_GBS, "unit": "GB/s",
                "frac": round(gbs / PEAK_HBM_GBS, 4), "kernel": kernel,
                "avg_us": round(t * 1e6, 3), "bytes_per_launch": dbytes,
                "traffic": traffic[cls]["traffic"] if cls in traffic else None}
        if t_iso is not None:
            line["isolated_us"] = round(t_iso * 1e6, 3)
        return line

    # skinny GEMM: packed weights + packed activations + sw, sums, sx, zx + out (fp16)
    gemv_line = hbm_line("w4a4_gemv_kernel", wbytes + M * KP // 2 + 8 * N + 8 * M + 2 * M * N,
                         t_gemv, "gemm")
    kernels = {"quantize": {"avg_us": round(t_quant * 1e6, 3)}, "gemv": gemv_line,
               "quantize_then_matmul": {"avg_us": round(t_two * 1e6, 3),
                                        "note": "two launches"}}
    if fused_ok:
        # weights + x (fp16) + sw, sums + out (fp16).  A step is this one launch,
        # so the kernel's time in the timed steps is its time back to back in a
        # graph; eager launches, each a few microseconds of work behind more of
        # host-side call overhead, leave the GPU idling between them (eager_us).
        line = hbm_line("w4a4_decode_kernel", wbytes + 2 * M * K + 8 * N + 2 * M * N,
                        t_fused_iso, "decode")
        line["eager_us"] = round(t_fused * 1e6, 3)
        kernels = {"decode_fused": line, **kernels}
        how = "fused quantize + skinny product (one launch)"
    else:
        line = gemv_line
        how = "quantize + skinny-M GEMM (M * K / 128 > 128: no fused kernel)"
    cpu = None if args.no_cpu else cpu_baseline(M, N, K, args.cpu_seconds)
    result = {
        "metric": METRIC,
        "value": round(ops / t_step / 1e12, 4),
        "unit": "TOPS",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(t_step * 1e3, 5),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "int4xint4->int32 (int8 MFMA), fp16 in/out",
        "data": "synthetic: X~N(0,1) fp16 with 1% outlier channels x50, W~N(0,0.02), seeded",
        "config": {"workload": f"{args.workload}: W4A4 linear M={M} K={K} N={N}, rotate_block="
                               f"{rot}, {how}, {nw} weight sets cycled (HBM-resident)",
                   "M": M, "N": N, "K": K, "rotate_block": rot, "weight_sets": nw},
        "roofline": dict(line, read_ceiling_us=round(t_read * 1e6, 3),
                         read_ceiling_bytes=wbytes,
                         read_ceiling_frac=round(wbytes / t_read / 1e9 / PEAK_HBM_GBS, 4)),
        "kernels": kernels,
        "cpu_baseline": cpu,
    }
    print(json.dumps(result))


def main_mlp(args, torch, _lib, w4a4):
    """The SiLU-gated MLP block: four launches per step (quantize x, gate|up GEMM with
    the SiLU-gated epilogue, quantize h, down GEMM)."""
    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)
    _lib.require_gfx950(dev)
    M, N, K, rot = WORKLOADS["mlp"]
    MP, KP, NKP = (M + 7) // 8 * 8, (K + 63) // 64 * 64, (N + 63) // 64 * 64
    x, wg = synthetic(M, N, K)
    wu = (torch.randn(N, K, generator=torch.Generator().manual_seed(11)) * 0.02).half()
    wd = (torch.randn(K, N, generator=torch.Generator().manual_seed(12)) * 0.02).half()
    nbuf = max(2, math.ceil(2 * MALL_BYTES / (M * K * 2)))
    xs = [x.to(dev)]
    for i in range(1, nbuf):
        xs.append(xs[0].roll(i, dims=0).contiguous())
    pg, swg, sg = w4a4.pack_weight(wg.to(dev), 1.0, 0)
    pu, swu, su = w4a4.pack_weight(wu.to(dev), 1.0, 0)
    il = w4a4.interleave_gate_up
    pgu, swgu, sgu = il(pg, pu), il(swg, swu), il(sg, su)
    pd, swd, sd = w4a4.pack_weight(wd.to(dev), 1.0, rot)
    pa = torch.empty((MP, KP // 2), dtype=torch.uint8, device=dev)
    sx = torch.empty((MP,), dtype=torch.float32, device=dev)
    zx = torch.empty((MP,), dtype=torch.int32, device=dev)
    h = torch.empty((M, N), dtype=torch.float16, device=dev)
    ph = torch.empty((MP, NKP // 2), dtype=torch.uint8, device=dev)
    sh = torch.empty((MP,), dtype=torch.float32, device=dev)
    zh = torch.empty((MP,), dtype=torch.int32, device=dev)
    out = torch.empty((M, K), dtype=torch.float16, device=dev)
    L = _lib.lib()

    def ok(rc):
        assert rc == 0, L.dscq_last_error()

    def quantize(i):
        ok(L.dscq_quantize(xs[i % nbuf].data_ptr(), _lib.F16, M, K, 1.0, 1, 0, pa.data_ptr(),
                           sx.data_ptr(), zx.data_ptr(), None, _lib.stream(dev)))

    def gemm_gu(i):
        ok(L.dscq_matmul_silu_mul(pa.data_ptr(), pgu.data_ptr(), sx.data_ptr(), zx.data_ptr(),
                                  swgu.data_ptr(), sgu.data_ptr(), None, M, N, KP, h.data_ptr(),
                                  _lib.stream(dev)))

    def gated(i):
        ok(L.dscq_quantize(h.data_ptr(), _lib.F16, M, N, 1.0, 1, rot, ph.data_ptr(),
                           sh.data_ptr(), zh.data_ptr(), None, _lib.stream(dev)))

    def gemm_down(i):
        ok(L.dscq_matmul(ph.data_ptr(), pd.data_ptr(), sh.data_ptr(), zh.data_ptr(),
                         swd.data_ptr(), sd.data_ptr(), None, M, K, NKP, 1, 0, 0,
                         out.data_ptr(), None, _lib.stream(dev)))

    def step(i):
        quantize(i)
        gemm_gu(i)
        gated(i)
        gemm_down(i)

    step(0)
    torch.cuda.synchronize()
    warm_up(step, args.warm_seconds, torch)
    names = ("quantize", "gemm_gate_up_silu", "quantize_h", "gemm_down")
    fns = (quantize, gemm_gu, gated, gemm_down)
    t = dict(zip(names, time_in_steps(fns, args.kernel_iters, torch)))
    t_iso = {name: time_kernel(fn, args.kernel_iters, torch, dev) for name, fn in zip(names, fns)}
    sec = run_graph_steps(args, torch, dev, step)
    ops = 2.0 * M * (2 * N) * K + 2.0 * M * K * N
    gu_ops = 2.0 * M * (2 * N) * K
    qbytes = 2 * M * K + M * KP // 2 + 8 * M
    hbytes = 2 * M * N + M * NKP // 2 + 8 * M  # read h fp16, write int4 + meta
    tg = t["gemm_gate_up_silu"]
    line = {"bound": "mfma", "achieved": round(gu_ops / tg / 1e12, 2),
            "peak": PEAK_INT8_TOPS, "unit": "TFLOP/s",
            "frac": round(gu_ops / tg / 1e12 / PEAK_INT8_TOPS, 4),
            "kernel": gated_kernel_name(M, N, K, args.gemm_kernel) + " (gate|up, SiLU-gated epilogue)",
            "avg_us": round(tg * 1e6, 3),
            "isolated_us": round(t_iso["gemm_gate_up_silu"] * 1e6, 3),
            "ops_per_launch": gu_ops, "traffic": None}
    result = {
        "metric": METRIC, "value": round(ops / sec / 1e12, 2), "unit": "TOPS", "n_gpus": 1,
        "steps": args.steps, "warmup": args.warmup, "ms_per_step": round(sec * 1e3, 5),
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
        "dtype": "int4xint4->int32 (int8 MFMA), fp16 in/out",
        "data": "synthetic: X~N(0,1) fp16 with 1% outlier channels x50, W~N(0,0.02), seeded",
        "config": {"workload": f"mlp: SiLU-gated W4A4 MLP block M={M} K={K} N={N}, gate|up as "
                               f"one GEMM writing h = silu(g) * u, rotate_block={rot} on the "
                               f"down projection input",
                   "M": M, "N": N, "K": K, "rotate_block": rot},
        "roofline": line,
        "kernels": {
            "quantize": {"bound": "hbm", "avg_us": round(t["quantize"] * 1e6, 3),
                         "isolated_us": round(t_iso["quantize"] * 1e6, 3),
                         "achieved": round(qbytes / t["quantize"] / 1e9, 1), "unit": "GB/s"},
            "gemm_gate_up_silu": dict(line),
            "quantize_h": {"bound": "hbm", "avg_us": round(t["quantize_h"] * 1e6, 3),
                           "isolated_us": round(t_iso["quantize_h"] * 1e6, 3),
                           "achieved": round(hbytes / t["quantize_h"] / 1e9, 1),
                           "unit": "GB/s"},
            "gemm_down": {"bound": "mfma", "avg_us": round(t["gemm_down"] * 1e6, 3),
                          "isolated_us": round(t_iso["gemm_down"] * 1e6, 3),
                          "achieved": round(2.0 * M * K * N / t["gemm_down"] / 1e12, 2),
                          "unit": "TOPS"},
        },
        "cpu_baseline": None,
    }
    print(json.dumps(result))


if __name__ == "__main__":
    main()
