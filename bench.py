"""Benchmark of the denoiser step on one MI355X.

Default workload (--config ns): Flux.2-Klein-4B-shaped denoiser (5 double +
20 single blocks, hidden 3072, 24 heads x 128, SwiGLU x3), 1024x1024 image =
64x64 latent tokens of 128 channels (4096 image tokens) + 512 text tokens of
7680 dims, 4-step official schedule, batch 1, random-init bf16 weights,
synthetic inputs. A step = one transformer forward + the Euler update, with
latent, text and weights resident in HBM (captured hipGraph replay + update
kernel). Other configs: c2 (512x512), c3 (2 reference images, 12800 tokens),
c4 (9B-shaped, CFG as batch 2), c5 (Z-Image-Turbo-6B-shaped, 8 NFE), qwen3
(the Qwen3-4B-shaped text encoder at 512 tokens; a "step" is one encode).

Prints one JSON line. `value` is images/s; ms_per_step is per denoise step.
`roofline` is the kernel class with the largest share of the step (the
gate/up projection GEMM with its SwiGLU epilogue, or the flash attention).
Its launch_ms is its average duration inside a step: after the timed steps
one more step runs launch by launch with two HIP events on the library
stream around every launch and the launches issued one after the other (in
the timed steps each single block's gate/up product runs on a side stream
beside its QKV product and attention); the per-kernel table is
`profiled_step` (iris_hip_profile_enable);
back_to_back_launch_ms times the same kernel alone over 30 launches on the
step's resident buffers. `cpu_baseline` times the oracle (C restatement of the reference's
f32 `make blas` path on OpenBLAS) on one block of each kind at the same shape,
extrapolated to a step. With the default workload the line also carries
`other_configs`: c2, c3, c4, c5, qwen3 and vae, each run by this script in a
child process after the default workload is measured (--no-other-configs
skips them).
"""
import argparse
import ctypes
import json
import os
import subprocess
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(ROOT, "tests"))
import iris_testlib as tl  # noqa: E402

METRIC = "ms per denoise step + images/s @4B-shape 1024²; % of bf16 MFMA peak"
PEAK_BF16 = 2.5e15          # MI355X dense bf16 MFMA, FLOP/s
F = ctypes.c_float

CONFIGS = {
    "ns": dict(kind="flux", h=3072, H=24, nd=5, ns=20, td=7680, ih=64, iw=64, T=512, steps=4, refs=[], B=1,
               golden="oracle_4b_ns_sample.npz",
               workload="Flux.2-Klein-4B-shaped denoise, 1024x1024 (4096 img + 512 txt tokens), 4 steps"),
    "c2": dict(kind="flux", h=3072, H=24, nd=5, ns=20, td=7680, ih=32, iw=32, T=512, steps=4, refs=[], B=1,
               workload="Flux.2-Klein-4B-shaped denoise, 512x512 (1024 img + 512 txt tokens), 4 steps"),
    "c3": dict(kind="flux", h=3072, H=24, nd=5, ns=20, td=7680, ih=64, iw=64, T=512, steps=4,
               refs=[(64, 64, 1), (64, 64, 2)], B=1,
               workload="Flux.2-Klein-4B-shaped, 1024x1024 + 2 references (T offsets 1, 2), 12800 tokens"),
    "c4": dict(kind="flux", h=4096, H=32, nd=8, ns=24, td=12288, ih=64, iw=64, T=512, steps=50, refs=[], B=2,
               workload="Flux.2-Klein-9B-base-shaped, 1024x1024, CFG 4.0 as batch 2, 50-step schedule"),
    "qwen3": dict(kind="qwen3", h=2560, inter=9728, H=32, KV=8, layers=36, vocab=151936, seq=512, n_real=512,
                  steps=1, metric="ms per text encode + encodes/s @Qwen3-4B-shape 512 tokens; % of bf16 MFMA peak",
                  unit="encodes/s", data="synthetic (seeded random-init bf16 weights, random token ids)",
                  workload="Qwen3-4B-shaped text encoder, Flux mode (hidden states after layers 8, 17, 26), "
                           "512 tokens"),
    "vae": dict(kind="vae", z=32, lh=64, lw=64, steps=1,
                metric="ms per VAE decode + decodes/s @Flux.2 VAE 1024x1024; % of bf16 MFMA peak",
                unit="images/s", data="synthetic (seeded random-init decoder weights, N(0,1) latent)",
                workload="Flux.2 VAE decoder, 128x64x64 latent -> 1024x1024 RGB (z_channels 32, batch-norm "
                         "denormalization, post_quant_conv, 16384-token bottleneck attention)"),
    "c5": dict(kind="zimage", d=3840, H=30, layers=30, refiners=2, cap_dim=2560, ffn=10240, t_mid=1024, lh=128,
               lw=128, cap=512, steps=8, golden="oracle_zimage_turbo_sample.npz",
               workload="Z-Image-Turbo-6B-shaped S3-DiT, 1024x1024 (4096 img + 512 caption tokens), 8 NFE"),
}


def flux_flops(c):
    """Algorithmic FLOP per step: 2MNK per linear, attention 4 S^2 h (QK^T + PV)."""
    h, mlp, T = c["h"], 3 * c["h"], c["T"]
    I0 = c["ih"] * c["iw"]
    I = I0 + sum(a * b for a, b, _ in c["refs"])
    S = I + T
    blk = 2 * S * h * (3 * h + h + 2 * mlp + mlp) + 4 * S * S * h
    f = (c["nd"] + c["ns"]) * blk
    f += 2 * I * 128 * h + 2 * T * c["td"] * h + 2 * I0 * h * 128
    return f * c["B"]


def zimage_flops(c):
    """Per block 8 S d^2 + 6 S d f + 4 S^2 d: main layers on S = I + caption,
    noise refiners on I, context refiners on the caption; plus embedders."""
    d, f = c["d"], c["ffn"]
    I = (c["lh"] // 2) * (c["lw"] // 2)
    T = c["cap"]

    def blk(S):
        return 8 * S * d * d + 6 * S * d * f + 4 * S * S * d
    return (c["layers"] * blk(I + T) + c["refiners"] * (blk(I) + blk(T))
            + 2 * I * 64 * d + 2 * T * c["cap_dim"] * d + 2 * I * d * 64)


def synth_f32(shape, seed, mean=0.0, std=1.0):
    """Seeded N(mean, std) float32 inputs from the HIP library's own generator
    (iris_synth_fill_f32, include/iris_synth.h): the same values the tests'
    helper draws, without loading anything else."""
    lib = tl.hip()
    lib.iris_synth_fill_f32.argtypes = [tl.FP, ctypes.c_size_t, ctypes.c_uint64, ctypes.c_uint64, ctypes.c_float,
                                        ctypes.c_float]
    n = int(np.prod(shape))
    a = np.empty(n, np.float32)
    lib.iris_synth_fill_f32(tl.fptr(a), n, seed, 0, mean, std)
    return a.reshape(shape)


def lscpu_model():
    """`Model name` as lscpu prints it (run as a child process before the GPU
    is touched), or None."""
    try:
        out = subprocess.run(["lscpu"], capture_output=True, text=True, timeout=10).stdout
    except (OSError, subprocess.SubprocessError):
        return None
    for line in out.splitlines():
        if line.startswith("Model name:"):
            return line.split(":", 1)[1].strip()
    return None


LSCPU_MODEL = None


def host_cpu():
    """(threads, description) of the host cores the CPU baseline runs on: the
    `model name` of /proc/cpuinfo, the online CPU count (nproc) and the
    threads used. One GPU of this machine is allotted 16 host cores, so the
    baseline uses min(the cores this process may run on, 16), or
    IRIS_ORACLE_THREADS when set."""
    model = "unknown CPU"
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                model = line.split(":", 1)[1].strip()
                break
    except OSError:
        pass
    online = os.cpu_count() or 1
    avail = len(os.sched_getaffinity(0)) if hasattr(os, "sched_getaffinity") else online
    threads = int(os.environ.get("IRIS_ORACLE_THREADS", min(avail, 16)))
    if LSCPU_MODEL and LSCPU_MODEL != model:
        model = f"{model} (lscpu: {LSCPU_MODEL})"
    return threads, (f"{model}, nproc {online}, {avail} available to the process, {threads} threads "
                     f"(the 16-core host share of one GPU)")


def time_launches(lib, fn, n=30, warm=3):
    """Average duration of one launch over n back-to-back launches, HIP events on the library stream."""
    for _ in range(warm):
        assert fn() == 0, lib.iris_hip_last_error()
    lib.iris_hip_event_record(2)
    for _ in range(n):
        fn()
    lib.iris_hip_event_record(3)
    assert lib.iris_hip_sync() == 0
    return lib.iris_hip_event_elapsed_ms(2, 3) / n


def kernel_entry(name, ms, flops, per_step, key=None, b2b_ms=None):
    """One kernel class: launch_ms is its average duration inside the step
    (profiled step), b2b_ms over back-to-back launches of it alone."""
    e = {"kernel": name, "key": key, "launch_ms": round(ms, 4), "flop_per_launch": flops,
         "achieved_tflops": round(flops / (ms * 1e-3) / 1e12, 1),
         "frac": round(flops / (ms * 1e-3) / PEAK_BF16, 4), "launches_per_step": per_step,
         "ms_per_step": round(ms * per_step, 3)}
    if b2b_ms is not None:
        e["back_to_back_launch_ms"] = round(b2b_ms, 4)
    return e


def profile_step(lib, step, i):
    """One more step launched kernel by kernel, each launch between two HIP
    events on the library stream (iris_hip_profile_enable): calls and
    durations per (kernel, grid) inside a step."""
    assert lib.iris_hip_profile_enable(1) == 0
    step(i)
    recs = (tl.KernelTime * 256)()
    n = lib.iris_hip_profile_read(recs, 256)
    assert n > 0, lib.iris_hip_last_error()
    assert lib.iris_hip_profile_enable(0) == 0
    rows = [{"kernel": r.kernel.decode(), "grid": r.grid, "calls": r.calls, "avg_ms": round(r.total_ms / r.calls, 4),
             "total_ms": round(r.total_ms, 3)} for r in recs[:n]]
    return sorted(rows, key=lambda r: -r["total_ms"])


def in_step(prof, kernel, grid):
    """Average in-step duration and calls of one (kernel, grid) entry."""
    for r in prof:
        if r["kernel"] == kernel and r["grid"] == grid:
            return r["total_ms"] / r["calls"], r["calls"]
    raise AssertionError(f"{kernel} with grid {grid} not in the profiled step")


def in_step_attn(prof, calls):
    """The attention launches of the profiled step (one block per unit or
    the balanced schedule, whichever the launch took)."""
    for r in prof:
        if r["kernel"].startswith("flash_attn_kernel<") and r["calls"] == calls:
            return r["total_ms"] / r["calls"], r["calls"]
    raise AssertionError(f"no flash_attn_kernel entry with {calls} calls in the profiled step")


def gemm_grid(shapes):
    """Workgroups of one iris_hip_gemm launch over (M, N) problems: 256x256
    tiles, rounded up to whole groups of 8 (one per XCD)."""
    t = sum(-(-m // 256) * -(-n // 256) for m, n in shapes)
    return 8 * -(-t // 8)


GOLDEN = os.path.join(ROOT, "tests", "golden")


def check_vs_golden(got, z0, g, sign, cfg_name):
    """The timed workload's own output against the oracle's sample of it
    (same seeds, same schedule): the final latent after all steps against the
    oracle's Euler trajectory rebuilt from its per-step velocities
    (z += dt * sign * v in float32). Data files only; nothing is run."""
    z = z0.copy()
    sched = g["schedule"]
    for i in range(len(sched) - 1):
        z = z + np.float32(sched[i + 1] - sched[i]) * (np.float32(sign) * g[f"velocity_{i}"])
    rel = float(np.linalg.norm((got - z).astype(np.float64)) / np.linalg.norm(z.astype(np.float64)))
    cos = float(np.dot(got.astype(np.float64), z.astype(np.float64)) /
                (np.linalg.norm(got.astype(np.float64)) * np.linalg.norm(z.astype(np.float64))))
    return {"golden": "tests/golden/" + cfg_name, "steps": len(sched) - 1,
            "final_latent_rel_l2": round(rel, 6), "final_latent_cosine": round(cos, 7),
            "pass": bool(rel <= 1e-2 and cos >= 0.999)}


def golden_for(name):
    path = os.path.join(GOLDEN, name)
    return np.load(path, allow_pickle=False) if os.path.exists(path) else None


def run_flux(lib, c, args):
    t0 = time.time()
    tf = ctypes.c_void_p(lib.iris_transformer_create_synthetic(c["h"], c["H"], c["nd"], c["ns"], c["td"], 128, 3.0,
                                                               2000.0, 20250101))
    assert tf, lib.iris_hip_last_error().decode()
    t_load = time.time() - t0
    I0 = c["ih"] * c["iw"]
    lib.iris_init_noise.argtypes = [ctypes.c_int] * 4 + [ctypes.c_int64]
    zp = lib.iris_init_noise(1, 128, c["ih"], c["iw"], 42)
    z = np.ctypeslib.as_array(ctypes.cast(zp, tl.FP), shape=(128 * I0,)).copy()
    txt = synth_f32((c["B"], c["T"], c["td"]), 7)
    refs_np = [synth_f32((128, rh, rw), 100 + i) for i, (rh, rw, _) in enumerate(c["refs"])]
    refs = (tl.IrisRef * max(1, len(refs_np)))(*[tl.IrisRef(tl.fptr(r), rh, rw, to) for r, (rh, rw, to)
                                                 in zip(refs_np, c["refs"])])
    nref = len(refs_np)
    assert lib.iris_flux_prepare(tf, c["ih"], c["iw"], refs if nref else None, nref, c["T"], c["B"]) == 0
    assert lib.iris_flux_upload(tf, tl.fptr(z), refs if nref else None, tl.fptr(txt)) == 0
    lib.iris_official_schedule.argtypes = [ctypes.c_int, ctypes.c_int]
    sp = lib.iris_official_schedule(c["steps"], I0)
    sched = np.ctypeslib.as_array(ctypes.cast(sp, tl.FP), shape=(c["steps"] + 1,)).copy()
    g_cfg = 4.0 if c["B"] == 2 else 0.0

    def step(i):
        j = i % c["steps"]
        assert lib.iris_flux_step(tf, float(sched[j]), float(sched[j + 1]), g_cfg) == 0, lib.iris_hip_last_error()

    ms_step, wall = timed_steps(lib, step, args)
    prof = profile_step(lib, step, args.warmup + args.steps)
    parity = None
    g = golden_for(c["golden"]) if c.get("golden") else None
    if g is not None:
        # the same workload once more from its noise, all steps, output kept
        # (on the golden's schedule: the reference build's, whose last bit
        # can differ from this host's by the CPU's reciprocal estimate)
        gs = g["schedule"]
        assert np.abs(gs - sched).max() <= 2.4e-7, (gs, sched)
        assert lib.iris_flux_upload(tf, tl.fptr(z), refs if nref else None, None) == 0
        for j in range(c["steps"]):
            assert lib.iris_flux_step(tf, float(gs[j]), float(gs[j + 1]), g_cfg) == 0, lib.iris_hip_last_error()
        got = np.empty_like(z)
        assert lib.iris_flux_download_latent(tf, tl.fptr(got)) == 0, lib.iris_hip_last_error()
        parity = check_vs_golden(got, z, g, 1.0, c["golden"])

    # kernel classes on the step's own resident buffers
    h, mlp, H, B = c["h"], 3 * c["h"], c["H"], c["B"]
    S = I0 + sum(a * b for a, b, _ in c["refs"]) + c["T"]
    S_pad = (S + 63) // 64 * 64
    BS = B * S
    dbuf = {n: lib.iris_flux_device_buffer(tf, n.encode()) for n in ("a", "qkv", "cat", "q", "k", "vt")}
    wdev = tl.Dev(2 * mlp * h * 2)
    wdev.put(tl.to_bf16(synth_f32((2 * mlp * h,), 9, 0, 0.02)))
    P = tl.GemmProblem
    probs = (P * 1)(P(dbuf["a"], wdev.ptr, dbuf["cat"] + h * 2, None, BS, 2 * mlp, h, h, h, h + mlp, 3))
    g_ms = time_launches(lib, lambda: lib.iris_hip_gemm(probs, 1))
    # the joint attention as the step runs it: Q normalised and rotated in the prologue
    wq = tl.Dev.of(np.ones(128, np.float32))
    rc, rs = (lib.iris_flux_device_buffer(tf, n) for n in (b"rope_pair_cos", b"rope_pair_sin"))
    wsb = lib.iris_hip_attention_workspace_bytes()
    aws = tl.Dev(wsb)
    assert lib.iris_hip_memset(aws.ptr, 0, wsb) == 0
    at = tl.AttnArgs(dbuf["qkv"], dbuf["k"], dbuf["vt"], dbuf["cat"], 3 * h, h, S_pad, h + mlp, S, S, H, B,
                     S * 3 * h, S * h, H * 128 * S_pad, S * (h + mlp), 1.0 / np.sqrt(128.0), 0, S, 0, 0, 0, 0, 0,
                     0.0, wq.ptr, wq.ptr, S, 1e-6, rc, rs, aws.ptr, wsb)
    a_ms = time_launches(lib, lambda: lib.iris_hip_attention(ctypes.byref(at)))
    wdev.close()
    wq.close()
    aws.close()
    # the gate/up launches of the single blocks and, when their text and image
    # rows are whole 256-row tiles, of the double blocks (the same M x N x K)
    g_in, g_n = in_step(prof, "gemm_bf16_kernel<0>", gemm_grid([(BS, 2 * mlp)]))
    a_in, a_n = in_step_attn(prof, c["nd"] + c["ns"])
    assert g_n in (c["ns"], c["nd"] + c["ns"]), g_n
    kernels = [kernel_entry("gemm_bf16_kernel: gate/up projection, SwiGLU epilogue", g_in,
                            2.0 * BS * h * 2 * mlp, g_n, f"gemm_gateup_{args.config}", g_ms),
               kernel_entry("flash_attn_kernel: joint attention, head_dim 128", a_in, 4.0 * B * S * S * h, a_n,
                            f"attn_{args.config}", a_ms)]
    lib.iris_transformer_free(tf)
    cfg = {"workload": c["workload"], "hidden": h, "heads": H, "double_blocks": c["nd"], "single_blocks": c["ns"],
           "image_tokens": I0, "reference_tokens": S - I0 - c["T"], "text_tokens": c["T"], "seq": S, "batch": B,
           "steps_per_image": c["steps"]}
    return ms_step, wall, flux_flops(c), kernels, cfg, t_load, prof, parity


def run_zimage(lib, c, args):
    t0 = time.time()
    axes = (ctypes.c_int * 3)(32, 48, 48)
    tf = lib.zi_transformer_create_synthetic(c["d"], c["H"], c["layers"], c["refiners"], c["cap_dim"], 16, 2,
                                             F(256.0), axes, c["ffn"], c["t_mid"], 20250101)
    assert tf, lib.iris_hip_last_error().decode()
    tf = ctypes.c_void_p(tf)
    t_load = time.time() - t0
    lib.iris_init_noise.argtypes = [ctypes.c_int] * 4 + [ctypes.c_int64]
    zp = lib.iris_init_noise(1, 16, c["lh"], c["lw"], 42)
    z = np.ctypeslib.as_array(ctypes.cast(zp, tl.FP), shape=(16 * c["lh"] * c["lw"],)).copy()
    cap = synth_f32((c["cap"], c["cap_dim"]), 7)
    assert lib.zi_prepare(tf, c["lh"], c["lw"], c["cap"]) == 0, lib.iris_hip_last_error()
    assert lib.zi_upload(tf, tl.fptr(z), tl.fptr(cap)) == 0
    I = (c["lh"] // 2) * (c["lw"] // 2)
    lib.iris_zimage_schedule.argtypes = [ctypes.c_int, ctypes.c_int]
    sp = lib.iris_zimage_schedule(c["steps"], I)
    sched = np.ctypeslib.as_array(ctypes.cast(sp, tl.FP), shape=(c["steps"] + 1,)).copy()

    def step(i):
        j = i % c["steps"]
        assert lib.zi_step(tf, float(sched[j]), float(sched[j + 1])) == 0, lib.iris_hip_last_error()

    ms_step, wall = timed_steps(lib, step, args)
    prof = profile_step(lib, step, args.warmup + args.steps)
    parity = None
    g = golden_for(c["golden"]) if c.get("golden") else None
    if g is not None:
        gs = g["schedule"]
        assert np.abs(gs - sched).max() <= 2.4e-7, (gs, sched)
        assert lib.zi_upload(tf, tl.fptr(z), None) == 0
        for j in range(c["steps"]):
            assert lib.zi_step(tf, float(gs[j]), float(gs[j + 1])) == 0, lib.iris_hip_last_error()
        got = np.empty_like(z)
        assert lib.zi_download_latent(tf, tl.fptr(got)) == 0, lib.iris_hip_last_error()
        parity = check_vs_golden(got, z, g, -1.0, c["golden"])

    d, f, H = c["d"], c["ffn"], c["H"]
    S = I + c["cap"]
    S_pad = (S + 63) // 64 * 64
    dbuf = {n: lib.zi_device_buffer(tf, n.encode()) for n in ("a", "qkv", "cat")}
    wdev = tl.Dev(2 * f * d * 2)
    wdev.put(tl.to_bf16(synth_f32((2 * f * d,), 9, 0, 0.02)))
    P = tl.GemmProblem
    prob = (P * 1)(P(dbuf["a"], wdev.ptr, dbuf["cat"], None, S, 2 * f, d, d, d, f, 3))
    g_ms = time_launches(lib, lambda: lib.iris_hip_gemm(prob, 1))
    wdev.close()
    q, k, vt, o = (tl.Dev(S * d * 2), tl.Dev(S * d * 2), tl.Dev(H * 128 * S_pad * 2), tl.Dev(S * d * 2))
    for b in (q, k, vt):
        b.put(tl.to_bf16(synth_f32((b.n // 2,), 11)))
    wsb = lib.iris_hip_attention_workspace_bytes()
    aws = tl.Dev(wsb)
    assert lib.iris_hip_memset(aws.ptr, 0, wsb) == 0
    at = tl.AttnArgs(q.ptr, k.ptr, vt.ptr, o.ptr, d, d, S_pad, d, S, S, H, 1, 0, 0, 0, 0, 1.0 / np.sqrt(128.0),
                     0, S, 0, 0)
    at.ws, at.ws_bytes = aws.ptr, wsb
    a_ms = time_launches(lib, lambda: lib.iris_hip_attention(ctypes.byref(at)))
    for b in (q, k, vt, o, aws):
        b.close()
    g_in, g_n = in_step(prof, "gemm_bf16_kernel<0>", gemm_grid([(S, 2 * f)]))
    a_in, a_n = in_step_attn(prof, c["layers"])
    assert g_n == c["layers"], g_n
    kernels = [kernel_entry("gemm_bf16_kernel: FFN w1/w3 (SwiGLU epilogue)", g_in, 2.0 * S * d * 2 * f, g_n,
                            f"gemm_ffn_{args.config}", g_ms),
               kernel_entry("flash_attn_kernel: unified attention, head_dim 128", a_in, 4.0 * S * S * d, a_n,
                            f"attn_{args.config}", a_ms)]
    lib.zi_transformer_free(tf)
    cfg = {"workload": c["workload"], "dim": d, "heads": H, "layers": c["layers"], "refiners": c["refiners"],
           "image_tokens": I, "caption_tokens": c["cap"], "seq": S, "batch": 1, "steps_per_image": c["steps"]}
    return ms_step, wall, zimage_flops(c), kernels, cfg, t_load, prof, parity


TRAFFIC_FILE = os.path.join(ROOT, "profiles", "traffic_rocprof_pmc.md")


def measured_traffic(key):
    """HBM-side bytes per launch of a kernel class, from the committed
    FETCH_SIZE / WRITE_SIZE counter runs (lines `traffic <key>: <bytes>`), or
    None when that class has not been measured."""
    if not key or not os.path.exists(TRAFFIC_FILE):
        return None
    for line in open(TRAFFIC_FILE):
        line = line.strip().strip("`")
        if line.startswith(f"traffic {key}:"):
            return float(line.split(":", 1)[1])
    return None


def probe(kind, n):
    """Launch one kernel class n times on synthetic NS-shaped buffers (the
    program that the counter runs profile): `gemm` = the gate/up
    projection GEMM, `attn` = the joint attention, `rownorm` = the AdaLN
    row pass, `kvprep` = K RMSNorm + RoPE and the V transpose, `copy` = a 1 GiB
    device-to-device copy (the calibration kernel of known size)."""
    lib = tl.hip()
    c = CONFIGS["ns"]
    h, H, mlp = c["h"], c["H"], 3 * c["h"]
    S = c["ih"] * c["iw"] + c["T"]
    S_pad = (S + 63) // 64 * 64
    bufs = []

    def dev(nbytes, seed=None, scale=1.0):
        d = tl.Dev(nbytes)
        if seed is not None:
            d.put(tl.to_bf16(synth_f32((nbytes // 2,), seed, 0, scale)))
        bufs.append(d)
        return d.ptr

    if kind == "gemm":
        # gate/up rows of the single block's first linear, SwiGLU epilogue into cat[:, h:]
        a, w = dev(S * h * 2, 3), dev(2 * mlp * h * 2, 9, 0.02)
        cat = dev(S * (h + mlp) * 2)
        P = tl.GemmProblem
        probs = (P * 1)(P(a, w, cat + h * 2, None, S, 2 * mlp, h, h, h, h + mlp, 3))
        fn = lambda: lib.iris_hip_gemm(probs, 1)  # noqa: E731
        alg = 2 * S * h + 2 * 2 * mlp * h + 2 * S * mlp
    elif kind == "attn":
        q, k = dev(S * 3 * h * 2, 11), dev(S * h * 2, 12)
        vt, o = dev(H * 128 * S_pad * 2, 13), dev(S * (h + mlp) * 2)
        wq = tl.Dev.of(np.ones(128, np.float32))
        ang = np.random.default_rng(5).uniform(-3, 3, (S, 64))
        rc, rs = (tl.Dev.of(f(ang).astype(np.float32)) for f in (np.cos, np.sin))
        bufs.extend([wq, rc, rs])
        wsb = lib.iris_hip_attention_workspace_bytes()
        aws = dev(wsb)
        assert lib.iris_hip_memset(aws, 0, wsb) == 0
        at = tl.AttnArgs(q, k, vt, o, 3 * h, h, S_pad, h + mlp, S, S, H, 1, 0, 0, 0, 0, 1.0 / np.sqrt(128.0), 0, S,
                         0, 0, 0, 0, 0, 0.0, wq.ptr, wq.ptr, S, 1e-6, rc.ptr, rs.ptr, aws, wsb)
        fn = lambda: lib.iris_hip_attention(ctypes.byref(at))  # noqa: E731
        alg = 2 * 4 * S * h + 2 * 64 * 4 * S
    elif kind == "rownorm":
        # the double block's AdaLN: LayerNorm + (1 + scale) x + shift of the f32 residual rows, bf16 out,
        # txt rows with one modulation set, img rows with the other
        x, a = dev(S * h * 4), dev(S * h * 2)
        mods = [tl.Dev.of(synth_f32((h,), 20 + i, 0, 0.1)) for i in range(4)]
        bufs.extend(mods)
        na = tl.NormArgs(x, h, a, h, 1, S, h, 0, 1e-6, c["T"], S, mods[0].ptr, mods[1].ptr, None, mods[2].ptr,
                         mods[3].ptr, None)
        fn = lambda: lib.iris_hip_rownorm(ctypes.byref(na))  # noqa: E731
        alg = S * h * 4 + S * h * 2 + 4 * h * 4
    elif kind == "kvprep":
        # K RMSNorm + RoPE (K-side tables) and the V transpose from the fused QKV rows
        qkv, k = dev(S * 3 * h * 2, 11), dev(S * h * 2)
        vt = dev(H * 128 * S_pad * 2)
        wk = tl.Dev.of(np.ones(128, np.float32))
        ang = np.random.default_rng(5).uniform(-3, 3, (S, 128))
        rc, rs = (tl.Dev.of(f(ang).astype(np.float32)) for f in (np.cos, np.sin))
        bufs.extend([wk, rc, rs])
        qa = tl.QkPrepArgs(qkv, 3 * h, h, 2 * h, None, k, vt, S_pad, S, H, None, wk.ptr, None, wk.ptr, S, rc.ptr,
                           rs.ptr, 0, 1e-6, 0, rc.ptr, rs.ptr)
        fn = lambda: lib.iris_hip_kv_prepare(ctypes.byref(qa))  # noqa: E731
        # K and V columns read, K and V^T written, the K-side tables read
        alg = 2 * S * h * 2 + 2 * S * h * 2 + 2 * S * 128 * 4
    else:
        nb = 1 << 30
        src, dst = dev(nb), dev(nb)
        lib.iris_hip_memcpy_d2d.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t]
        fn = lambda: lib.iris_hip_memcpy_d2d(dst, src, nb)  # noqa: E731
        alg = 2 * nb
    for _ in range(n):
        assert fn() == 0, lib.iris_hip_last_error()
    assert lib.iris_hip_sync() == 0
    print(json.dumps({"probe": kind, "launches": n, "algorithmic_bytes_per_launch": alg}))


def timed_steps(lib, step, args):
    for i in range(args.warmup):
        step(i)
    assert lib.iris_hip_sync() == 0
    lib.iris_hip_event_record(0)
    t1 = time.perf_counter()
    for i in range(args.steps):
        step(i)
    lib.iris_hip_event_record(1)
    assert lib.iris_hip_sync() == 0
    wall = time.perf_counter() - t1
    return lib.iris_hip_event_elapsed_ms(0, 1) / args.steps, wall * 1000 / args.steps


def qwen3_flops(c, layers=27):
    """Per layer 2 S h (q + 2 kv) + 2 S q h + 2 S h 2I + 2 S I h for the
    linears and 2 S^2 d H for causal attention (half of QK^T + PV)."""
    S, h, I = c["seq"], c["h"], c["inter"]
    qd, kd = c["H"] * 128, c["KV"] * 128
    lin = 2 * S * h * (qd + 2 * kd) + 2 * S * qd * h + 2 * S * h * 2 * I + 2 * S * I * h
    return layers * (lin + 2 * S * S * 128 * c["H"])


def run_qwen3(lib, c, args):
    t0 = time.time()
    m = ctypes.c_void_p(lib.qwen3_model_create_synthetic(c["h"], c["inter"], c["H"], c["KV"], c["layers"],
                                                        c["vocab"], 20250101))
    assert m.value, lib.iris_hip_last_error().decode()
    t_load = time.time() - t0
    S = c["seq"]
    rng = np.random.default_rng(1)
    ids = rng.integers(0, c["vocab"], S).astype(np.int32)
    mask = np.zeros(S, np.int32)
    mask[:c["n_real"]] = 1

    def step(i):
        p = lib.qwen3_forward(m, ids.ctypes.data_as(tl.IP), mask.ctypes.data_as(tl.IP), S)
        assert p, lib.iris_hip_last_error()
        ctypes.CDLL(None).free(ctypes.c_void_p(p))

    ms_step, wall = timed_steps(lib, step, args)
    lib.qwen3_model_free(m)
    # the dominant launch, on buffers of its shape: gate/up with the SwiGLU epilogue
    h, I = c["h"], c["inter"]
    a = tl.Dev(S * h * 2)
    a.put(tl.to_bf16(synth_f32((S * h,), 3)))
    w = tl.Dev(2 * I * h * 2)
    w.put(tl.to_bf16(synth_f32((2 * I * h,), 9, 0, 0.02)))
    o = tl.Dev(S * I * 2)
    P = tl.GemmProblem
    pr = (P * 1)(P(a.ptr, w.ptr, o.ptr, None, S, 2 * I, h, h, h, I, 3))
    g_ms = time_launches(lib, lambda: lib.iris_hip_gemm(pr, 1))
    for d in (a, w, o):
        d.close()
    kernels = [kernel_entry("gemm_bf16_kernel: gate/up (SwiGLU epilogue), M 512", g_ms, 2.0 * S * h * 2 * I, 27,
                            "gemm_qwen3_gateup")]
    cfg = {"workload": c["workload"], "hidden": h, "intermediate": I, "heads": c["H"], "kv_heads": c["KV"],
           "layers": c["layers"], "layers_run": 27, "tokens": S, "real_tokens": c["n_real"], "vocab": c["vocab"]}
    return ms_step, wall, qwen3_flops(c), kernels, cfg, t_load, None, None


def cpu_baseline_qwen3(c):
    """Oracle on the host cores: one layer at 512 tokens, extrapolated to 27."""
    orc = tl.oracle()
    threads, host = host_cpu()
    tl.bind_blas(orc, threads)
    m = ctypes.c_void_p(orc.orc_qwen3_create_synth(c["h"], c["inter"], c["H"], c["KV"], 2, 4096, 20250101))
    S = c["seq"]
    ids = np.random.default_rng(1).integers(0, 4096, S).astype(np.int32)
    t0 = time.perf_counter()
    p = orc.orc_qwen3_forward(m, ids.ctypes.data_as(tl.IP), None, S, 0)
    t1 = time.perf_counter() - t0
    tl.take_f32(orc, p, S * c["h"])
    orc.orc_qwen3_free(m)
    ms = t1 * 27 * 1000
    return {"value": round(1000.0 / ms, 6), "unit": "encodes/s", "cores": threads, "kind": "port",
            "ms_per_step": round(ms, 1),
            "sample": f"oracle (C restatement of the reference qwen3_forward, {orc.orc_blas_info().decode()}) on "
                      f"{host}: 1 layer {t1:.2f} s at 512 tokens, hidden {c['h']}, extrapolated x27"}


def vae_flops(c):
    """Algorithmic FLOPs of one decode: 2 P cin cout 9 per 3x3 conv (conv_in
    at its real z input channels), 2 P cin cout per 1x1, and 2 S (3C) C + 4 S^2 C
    + 2 S C C for the bottleneck attention (S pixels at 1/8 resolution)."""
    z, h, w = c["z"], 2 * c["lh"], 2 * c["lw"]
    S = h * w
    f = 2 * S * z * z + 2 * S * z * 512 * 9

    def res(P, ci, co):
        return 2 * P * 9 * (ci * co + co * co) + (2 * P * ci * co if ci != co else 0)

    f += 2 * res(S, 512, 512) + 2 * S * 512 * 1536 + 4 * S * S * 512 + 2 * S * 512 * 512
    P, prev = S, 512
    for level in (3, 2, 1, 0):
        ch = 128 * [1, 2, 4, 4][level]
        f += res(P, prev, ch) + 2 * res(P, ch, ch)
        prev = ch
        if level:
            P *= 4
            f += 2 * P * ch * ch * 9
    return f + 2 * P * 128 * 3 * 9


def run_vae(lib, c, args):
    t0 = time.time()
    v = ctypes.c_void_p(lib.iris_vae_gpu_create_synthetic(c["z"], 0.0, 0.0, 20250101))
    assert v.value, lib.iris_hip_last_error().decode()
    t_load = time.time() - t0
    lh, lw = c["lh"], c["lw"]
    lat = tl.Dev.of(np.random.default_rng(1).standard_normal((4 * c["z"], lh, lw)).astype(np.float32))
    P = 256 * lh * lw
    rgb = tl.Dev(P * 3)

    def step(i):
        assert lib.iris_vae_gpu_decode_device(v, lat.ptr, lh, lw, rgb.ptr, None) == 0, lib.iris_hip_last_error()

    ms_step, wall = timed_steps(lib, step, args)
    lib.iris_vae_gpu_free(v)
    # the 3x3 convolution 256 -> 256 at a quarter of the pixels, with its
    # GroupNorm sums: bf16 out (2 per decode) and added to the f32 stream (2;
    # a third leaves its sum in bf16 only)
    H = W = 8 * lh
    cin = cout = 256
    x = tl.Dev(H * W * cin * 2)
    x.put(tl.to_bf16(synth_f32((H * W * cin,), 3)))
    wt = tl.Dev(cout * 9 * cin * 2)
    wt.put(tl.to_bf16(synth_f32((cout * 9 * cin,), 9, 0, 1.0 / 48)))
    o, part = tl.Dev(H * W * cout * 4), tl.Dev(H * W // 256 * 32 * 16)
    assert lib.iris_hip_memset(o.ptr, 0, H * W * cout * 4) == 0
    lib.iris_hip_conv3x3_tiled.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
    kernels = []
    for epi, key, what in ((1, "conv_256_512", "bf16 out"), (5, "conv_256_512_add", "residual sum")):
        conv = tl.Conv3x3(x.ptr, wt.ptr, o.ptr, None, H, W, cin, cout, 0, cout, epi, 0, None, 0, part.ptr, 32)
        c_ms = time_launches(lib, lambda: lib.iris_hip_conv3x3_tiled(ctypes.byref(conv), None))
        kernels.append(kernel_entry(f"conv3x3_patch_kernel (3x3 conv on pixel tiles): 256->256, 512x512 pixels, {what}",
                                    c_ms, 2.0 * H * W * cin * cout * 9, 2, key))
    for d in (x, wt, o, part, lat, rgb):
        d.close()
    cfg = {"workload": c["workload"], "latent": [4 * c["z"], lh, lw], "image": [16 * lh, 16 * lw],
           "z_channels": c["z"], "bottleneck_tokens": 4 * lh * lw}
    return ms_step, wall, vae_flops(c), kernels, cfg, t_load, None, None


def cpu_baseline_vae(c):
    """Oracle decode of a 256x256 image (16x16 latent) on the host cores,
    scaled to 1024x1024 by the ratio of algorithmic FLOPs."""
    orc = tl.oracle()
    threads, host = host_cpu()
    tl.bind_blas(orc, threads)
    os.environ.setdefault("OMP_NUM_THREADS", str(threads))
    v = ctypes.c_void_p(orc.orc_vae_create_synth(c["z"], 0.0, 0.0, 20250101))
    lh = lw = 16
    lat = np.random.default_rng(1).standard_normal((4 * c["z"], lh, lw)).astype(np.float32)
    rgb = np.zeros(256 * lh * lw * 3, np.uint8)
    t0 = time.perf_counter()
    assert orc.orc_vae_decode(v, tl.fptr(lat), lh, lw, rgb.ctypes.data, None, -1) == 0
    t1 = time.perf_counter() - t0
    orc.orc_vae_free(v)
    scale = vae_flops(c) / vae_flops(dict(c, lh=lh, lw=lw))
    ms = t1 * scale * 1000
    return {"value": round(1000.0 / ms, 6), "unit": "images/s", "cores": threads, "kind": "port",
            "ms_per_step": round(ms, 1),
            "sample": f"oracle (C restatement of the reference iris_vae_decode, OpenMP) on {host}: 256x256 decode "
                      f"{t1:.2f} s, scaled x{scale:.2f} by algorithmic FLOPs to 1024x1024"}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=12)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--config", default="ns", choices=sorted(CONFIGS))
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--probe", choices=["gemm", "attn", "copy", "rownorm", "kvprep"],
                    help="only launch one kernel class a few times (for counter runs)")
    ap.add_argument("--probe-launches", type=int, default=3)
    ap.add_argument("--no-other-configs", action="store_true",
                    help="with the default workload, skip measuring the other workloads in child processes")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py: runs on one GPU; --gpus {args.gpus} is not supported "
              "(sharding across GPUs is designed, not implemented)", file=sys.stderr)
        sys.exit(2)
    if args.probe:
        probe(args.probe, args.probe_launches)
        return
    c = CONFIGS[args.config]
    if not args.no_cpu_baseline:
        global LSCPU_MODEL
        LSCPU_MODEL = lscpu_model()
    lib = tl.hip()
    run = {"flux": run_flux, "zimage": run_zimage, "qwen3": run_qwen3, "vae": run_vae}[c["kind"]]
    ms_step, wall_ms, flops, kernels, cfg, t_load, prof, parity = run(lib, c, args)
    images_per_s = 1000.0 / (ms_step * c["steps"])   # one image per pass (CFG: both branches in one)
    dom = max(kernels, key=lambda k: k["ms_per_step"])
    result = {
        "metric": c.get("metric", METRIC),
        "value": round(images_per_s, 4),
        "unit": c.get("unit", "images/s"),
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms_step, 4),
        "ms_per_image": round(ms_step * c["steps"], 3),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "bf16",
        "data": c.get("data", "synthetic (seeded random-init bf16 weights, N(0,1) text embeddings, "
                              "seeded noise latent)"),
        "config": cfg,
        "step_tflop": round(flops / 1e12, 3),
        "mfma_frac_step": round(flops / (ms_step * 1e-3) / PEAK_BF16, 4),
        "achieved_tflops_step": round(flops / (ms_step * 1e-3) / 1e12, 1),
        "wall_ms_per_step": round(wall_ms, 4),
        "model_create_s": round(t_load, 1),
        "roofline": {"kernel": dom["kernel"], "bound": "mfma", "achieved": dom["achieved_tflops"],
                     "peak": PEAK_BF16 / 1e12, "unit": "TFLOP/s", "frac": dom["frac"],
                     "traffic": measured_traffic(dom["key"]),
                     "launch_ms": dom["launch_ms"], "flop_per_launch": dom["flop_per_launch"]},
        "kernels": kernels,
        "device": lib.iris_hip_device_name().decode(),
    }
    if parity:
        result["parity"] = parity
    if prof:
        # the profiled step: every launch between two events, the launches issued one by one
        result["profiled_step"] = {"kernel_ms": round(sum(r["total_ms"] for r in prof), 3),
                                   "top": prof[:10]}
    if args.config == "ns" and not args.no_other_configs:
        result["other_configs"] = other_configs(args)
    if not args.no_cpu_baseline:
        result["cpu_baseline"] = {"qwen3": cpu_baseline_qwen3, "vae": cpu_baseline_vae}.get(c["kind"], cpu_baseline)(c)
    print(json.dumps(result))


OTHER_CONFIGS = ["c2", "c3", "c4", "c5", "qwen3", "vae"]


def other_configs(args):
    """The other workloads, each measured by this script in a child process
    (`--config X --no-cpu-baseline`, the same steps and warm-up), one after
    the other once the default workload's line is complete, so that a failure
    in one leaves this line and the others intact. Per workload: its metric,
    value and ms per step, the step's MFMA fraction, the dominant kernel in
    the step and, where the workload has a committed golden, its parity."""
    out = {}
    for name in OTHER_CONFIGS:
        t0 = time.time()
        cmd = [sys.executable, os.path.abspath(__file__), "--config", name, "--no-cpu-baseline",
               "--steps", str(args.steps), "--warmup", str(args.warmup)]
        try:
            p = subprocess.run(cmd, capture_output=True, text=True, timeout=150)
            lines = [ln for ln in p.stdout.splitlines() if ln.startswith("{")]
            if p.returncode != 0 or not lines:
                tail = (p.stderr.strip().splitlines() or [""])[-1]
                out[name] = {"error": f"exit status {p.returncode}: {tail[:300]}"}
            else:
                r = json.loads(lines[-1])
                rl = r["roofline"]
                entry = {"value": r["value"], "unit": r["unit"],
                         "ms_per_step": r["ms_per_step"], "mfma_frac_step": r["mfma_frac_step"],
                         "workload": r["config"]["workload"],
                         "roofline": {"kernel": rl["kernel"], "launch_ms": rl["launch_ms"], "frac": rl["frac"]},
                         "kernels": [{"key": k["key"], "launch_ms": k["launch_ms"], "frac": k["frac"]}
                                     for k in r["kernels"]]}
                if r["metric"] != METRIC:
                    entry = {"metric": r["metric"], **entry}
                if "parity" in r:
                    entry["parity"] = r["parity"]
                out[name] = entry
        except subprocess.TimeoutExpired:
            out[name] = {"error": "no result within 150 s"}
        print(f"bench.py: {name} measured in {time.time() - t0:.1f} s", file=sys.stderr, flush=True)
    return out


def cpu_baseline(c):
    """Oracle (C restatement of the reference f32 BLAS path) on the host cores:
    one block of each kind at the benchmark's shape, timed once each,
    extrapolated to one step."""
    orc = tl.oracle()
    threads, host = host_cpu()
    tl.bind_blas(orc, threads)
    if c["kind"] == "zimage":
        return cpu_baseline_zimage(orc, c, threads, host)
    h, T, I0 = c["h"], c["T"], c["ih"] * c["iw"]
    I = I0 + sum(a * b for a, b, _ in c["refs"])
    m = ctypes.c_void_p(orc.orc_flux_create_synth(h, c["H"], 1, 1, c["td"], 128, 3.0, 2000.0, 20250101))
    ic, is_ = np.zeros(I * 128, np.float32), np.zeros(I * 128, np.float32)
    orc.orc_rope_img(tl.fptr(ic), tl.fptr(is_), c["ih"], c["iw"], 32, F(2000.0), 0)
    tc, ts = np.zeros(T * 128, np.float32), np.zeros(T * 128, np.float32)
    orc.orc_rope_txt(tl.fptr(tc), tl.fptr(ts), T, 32, F(2000.0))
    img, txt = tl.synth_f32((I, h), 1), tl.synth_f32((T, h), 2)
    mi, mt = tl.synth_f32((6 * h,), 3, 0, 0.1), tl.synth_f32((6 * h,), 4, 0, 0.1)
    t0 = time.perf_counter()
    orc.orc_flux_double_block(m, 0, tl.fptr(img), tl.fptr(txt), tl.fptr(mi), tl.fptr(mt), tl.fptr(ic), tl.fptr(is_),
                              tl.fptr(tc), tl.fptr(ts), I, T)
    t_d = time.perf_counter() - t0
    x, temb = tl.synth_f32((T + I, h), 5), tl.synth_f32((h,), 6)
    t0 = time.perf_counter()
    orc.orc_flux_single_block(m, 0, tl.fptr(x), tl.fptr(temb), tl.fptr(ic), tl.fptr(is_), tl.fptr(tc), tl.fptr(ts),
                              T + I, T)
    t_s = time.perf_counter() - t0
    orc.orc_flux_free(m)
    ms_step = (c["nd"] * t_d + c["ns"] * t_s) * 1000 * c["B"]
    return {"value": round(1000.0 / (ms_step * c["steps"]), 6), "unit": "images/s", "cores": threads,
            "kind": "port", "ms_per_step": round(ms_step, 1),
            "sample": f"oracle (C restatement of the reference make-blas path, "
                      f"{orc.orc_blas_info().decode()}) on {host}: 1 double block {t_d:.2f} s + 1 single block {t_s:.2f} s "
                      f"at S={T + I}, h={h}, extrapolated x{c['nd']} + x{c['ns']} per step"}


def cpu_baseline_zimage(orc, c, threads, host):
    d, T = c["d"], c["cap"]
    I = (c["lh"] // 2) * (c["lw"] // 2)
    S = I + T
    orc.orc_zi_create_synth.restype = ctypes.c_void_p
    orc.orc_zi_create_synth.argtypes = [ctypes.c_int] * 7 + [F, ctypes.c_void_p, ctypes.c_int, ctypes.c_int,
                                                             ctypes.c_uint64]
    axes = (ctypes.c_int * 3)(32, 48, 48)
    m = ctypes.c_void_p(orc.orc_zi_create_synth(d, c["H"], 1, 1, c["cap_dim"], 16, 2, F(256.0), axes, c["ffn"],
                                                c["t_mid"], 20250101))
    Wt = c["lw"] // 2
    pos = np.zeros((S, 3), np.int32)
    pos[:I, 0], pos[:I, 1], pos[:I, 2] = T + 1, np.arange(I) // Wt, np.arange(I) % Wt
    pos[I:, 0] = 1 + np.arange(T)
    mask = np.ones(S, np.int32)
    x, temb = tl.synth_f32((S, d), 5), tl.synth_f32((256,), 6)
    t0 = time.perf_counter()
    orc.orc_zi_block(m, 2, 0, tl.fptr(x), pos.ctypes.data_as(tl.IP), mask.ctypes.data_as(tl.IP), tl.fptr(temb), S)
    t_main = time.perf_counter() - t0
    orc.orc_zi_free(m)
    # refiners at their own lengths scale with their share of the block work
    blk = lambda s: 8 * s * d * d + 6 * s * d * c["ffn"] + 4 * s * s * d  # noqa: E731
    n_eq = c["layers"] + c["refiners"] * (blk(I) + blk(T)) / blk(S)
    ms_step = t_main * n_eq * 1000
    return {"value": round(1000.0 / (ms_step * c["steps"]), 6), "unit": "images/s", "cores": threads,
            "kind": "port", "ms_per_step": round(ms_step, 1),
            "sample": f"oracle (C restatement of the reference f32 path with sgemm attention, "
                      f"{orc.orc_blas_info().decode()}) on {host}: 1 main block {t_main:.2f} s at S={S}, d={d}, "
                      f"extrapolated to {n_eq:.2f} block-equivalents per step"}


if __name__ == "__main__":
    main()
