"""The workloads whose speed is measured: what a program that makes images
with this library has it compute, through the C entry points of
iris.c_amd/libiris_hip.so.

listed() names them, draw() draws more from the same ranges, prepare() makes
the inputs and the loaded model, run() is one pass, exact() the same outputs
in 64 bits from plain torch.

The denoisers run at their real widths and a fraction of their depth (Flux: 1
double-stream to 4 single-stream blocks, the 4B and 9B models' ratio; Z-Image:
3 of 30 layers with one refiner of each kind), so a pass holds every kernel of
a step in the step's proportions and the outputs stay close enough to the
64-bit ones to be compared. The text encoder runs all the layers its
extraction mode needs, the VAE is whole. Weights are the library's seeded
random-init ones, made once per process for each architecture as a program
loads its model once; inputs are made from the seed.
"""
import ctypes
import functools
import math
import os
import random
import weakref

import numpy as np
import torch

HERE = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
WEIGHTS_SEED = 20250101
VP, FP, I, F = ctypes.c_void_p, ctypes.POINTER(ctypes.c_float), ctypes.c_int, ctypes.c_float

FLUX = {"4b": dict(h=3072, heads=24, td=7680), "9b": dict(h=4096, heads=32, td=12288)}
FLUX_ND, FLUX_NS, FLUX_T, FLUX_THETA, LATENT_CH = 1, 4, 512, 2000.0, 128
ZI = dict(d=3840, heads=30, ffn=10240, cap_dim=2560, t_mid=1024, ch=16, theta=256.0, axes=(32, 48, 48))
ZI_LAYERS, ZI_REFINERS, ZI_EPS = 3, 1, 1e-5
QW = dict(h=2560, inter=9728, heads=32, kv=8, vocab=151936, layers=28, theta=1e6)
# the VAE scaling of the two model families: batch-norm statistics (Flux, 32
# channels), scale and shift (Z-Image, 16 channels)
VAE = {32: (0.0, 0.0), 16: (0.3611, 0.1159)}


# ------------------------------------------------------------------ the cases

def _flux(model, ih, iw, refs=0, rh=0, rw=0, batch=1):
    return {"kind": "flux", "model": model, "ih": ih, "iw": iw, "refs": refs, "rh": rh, "rw": rw, "batch": batch}


def _zimage(lh, lw, cap):
    return {"kind": "zimage", "lh": lh, "lw": lw, "cap": cap}


def _qwen3(mode, seq, real):
    return {"kind": "qwen3", "mode": mode, "seq": seq, "real": real}


def _vae(kind, z, lh, lw):
    return {"kind": kind, "z": z, "lh": lh, "lw": lw}


def listed():
    return [
        # the smallest image in common use, 256x256: previews, thumbnails
        dict(_flux("4b", 16, 16), name="flux4b_256"),
        # 512x512
        dict(_flux("4b", 32, 32), name="flux4b_512"),
        # 1024x1024, the size the models are made for
        dict(_flux("4b", 64, 64), name="flux4b_1024"),
        # an image of odd sides (720x1328) edited after one reference of another size
        dict(_flux("4b", 45, 83, refs=1, rh=33, rw=47), name="flux4b_wide_ref"),
        # 1024x1024 after two references of 1024x1024: 12800 tokens
        dict(_flux("4b", 64, 64, refs=2, rh=64, rw=64), name="flux4b_1024_refs2"),
        # the 9B base model at 512x512, both branches of classifier-free guidance in one batch
        dict(_flux("9b", 32, 32, batch=2), name="flux9b_512_cfg"),
        # Z-Image at 512x512 with a sentence as its caption
        dict(_zimage(64, 64, 77), name="zimage_512"),
        # Z-Image at 1024x1024 with a paragraph as its caption
        dict(_zimage(128, 128, 203), name="zimage_1024"),
        # Flux's text encoder: always 512 tokens, of which the prompt fills some
        dict(_qwen3(0, 512, 90), name="qwen3_flux_512"),
        # Z-Image's text encoder on a short prompt: no padding
        dict(_qwen3(1, 37, 37), name="qwen3_zimage_37"),
        # latent to picture at 1024x1024
        dict(_vae("vae_decode", 32, 64, 64), name="vae_decode_1024"),
        # picture to latent at 512x512: a reference image
        dict(_vae("vae_encode", 32, 32, 32), name="vae_encode_512"),
    ]


def _between(rng, lo, hi):
    """A whole number of [lo, hi], spread evenly over the logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["flux", "flux", "flux", "zimage", "zimage", "qwen3", "qwen3", "vae_decode", "vae_encode"])
    if kind == "flux":
        # image sides of 192 to 1424 pixels; sometimes references, or guidance as a batch of two
        model, ih, iw = rng.choice(["4b", "4b", "9b"]), _between(rng, 12, 89), _between(rng, 12, 89)
        refs, batch = (0, 2) if rng.random() < 0.25 else (rng.choice([0, 0, 1, 2]), 1)
        rh, rw = (_between(rng, 12, 64), _between(rng, 12, 64)) if refs else (0, 0)
        c = _flux(model, ih, iw, refs, rh, rw, batch)
        most = work(listed()[4])["flops"]
        return c if work(c)["flops"] <= most else _flux(model, ih // 2, iw // 2, min(refs, 1), rh, rw, batch)
    if kind == "zimage":
        return _zimage(2 * _between(rng, 12, 80), 2 * _between(rng, 12, 80), _between(rng, 8, 512))
    if kind == "qwen3":
        if rng.random() < 0.5:
            return _qwen3(0, 512, _between(rng, 6, 512))
        n = _between(rng, 6, 512)
        return _qwen3(1, n, n)
    return _vae(kind, rng.choice([16, 32]), _between(rng, 12, 72), _between(rng, 12, 72))


def _flux_tokens(c):
    i0 = c["ih"] * c["iw"]
    return i0, i0 + c["refs"] * c["rh"] * c["rw"]


def _vae_blocks(c):
    """(cin, cout, pixels, 3x3) of each convolution of the decoder or encoder, and the bottleneck's pixels."""
    p = 4 * c["lh"] * c["lw"]
    mult, z, out = (1, 2, 4, 4), c["z"], []
    if c["kind"] == "vae_decode":
        out += [(z, z, p, 1), (z, 512, p, 9)] + [(512, 512, p, 9)] * 4
        q, prev = p, 512
        for level in (3, 2, 1, 0):
            ch = 128 * mult[level]
            for r in range(3):
                out += [(prev, ch, q, 9), (ch, ch, q, 9)] + ([(prev, ch, q, 1)] if prev != ch else [])
                prev = ch
            if level:
                q *= 4
                out.append((ch, ch, q, 9))
        out.append((128, 3, q, 9))
    else:
        q, prev = 64 * p, 128
        out.append((3, 128, q, 9))
        for level in range(4):
            ch = 128 * mult[level]
            for r in range(2):
                out += [(prev, ch, q, 9), (ch, ch, q, 9)] + ([(prev, ch, q, 1)] if prev != ch else [])
                prev = ch
            if level < 3:
                q //= 4
                out.append((ch, ch, q, 9))
        out += [(512, 512, p, 9)] * 4 + [(512, 2 * z, p, 9), (2 * z, z, p, 1)]
    return out, p


def work(c):
    """What a pass cannot do without: each product once (2 M N K), attention
    4 Sq Sk d (causal: half); each weight, input and output once."""
    if c["kind"] == "flux":
        m = FLUX[c["model"]]
        h, td, b = m["h"], m["td"], c["batch"]
        i0, i = _flux_tokens(c)
        s = i + FLUX_T
        n = FLUX_ND + FLUX_NS
        flops = n * (26 * s * h * h + 4 * s * s * h) + 2 * FLUX_T * td * h + 2 * i * LATENT_CH * h
        flops = (flops + 2 * i0 * LATENT_CH * h) * b + 2 * (256 * h + 18 * h * h)
        weights = (26 * FLUX_ND + 13 * FLUX_NS + 18) * h * h + (td + 2 * LATENT_CH + 256) * h
        return {"bytes": 2 * weights + 4 * (i * LATENT_CH + b * (FLUX_T * td + i0 * LATENT_CH)), "flops": flops}
    if c["kind"] == "zimage":
        d, f = ZI["d"], ZI["ffn"]
        n, t, pix = c["lh"] * c["lw"] // 4, c["cap"], c["lh"] * c["lw"]

        def blk(s):
            return 8 * s * d * d + 6 * s * d * f + 4 * s * s * d
        blocks = ZI_LAYERS + 2 * ZI_REFINERS
        flops = ZI_LAYERS * blk(n + t) + ZI_REFINERS * (blk(n) + blk(t)) + 4 * n * 64 * d + 2 * t * ZI["cap_dim"] * d
        weights = blocks * (4 * d * d + 3 * d * f) + (ZI_LAYERS + ZI_REFINERS) * 4 * d * 256 + d * (ZI["cap_dim"] + 128)
        return {"bytes": 2 * weights + 4 * (2 * ZI["ch"] * pix + t * ZI["cap_dim"]), "flops": flops}
    if c["kind"] == "qwen3":
        h, inter, qd, kd, s = QW["h"], QW["inter"], QW["heads"] * 128, QW["kv"] * 128, c["seq"]
        layers = 27 if c["mode"] == 0 else QW["layers"] - 1
        per = h * (qd + 2 * kd) + qd * h + 3 * h * inter
        out = s * h * (3 if c["mode"] == 0 else 1)
        return {"bytes": 2 * layers * per + 2 * s * h + 4 * (s + out), "flops": layers * (2 * s * per + 2 * s * s * qd)}
    convs, p = _vae_blocks(c)
    flops = sum(2 * a * b * q * k for a, b, q, k in convs) + 8 * p * 512 * 512 + 4 * p * p * 512
    weights = sum(a * b * k for a, b, q, k in convs) + 4 * 512 * 512
    return {"bytes": 2 * weights + 4 * (4 * c["z"] * c["lh"] * c["lw"] + 3 * 64 * p), "flops": flops}


def tolerance(c):
    # bf16 operands into every product, f32 sums. Measured against exact():
    # flux 3.8e-3 (9B 5.7e-3), zimage 2.7e-3, qwen3 1.6e-2 to 1.9e-2 after its
    # 27 layers, decode 6.0e-3, encode 1.2e-2; another order of the sums moves
    # a result by up to about the same amount. About four times that, or what
    # the rounding of 27 layers makes of it
    rel = {"flux": 1.6e-2, "zimage": 1.1e-2, "qwen3": 3e-2, "vae_decode": 2.4e-2, "vae_encode": 3e-2}[c["kind"]]
    return {"rel": rel, "max": 0.2 if c["kind"] in ("flux", "zimage") else 0.8}


# ------------------------------------------------------------ library, models

class _Ref(ctypes.Structure):     # iris_ref_t
    _fields_ = [("latent", FP), ("h", I), ("w", I), ("t_offset", I)]


@functools.lru_cache(maxsize=1)
def _lib():
    torch.cuda.init()             # one HIP runtime in the process: torch's
    lib = ctypes.CDLL(os.path.join(HERE, "iris.c_amd", "libiris_hip.so"))
    for name, res, args in (
            ("iris_hip_memcpy_d2d", I, [VP, VP, ctypes.c_size_t]), ("iris_hip_sync", I, []),
            ("iris_hip_last_error", ctypes.c_char_p, []),
            ("iris_transformer_create_synthetic", VP, [I, I, I, I, I, I, F, F, ctypes.c_uint64]),
            ("iris_transformer_free", None, [VP]), ("iris_flux_prepare", I, [VP, I, I, VP, I, I, I]),
            ("iris_flux_velocity", I, [VP, F]), ("iris_flux_device_buffer", VP, [VP, ctypes.c_char_p]),
            ("zi_transformer_create_synthetic", VP, [I] * 7 + [F, ctypes.POINTER(I), I, I, ctypes.c_uint64]),
            ("zi_transformer_free", None, [VP]), ("zi_prepare", I, [VP, I, I, I]), ("zi_velocity", I, [VP, F]),
            ("zi_upload", I, [VP, VP, VP]), ("zi_device_buffer", VP, [VP, ctypes.c_char_p]),
            ("qwen3_model_create_synthetic", VP, [I] * 6 + [ctypes.c_uint64]), ("qwen3_model_free", None, [VP]),
            ("qwen3_model_set_extraction_mode", None, [VP, I]), ("qwen3_forward", VP, [VP, VP, VP, I]),
            ("iris_vae_gpu_create_synthetic", VP, [I, F, F, ctypes.c_uint64]), ("iris_vae_gpu_free", None, [VP]),
            ("iris_vae_gpu_decode_device", I, [VP, VP, I, I, VP, VP]),
            ("iris_vae_gpu_encode_device", I, [VP, VP, I, I, VP])):
        f = getattr(lib, name)
        f.restype, f.argtypes = res, args
    return lib


def _ok(rc):
    if rc:
        raise RuntimeError("iris: %s" % _lib().iris_hip_last_error().decode())


class Handle:
    """A model of the library, freed with its last holder."""

    def __init__(self, ptr, free):
        if not ptr:
            raise RuntimeError("iris: %s" % _lib().iris_hip_last_error().decode())
        self.ptr, self.bufs = ptr, {}
        weakref.finalize(self, free, ptr)


@functools.lru_cache(maxsize=1)
def _flux_model(model, ih, iw, refs, rh, rw, batch):
    m, lib = FLUX[model], _lib()
    tf = Handle(lib.iris_transformer_create_synthetic(m["h"], m["heads"], FLUX_ND, FLUX_NS, m["td"], LATENT_CH, 3.0,
                                                      FLUX_THETA, WEIGHTS_SEED), lib.iris_transformer_free)
    r = (_Ref * max(1, refs))(*[_Ref(None, rh, rw, k + 1) for k in range(refs)])
    _ok(lib.iris_flux_prepare(tf.ptr, ih, iw, r if refs else None, refs, FLUX_T, batch))
    tf.bufs = {n: lib.iris_flux_device_buffer(tf.ptr, n.encode()) for n in ("latent", "txt", "velocity")}
    return tf


@functools.lru_cache(maxsize=1)
def _zi_model(lh, lw, cap):
    lib, z = _lib(), ZI
    tf = Handle(lib.zi_transformer_create_synthetic(z["d"], z["heads"], ZI_LAYERS, ZI_REFINERS, z["cap_dim"], z["ch"],
                                                    2, z["theta"], (I * 3)(*z["axes"]), z["ffn"], z["t_mid"],
                                                    WEIGHTS_SEED), lib.zi_transformer_free)
    _ok(lib.zi_prepare(tf.ptr, lh, lw, cap))
    return tf


@functools.lru_cache(maxsize=1)
def _qwen3_model():
    lib, q = _lib(), QW
    return Handle(lib.qwen3_model_create_synthetic(q["h"], q["inter"], q["heads"], q["kv"], q["layers"], q["vocab"],
                                                   WEIGHTS_SEED), lib.qwen3_model_free)


@functools.lru_cache(maxsize=1)
def _vae_model(z):
    lib = _lib()
    return Handle(lib.iris_vae_gpu_create_synthetic(z, *VAE[z], WEIGHTS_SEED), lib.iris_vae_gpu_free)


_KINDS = {"flux": _flux_model, "zimage": _zi_model, "qwen3": _qwen3_model, "vae": _vae_model}


def _only(kind):
    """The models of the other kinds are let go."""
    for k, f in _KINDS.items():
        if k != kind:
            f.cache_clear()


# --------------------------------------------------------------------- inputs

def _inputs(c, seed):
    """The inputs of a pass, the same for run() and exact()."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)

    def normal(*shape):
        return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)
    # a step's time: anywhere in the schedule
    t = float(np.float32(random.Random(seed).uniform(0.02, 1.0)))
    if c["kind"] == "flux":
        _, i = _flux_tokens(c)
        return {"t": t, "lat": normal(LATENT_CH * i), "txt": normal(c["batch"], FLUX_T, FLUX[c["model"]]["td"])}
    if c["kind"] == "zimage":
        return {"t": t, "lat": normal(ZI["ch"], c["lh"], c["lw"]), "cap": normal(c["cap"], ZI["cap_dim"])}
    if c["kind"] == "qwen3":
        ids = torch.randint(0, QW["vocab"], (c["seq"],), generator=g, device="cuda").cpu().numpy().astype(np.int32)
        return {"ids": ids, "mask": (np.arange(c["seq"]) < c["real"]).astype(np.int32)}
    if c["kind"] == "vae_decode":
        return {"lat": normal(4 * c["z"], c["lh"], c["lw"])}
    # a picture: smooth shapes and some grain, in [-1, 1]
    h, w = 16 * c["lh"], 16 * c["lw"]
    low = torch.nn.functional.interpolate(normal(1, 3, 9, 9), size=(h, w), mode="bicubic")[0]
    return {"img": (0.5 * low + 0.05 * normal(3, h, w)).clamp(-1, 1).contiguous()}


def prepare(c, seed):
    lib = _lib()
    s = dict(_inputs(c, seed), kind=c["kind"], case=c, lib=lib)
    if c["kind"] == "flux":
        _only("flux")
        s["model"] = _flux_model(c["model"], c["ih"], c["iw"], c["refs"], c["rh"], c["rw"], c["batch"])
        s["out"] = torch.empty(c["batch"], LATENT_CH, c["ih"], c["iw"], device="cuda")
    elif c["kind"] == "zimage":
        _only("zimage")
        s["model"] = _zi_model(c["lh"], c["lw"], c["cap"])
        s["lat_buf"] = lib.zi_device_buffer(s["model"].ptr, b"latent")
        s["vel_buf"] = lib.zi_device_buffer(s["model"].ptr, b"velocity")
        s["cap_host"] = s["cap"].cpu().numpy()
        s["out"] = torch.empty(ZI["ch"], c["lh"], c["lw"], device="cuda")
    elif c["kind"] == "qwen3":
        _only("qwen3")
        s["model"] = _qwen3_model()
    else:
        _only("vae")
        s["model"] = _vae_model(c["z"])
        if c["kind"] == "vae_decode":
            s["rgb"] = torch.empty(16 * c["lh"], 16 * c["lw"], 3, device="cuda", dtype=torch.uint8)
            s["out"] = torch.empty(3, 16 * c["lh"], 16 * c["lw"], device="cuda")
        else:
            s["out"] = torch.empty(4 * c["z"], c["lh"], c["lw"], device="cuda")
    torch.cuda.synchronize()      # the library works on streams of its own
    return s


def run(s):
    lib, tf, kind = s["lib"], s["model"], s["kind"]
    if kind == "flux":
        # a program's own sampler: its latent and text into the resident
        # buffers, one evaluation, the velocity out of them
        lat, txt, out = s["lat"], s["txt"], s["out"]
        _ok(lib.iris_hip_memcpy_d2d(tf.bufs["latent"], lat.data_ptr(), lat.numel() * 4) or
            lib.iris_hip_memcpy_d2d(tf.bufs["txt"], txt.data_ptr(), txt.numel() * 4) or
            lib.iris_flux_velocity(tf.ptr, s["t"]) or
            lib.iris_hip_memcpy_d2d(out.data_ptr(), tf.bufs["velocity"], out.numel() * 4))
        return out
    if kind == "zimage":
        # the caption comes from host memory, as the library's samplers pass it
        lat, out = s["lat"], s["out"]
        _ok(lib.iris_hip_memcpy_d2d(s["lat_buf"], lat.data_ptr(), lat.numel() * 4) or
            lib.zi_upload(tf.ptr, None, s["cap_host"].ctypes.data) or lib.zi_velocity(tf.ptr, s["t"]) or
            lib.iris_hip_memcpy_d2d(out.data_ptr(), s["vel_buf"], out.numel() * 4))
        return out
    if kind == "qwen3":
        c = s["case"]
        lib.qwen3_model_set_extraction_mode(tf.ptr, c["mode"])
        p = lib.qwen3_forward(tf.ptr, s["ids"].ctypes.data, s["mask"].ctypes.data, c["seq"])
        if not p:
            raise RuntimeError("iris: %s" % lib.iris_hip_last_error().decode())
        shape = (c["seq"], QW["h"] * (3 if c["mode"] == 0 else 1))
        held = (F * (shape[0] * shape[1])).from_address(p)
        weakref.finalize(held, ctypes.CDLL(None).free, VP(p))
        return np.frombuffer(held, dtype=np.float32).reshape(shape)
    c, out = s["case"], s["out"]
    if kind == "vae_decode":
        # the bytes of the picture are this output rounded, element by element
        _ok(lib.iris_vae_gpu_decode_device(tf.ptr, s["lat"].data_ptr(), c["lh"], c["lw"], s["rgb"].data_ptr(),
                                           out.data_ptr()))
    else:
        _ok(lib.iris_vae_gpu_encode_device(tf.ptr, s["img"].data_ptr(), 16 * c["lh"], 16 * c["lw"], out.data_ptr()))
    return out


# ------------------------------------------------------- the same in 64 bits

_M64 = (1 << 64) - 1


def _splitmix(z):
    z = (z + 0x9E3779B97F4A7C15) & _M64
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & _M64
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & _M64
    return z ^ (z >> 31)


def _tensor_seed(name):
    h = 0xCBF29CE484222325
    for ch in name.encode():
        h = ((h ^ ch) * 0x100000001B3) & _M64
    return _splitmix(h ^ _splitmix(WEIGHTS_SEED))


def _signed(v):
    return v - (1 << 64) if v >= 1 << 63 else v


def _shr(x, n):
    return (x >> n) & ((1 << (64 - n)) - 1)


def _weight(name, *shape, mean=0.0, std=0.02, bf16=True):
    """The seeded tensor of include/iris_synth.h, in 64 bits."""
    n = math.prod(shape)
    out = torch.empty(n, dtype=torch.float64, device="cuda")
    base = _tensor_seed(name) * 0x9E3779B97F4A7C15
    std32, scale = float(np.float32(std)), float(np.float32(1.0) / np.float32(37837.2273))
    for at in range(0, n, 1 << 25):
        m = min(1 << 25, n - at)
        z = torch.arange(m, dtype=torch.int64, device="cuda") + _signed((base + at + 0x9E3779B97F4A7C15) & _M64)
        z = (z ^ _shr(z, 30)) * _signed(0xBF58476D1CE4E5B9)
        z = (z ^ _shr(z, 27)) * _signed(0x94D049BB133111EB)
        z = z ^ _shr(z, 31)
        u = (z & 0xFFFF) + (_shr(z, 16) & 0xFFFF) + (_shr(z, 32) & 0xFFFF) + _shr(z, 48) - 131070
        v = (u.to(torch.float32) * scale).to(torch.float64) * std32 + mean
        v = v.to(torch.float32)
        out[at:at + m] = v.to(torch.bfloat16) if bf16 else v
    return out.view(*shape)


def _norm_w(name, n):
    return _weight(name, n, mean=1.0)


def _silu(x):
    return x * torch.sigmoid(x)


def _rms(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w


def _ln(x, eps=1e-6):
    x = x - x.mean(-1, keepdim=True)
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps)


def _time_sincos(t):
    a = t * 1000.0 * torch.exp(-math.log(10000.0) * torch.arange(128, dtype=torch.float64, device="cuda") / 128)
    return torch.cat([a.cos(), a.sin()])


def _angles(pos, dims, theta):
    """Rotation angles [tokens][sum dims / 2] of positions [tokens][axes]."""
    out = []
    for ax, d in enumerate(dims):
        f = theta ** (-torch.arange(0, d, 2, dtype=torch.float64, device="cuda") / d)
        out.append(pos[:, ax:ax + 1].double() * f)
    return torch.cat(out, 1)


def _rotate(x, ang):
    """Adjacent pairs of x [tokens][heads][128] by ang [tokens][64]."""
    c, s = ang.cos()[:, None], ang.sin()[:, None]
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * c - b * s, b * c + a * s], -1).flatten(-2)


def _attend(q, k, v, keep=None):
    """softmax(q k^T / sqrt(128)) v per head; q, k, v [tokens][heads][128]."""
    out = torch.empty_like(q)
    group = q.shape[1] // k.shape[1]
    for h in range(q.shape[1]):
        kh, vh = k[:, h // group], v[:, h // group]
        for at in range(0, q.shape[0], 4096):
            s = q[at:at + 4096, h] @ kh.T / math.sqrt(128.0)
            if keep is not None:
                s.masked_fill_(~(keep if keep.dim() == 1 else keep[at:at + 4096]), -math.inf)
            out[at:at + 4096, h] = torch.softmax(s, -1) @ vh
    return out


def _flux_exact(c, x):
    m = FLUX[c["model"]]
    h, heads, td = m["h"], m["heads"], m["td"]
    mlp, T = 3 * h, FLUX_T
    i0, i = _flux_tokens(c)
    lat, rp = x["lat"].double(), c["rh"] * c["rw"]
    tokens = [lat[:LATENT_CH * i0].view(LATENT_CH, i0).T]
    for r in range(c["refs"]):
        at = LATENT_CH * (i0 + r * rp)
        tokens.append(lat[at:at + LATENT_CH * rp].view(LATENT_CH, rp).T)
    tokens = torch.cat(tokens)
    pos = torch.zeros(T + i, 4, dtype=torch.int64, device="cuda")
    pos[:T, 3] = torch.arange(T, device="cuda")
    at = T
    for k, (ph, pw) in enumerate([(c["ih"], c["iw"])] + [(c["rh"], c["rw"])] * c["refs"]):
        n = torch.arange(ph * pw, device="cuda")
        pos[at:at + ph * pw] = torch.stack([torch.full_like(n, k), n // pw, n % pw, torch.zeros_like(n)], 1)
        at += ph * pw
    ang = _angles(pos, (32, 32, 32, 32), FLUX_THETA)
    tn = "time_guidance_embed.timestep_embedder.linear_%d.weight"
    temb = _weight(tn % 2, h, h) @ _silu(_weight(tn % 1, h, 256) @ _time_sincos(x["t"]))
    st = _silu(temb)
    mi = (_weight("double_stream_modulation_img.linear.weight", 6 * h, h) @ st).view(6, h)
    mt = (_weight("double_stream_modulation_txt.linear.weight", 6 * h, h) @ st).view(6, h)
    ms = (_weight("single_stream_modulation.linear.weight", 3 * h, h) @ st).view(3, h)
    fm = (_weight("norm_out.linear.weight", 2 * h, h) @ st).view(2, h)
    img0 = tokens @ _weight("x_embedder.weight", h, LATENT_CH).T
    ctx = _weight("context_embedder.weight", h, td)
    xs = [torch.cat([x["txt"][b].double() @ ctx.T, img0]) for b in range(c["batch"])]
    del ctx

    def heads_of(y):
        return y.view(y.shape[0], heads, 128)

    def swiglu(y):
        return _silu(y[:, :mlp]) * y[:, mlp:]
    for n in range(FLUX_ND):
        p = "transformer_blocks.%d." % n
        side = []
        for a, o, ff, nq, nk in ((("to_q", "to_k", "to_v"), "to_out.0", "ff", "norm_q", "norm_k"),
                                 (("add_q_proj", "add_k_proj", "add_v_proj"), "to_add_out", "ff_context",
                                  "norm_added_q", "norm_added_k")):
            side.append(([_weight(p + "attn.%s.weight" % q, h, h) for q in a], _weight(p + "attn.%s.weight" % o, h, h),
                         _weight(p + ff + ".linear_in.weight", 2 * mlp, h),
                         _weight(p + ff + ".linear_out.weight", h, mlp), _norm_w(p + "attn.%s.weight" % nq, 128),
                         _norm_w(p + "attn.%s.weight" % nk, 128)))
        for b in range(c["batch"]):
            parts, qkv = (xs[b][T:], xs[b][:T]), []
            for y, mod, w in zip(parts, (mi, mt), side):
                a = (1 + mod[1]) * _ln(y) + mod[0]
                q, k, v = (heads_of(a @ u.T) for u in w[0])
                qkv.append((_rms(q, w[4], 1e-6), _rms(k, w[5], 1e-6), v))
            q, k, v = (torch.cat([qkv[1][j], qkv[0][j]]) for j in range(3))
            o = _attend(_rotate(q, ang), _rotate(k, ang), v).flatten(1)
            new = []
            for y, att, mod, w in zip(parts, (o[T:], o[:T]), (mi, mt), side):
                y = y + mod[2] * (att @ w[1].T)
                a = (1 + mod[4]) * _ln(y) + mod[3]
                new.append(y + mod[5] * (swiglu(a @ w[2].T) @ w[3].T))
            xs[b] = torch.cat([new[1], new[0]])
        del side
    for n in range(FLUX_NS):
        p = "single_transformer_blocks.%d.attn." % n
        win, wout = _weight(p + "to_qkv_mlp_proj.weight", 3 * h + 2 * mlp, h), _weight(p + "to_out.weight", h, h + mlp)
        nq, nk = _norm_w(p + "norm_q.weight", 128), _norm_w(p + "norm_k.weight", 128)
        for b in range(c["batch"]):
            y = ((1 + ms[1]) * _ln(xs[b]) + ms[0]) @ win.T
            q, k, v = (heads_of(y[:, j * h:(j + 1) * h]) for j in range(3))
            o = _attend(_rotate(_rms(q, nq, 1e-6), ang), _rotate(_rms(k, nk, 1e-6), ang), v).flatten(1)
            xs[b] = xs[b] + ms[2] * (torch.cat([o, swiglu(y[:, 3 * h:])], 1) @ wout.T)
    pw = _weight("proj_out.weight", LATENT_CH, h)
    out = [(((1 + fm[0]) * _ln(y[T:T + i0]) + fm[1]) @ pw.T).T.reshape(LATENT_CH, c["ih"], c["iw"]) for y in xs]
    return torch.stack(out)


def _zimage_exact(c, x):
    d, heads, f, cd = ZI["d"], ZI["heads"], ZI["ffn"], ZI["cap_dim"]
    ht, wt, cap, ch = c["lh"] // 2, c["lw"] // 2, c["cap"], ZI["ch"]
    n = ht * wt
    ip, cp = (n + 31) // 32 * 32, (cap + 31) // 32 * 32
    u = ip + cp
    temb = _weight("t_embedder.mlp.0.weight", 1024, 256) @ _time_sincos(x["t"]) + _weight("t_embedder.mlp.0.bias", 1024)
    temb = _weight("t_embedder.mlp.2.weight", 256, 1024) @ _silu(temb) + _weight("t_embedder.mlp.2.bias", 256)
    patches = x["lat"].double().view(ch, ht, 2, wt, 2).permute(1, 3, 2, 4, 0).reshape(n, 4 * ch)
    img = patches @ _weight("all_x_embedder.2-1.weight", d, 4 * ch).T + _weight("all_x_embedder.2-1.bias", d)
    y = _rms(x["cap"].double(), _norm_w("cap_embedder.0.weight", cd), ZI_EPS)
    y = y @ _weight("cap_embedder.1.weight", d, cd).T + _weight("cap_embedder.1.bias", d)
    xs = torch.cat([img, _weight("x_pad_token", d, std=1.0).expand(ip - n, d), y,
                    _weight("cap_pad_token", d, std=1.0).expand(cp - cap, d)])
    pos = torch.zeros(u, 3, dtype=torch.int64, device="cuda")
    at = torch.arange(n, device="cuda")
    pos[:n] = torch.stack([torch.full_like(at, cp + 1), at // wt, at % wt], 1)
    pos[ip:, 0] = 1 + torch.arange(cp, device="cuda")
    ang = _angles(pos, ZI["axes"], ZI["theta"])
    keep = torch.zeros(u, dtype=torch.bool, device="cuda")
    keep[:n] = True
    keep[ip:ip + cap] = True

    def block(pre, y, ang, keep, modulated):
        one = torch.ones(d, dtype=torch.float64, device="cuda")
        s1, g1, s2, g2 = one, one, one, one
        if modulated:
            mod = _weight(pre + ".adaLN_modulation.0.weight", 4 * d, 256) @ temb
            mod = (mod + _weight(pre + ".adaLN_modulation.0.bias", 4 * d)).view(4, d)
            s1, g1, s2, g2 = 1 + mod[0], mod[1].tanh(), 1 + mod[2], mod[3].tanh()
        a = _rms(y, _norm_w(pre + ".attention_norm1.weight", d), ZI_EPS) * s1
        q, k, v = ((a @ _weight(pre + ".attention.%s.weight" % p, d, d).T).view(-1, heads, 128)
                   for p in ("to_q", "to_k", "to_v"))
        q = _rotate(_rms(q, _norm_w(pre + ".attention.norm_q.weight", 128), ZI_EPS), ang)
        k = _rotate(_rms(k, _norm_w(pre + ".attention.norm_k.weight", 128), ZI_EPS), ang)
        o = _attend(q, k, v, keep).flatten(1) @ _weight(pre + ".attention.to_out.0.weight", d, d).T
        y = y + g1 * _rms(o, _norm_w(pre + ".attention_norm2.weight", d), ZI_EPS)
        a = _rms(y, _norm_w(pre + ".ffn_norm1.weight", d), ZI_EPS) * s2
        o = _silu(a @ _weight(pre + ".feed_forward.w1.weight", f, d).T)
        o = (o * (a @ _weight(pre + ".feed_forward.w3.weight", f, d).T)) @ _weight(pre + ".feed_forward.w2.weight", d, f).T
        return y + g2 * _rms(o, _norm_w(pre + ".ffn_norm2.weight", d), ZI_EPS)
    for k in range(ZI_REFINERS):
        xs = torch.cat([block("noise_refiner.%d" % k, xs[:ip], ang[:ip], keep[:ip], True),
                        block("context_refiner.%d" % k, xs[ip:], ang[ip:], keep[ip:], False)])
    for k in range(ZI_LAYERS):
        xs = block("layers.%d" % k, xs, ang, keep, True)
    p = "all_final_layer.2-1."
    scale = 1 + _weight(p + "adaLN_modulation.1.weight", d, 256) @ _silu(temb) + _weight(p + "adaLN_modulation.1.bias", d)
    y = (_ln(xs[:n]) * scale) @ _weight(p + "linear.weight", 4 * ch, d).T + _weight(p + "linear.bias", 4 * ch)
    return y.view(ht, wt, 2, 2, ch).permute(4, 0, 2, 1, 3).reshape(ch, c["lh"], c["lw"])


def _qwen3_exact(c, x):
    h, inter, heads, kv, s = QW["h"], QW["inter"], QW["heads"], QW["kv"], c["seq"]
    ids = torch.from_numpy(x["ids"].astype(np.int64)).cuda()
    y = _weight("model.embed_tokens.weight", QW["vocab"], h)[ids]
    at = torch.arange(s, device="cuda")
    keep = (at[None] <= at[:, None]) & (at[None] < c["real"])
    ang = _angles(at[:, None], (128,), QW["theta"])
    cs, sn = ang.cos()[:, None], ang.sin()[:, None]

    def rotate(q):                # the two halves of a head rotate against each other
        a, b = q[..., :64], q[..., 64:]
        return torch.cat([a * cs - b * sn, b * cs + a * sn], -1)
    outs, last = [], 26 if c["mode"] == 0 else QW["layers"] - 2
    for k in range(last + 1):
        p = "model.layers.%d." % k
        a = _rms(y, _norm_w(p + "input_layernorm.weight", h), 1e-6)
        q = (a @ _weight(p + "self_attn.q_proj.weight", heads * 128, h).T).view(s, heads, 128)
        kk = (a @ _weight(p + "self_attn.k_proj.weight", kv * 128, h).T).view(s, kv, 128)
        v = (a @ _weight(p + "self_attn.v_proj.weight", kv * 128, h).T).view(s, kv, 128)
        q = rotate(_rms(q, _norm_w(p + "self_attn.q_norm.weight", 128), 1e-6))
        kk = rotate(_rms(kk, _norm_w(p + "self_attn.k_norm.weight", 128), 1e-6))
        y = y + _attend(q, kk, v, keep).flatten(1) @ _weight(p + "self_attn.o_proj.weight", h, heads * 128).T
        a = _rms(y, _norm_w(p + "post_attention_layernorm.weight", h), 1e-6)
        a = _silu(a @ _weight(p + "mlp.gate_proj.weight", inter, h).T) * (a @ _weight(p + "mlp.up_proj.weight", inter, h).T)
        y = y + a @ _weight(p + "mlp.down_proj.weight", h, inter).T
        if c["mode"] == 1 and k == last or c["mode"] == 0 and k in (8, 17, 26):
            outs.append(y)
    return torch.cat(outs, 1)


def _vae_w(name, *shape, fan_in=0):
    if name.endswith("running_var"):
        mean, std = 1.0, 0.1
    elif name.endswith("running_mean"):
        mean, std = 0.0, 0.1
    elif name.endswith(".bias"):
        mean, std = 0.0, 0.05
    elif "norm" in name and name.endswith(".weight"):
        mean, std = 1.0, 0.1
    else:
        mean = 0.0
        std = float(np.float32(0.5 if name == "decoder.conv_out.weight" else 1.0) / np.sqrt(np.float32(max(fan_in, 1))))
    return _weight(name, *shape, mean=mean, std=std, bf16=False)


class _VaeExact:
    def __init__(self, c):
        self.z, self.eps = c["z"], 1e-6 if VAE[c["z"]][0] else 1e-4

    def conv(self, name, y, cin, cout, stride=1):
        """3x3 on [H][W][cin]: zero padding all round, or right and below for stride 2."""
        w = _vae_w(name + ".weight", cout, cin, 3, 3, fan_in=9 * cin)
        out = _vae_w(name + ".bias", cout).expand((y.shape[0] // stride) * (y.shape[1] // stride), cout).clone()
        p = torch.nn.functional.pad(y, (0, 0, 1, 1, 1, 1) if stride == 1 else (0, 0, 0, 1, 0, 1))
        H, W = y.shape[:2]
        for dy in range(3):
            for dx in range(3):
                v = p[dy:dy + H, dx:dx + W] if stride == 1 else p[dy:dy + H:2, dx:dx + W:2]
                out.addmm_(v.reshape(-1, cin), w[:, :, dy, dx].T)
        return out.view(H // stride, W // stride, cout)

    def gn(self, name, y):
        C = y.shape[-1]
        v = y.reshape(-1, 32, C // 32)
        mean, var = v.mean((0, 2), keepdim=True), v.var((0, 2), unbiased=False, keepdim=True)
        v = ((v - mean) * torch.rsqrt(var + self.eps)).view(y.shape)
        return v * _vae_w(name + ".weight", C) + _vae_w(name + ".bias", C)

    def res(self, p, y, cout):
        cin = y.shape[-1]
        a = self.conv(p + ".conv1", _silu(self.gn(p + ".norm1", y)), cin, cout)
        a = self.conv(p + ".conv2", _silu(self.gn(p + ".norm2", a)), cout, cout)
        if cin != cout:
            y = y @ _vae_w(p + ".conv_shortcut.weight", cout, cin, fan_in=cin).T + _vae_w(p + ".conv_shortcut.bias", cout)
        return y + a

    def attn(self, p, y):
        a = self.gn(p + ".group_norm", y).view(-1, 512)
        q, k, v = (a @ _vae_w("%s.%s.weight" % (p, n), 512, 512, fan_in=512).T + _vae_w("%s.%s.bias" % (p, n), 512)
                   for n in ("to_q", "to_k", "to_v"))
        o = torch.empty_like(q)
        for at in range(0, q.shape[0], 4096):
            o[at:at + 4096] = torch.softmax(q[at:at + 4096] @ k.T / math.sqrt(512.0), -1) @ v
        o = o @ _vae_w(p + ".to_out.0.weight", 512, 512, fan_in=512).T + _vae_w(p + ".to_out.0.bias", 512)
        return y + o.view(y.shape)

    def mid(self, p, y):
        return self.res(p + ".resnets.1", self.attn(p + ".attentions.0", self.res(p + ".resnets.0", y, 512)), 512)

    def stats(self):
        """(scale, shift) of the latent channels: x scale + shift is what the decoder reads."""
        scaling, shift = VAE[self.z]
        if scaling:
            return 1.0 / scaling, shift
        n = 4 * self.z
        return (_vae_w("bn.running_var", n) + self.eps).sqrt()[:, None, None], _vae_w("bn.running_mean", n)[:, None, None]

    def decode(self, lat):
        z = self.z
        sc, sh = self.stats()
        y = lat.double() * sc + sh
        h, w = y.shape[1:]
        y = y.view(z, 2, 2, h, w).permute(3, 1, 4, 2, 0).reshape(2 * h, 2 * w, z)
        y = y @ _vae_w("post_quant_conv.weight", z, z).T + _vae_w("post_quant_conv.bias", z)
        y = self.mid("decoder.mid_block", self.conv("decoder.conv_in", y, z, 512))
        for k, ch in enumerate((512, 512, 256, 128)):
            for r in range(3):
                y = self.res("decoder.up_blocks.%d.resnets.%d" % (k, r), y, ch)
            if k < 3:
                y = y.repeat_interleave(2, 0).repeat_interleave(2, 1)
                y = self.conv("decoder.up_blocks.%d.upsamplers.0.conv" % k, y, ch, ch)
        return self.conv("decoder.conv_out", _silu(self.gn("decoder.conv_norm_out", y)), 128, 3).permute(2, 0, 1)

    def encode(self, img):
        z = self.z
        y = self.conv("encoder.conv_in", img.double().permute(1, 2, 0), 3, 128)
        for k, ch in enumerate((128, 256, 512, 512)):
            for r in range(2):
                y = self.res("encoder.down_blocks.%d.resnets.%d" % (k, r), y, ch)
            if k < 3:
                y = self.conv("encoder.down_blocks.%d.downsamplers.0.conv" % k, y, ch, ch, 2)
        y = _silu(self.gn("encoder.conv_norm_out", self.mid("encoder.mid_block", y)))
        y = self.conv("encoder.conv_out", y, 512, 2 * z)
        y = (y @ _vae_w("quant_conv.weight", 2 * z, 2 * z).T + _vae_w("quant_conv.bias", 2 * z))[..., :z]
        h, w = y.shape[0] // 2, y.shape[1] // 2
        y = y.view(h, 2, w, 2, z).permute(4, 1, 3, 0, 2).reshape(4 * z, h, w)
        sc, sh = self.stats()
        return (y - sh) / sc


@torch.no_grad()
def exact(c, seed):
    _only(None)
    x = _inputs(c, seed)
    if c["kind"] == "flux":
        return _flux_exact(c, x)
    if c["kind"] == "zimage":
        return _zimage_exact(c, x)
    if c["kind"] == "qwen3":
        return _qwen3_exact(c, x).cpu().numpy()
    return _VaeExact(c).decode(x["lat"]) if c["kind"] == "vae_decode" else _VaeExact(c).encode(x["img"])
