"""Performance cases: the transforms a user of this library runs, through its public entry
points, from single small calls to training steps and serving batches.

listed() gives the fixed cases, draw(rng) one more of the same ranges; prepare / run / work /
exact make a case's inputs and plans, run one pass, count its compulsory work and give its
outputs in 64 bits. Kinds of cases:

  plan    make_plan(descriptor) and Plan.execute, out of place: 1-D, 2-D and 3-D, c2c / r2c /
          c2r, fp32 / fp64, the layouts M x N1 x .. x Nd x K of the descriptors
  trip    two plans: a transform and its unnormalised inverse, as in one step of a spectral
          solver (the smallest calls come in such pairs)
  half    make_half_input_plan: c2c fp32 whose input is stored as f16 or bf16 pairs, through
          the matrix cores or the vector kernel
  filter  a differentiated spectral filter, irfftn(rfftn(x) * H) * scale and its gradient
  ragged  make_ragged_plan: many c2c jobs of mixed lengths and batch counts in one launch
"""
import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "double-batched-fft-library_amd"))

import bbfft_amd as bb  # noqa: E402
from bbfft_amd import autograd, ragged  # noqa: E402

POWERS = (16, 32, 64, 128, 256, 512)
# lengths of the tests, the benchmark sweep and the serving mix that are no powers of two
COMPOSITE = (12, 27, 60, 63, 96, 100, 102, 105, 212, 220, 243, 300, 315, 363, 384, 500)


def _plan(name, desc):
    return {"name": name, "kind": "plan", "desc": desc}


def _trip(name, desc):
    return {"name": name, "kind": "trip", "desc": desc}


def listed():
    return [
        # a time step over a small field, to its spectrum and back: launch latency
        _trip("trip_r2c_m1_n64_k16", "srfo1.64*16"),
        # the CPU configuration's shape on the GPU: a batch of contiguous short signals, to
        # their spectra and back
        _trip("trip_c2c_m1_n64_k16384", "scfo1.64*16384"),
        # the benchmark's headline: double-batched, eight interleaved columns
        _plan("c2c_m8_n256_k32768", "scfo8.256*32768"),
        # double precision, three interleaved fields (a vector quantity), backward
        _plan("c2c_f64_m3_n100_k32768", "dcbo3.100*32768"),
        # odd sizes in every mode (the lengths of the known-answer tests)
        _plan("c2c_m17_n363_k2048", "scfo17.363*2048"),
        # a prime length, which no radix splits
        _plan("c2c_m8_n509_k8192", "scfo8.509*8192"),
        # spectra of a batch of contiguous real frames
        _plan("r2c_m1_n512_k65536", "srfo1.512*65536"),
        # back to real fields of odd length in double precision, five interleaved columns
        _plan("c2r_f64_m5_n315_k8192", "drbo5.315*8192"),
        # real 3-D fields from their spectra, sizes of a solver grid
        _plan("c2r_96x96x80_k16", "srbo96x96x80*16"),
        # one layer of a spectral network: forward and backward of a filtered 3-D transform
        {"name": "filter_32x128x128x128", "kind": "filter", "batch": 32, "n1": 128, "n2": 128,
         "n3": 128},
        # half-precision storage, the first stage on the matrix cores
        {"name": "half_f16_m4_n512_k262144", "kind": "half", "storage": "f16", "mfma": True,
         "desc": "scfo4.512*262144"},
        # serving: mixed lengths, batch counts and directions in one launch
        {"name": "ragged_256_jobs", "kind": "ragged", "jobs": 256, "seed": 2002, "k_max": 16384,
         "lengths": ",".join(str(n) for n in ragged.SERVING_LENGTHS)},
    ]


def _log_uniform(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _length(rng):
    u = rng.random()
    if u < 0.4:
        return rng.choice(POWERS)
    return rng.choice(COMPOSITE) if u < 0.8 else rng.randint(8, 512)


def _largest_prime(n):
    p, d = 1, 2
    while n > 1:
        while n % d == 0:
            n //= d
            p = d
        d += 1
    return p


def draw(rng):
    u = rng.random()
    if u < 0.08:
        n = [rng.choice((32, 48, 64, 96, 128)) for _ in range(3)]
        batch = _log_uniform(rng, 1, max(1, (1 << 25) // math.prod(n)))
        return {"kind": "filter", "batch": batch, "n1": n[0], "n2": n[1], "n3": n[2]}
    if u < 0.16:
        mfma = rng.random() < 0.5
        N = rng.choice((32, 64, 128, 256, 384, 512)) if mfma else _length(rng)
        if _largest_prime(N) > 64:
            N = 500
        M = _log_uniform(rng, 1, 16)
        K = max(1, _log_uniform(rng, 1 << 16, 1 << 26) // (M * N))
        return {"kind": "half", "storage": rng.choice(("f16", "bf16")), "mfma": mfma,
                "desc": f"sc{rng.choice('fb')}o{M}.{N}*{K}"}
    if u < 0.22:
        lengths = sorted(rng.sample(ragged.SERVING_LENGTHS, 2))
        return {"kind": "ragged", "jobs": _log_uniform(rng, 16, 256),
                "seed": rng.randint(0, 1 << 20), "k_max": _log_uniform(rng, 512, 8192),
                "lengths": ",".join(str(n) for n in lengths)}
    prec = "s" if rng.random() < 0.65 else "d"
    domain = rng.choice(("cf", "cb", "rf", "rb"))
    ndim = 1 if u < 0.8 else rng.choice((2, 3))
    M = _log_uniform(rng, 1, 64) if rng.random() < 0.7 else rng.choice((1, 8))
    if ndim == 1:
        N = [_length(rng)]
    else:
        M = rng.choice((1, 1, 1, 3))
        N = [rng.choice((8, 16, 24, 32, 48, 60, 64, 80, 96, 128)) for _ in range(ndim)]
    most = 1 << (25 if prec == "s" else 24)
    if _largest_prime(N[0]) > 64:
        most = 1 << 22
    K = max(1, _log_uniform(rng, 1 << 10, most) // (M * math.prod(N)))
    kind = "trip" if M * math.prod(N) * K < 1 << 20 else "plan"
    if kind == "trip" and domain == "rb":
        domain = "rf"
    return {"kind": kind,
            "desc": f"{prec}{domain}o{M}." + "x".join(str(n) for n in N) + f"*{K}"}


# ---- inputs --------------------------------------------------------------------------------
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _real_of(cfg):
    return torch.float32 if int(cfg.fp) == 4 else torch.float64


def _complex_of(cfg):
    return torch.complex64 if int(cfg.fp) == 4 else torch.complex128


def _shapes(cfg):
    """Row-major shapes (K, Nd, .., N1, M) of the real side and of the half-spectrum side."""
    M, N, K = cfg.shape[0], list(cfg.shape[1:cfg.dim + 1]), cfg.shape[cfg.dim + 1]
    full = [K] + N[::-1] + [M]
    half = list(full)
    half[-2] = N[0] // 2 + 1
    return full, half


def _uniform_complex(shape, cfg, g):
    x = torch.empty(list(shape) + [2], dtype=_real_of(cfg), device="cuda")
    return torch.view_as_complex(x.uniform_(-1.0, 1.0, generator=g))


def _normal(shape, dtype, g):
    return torch.empty(shape, dtype=dtype, device="cuda").normal_(generator=g)


def _plan_input(cfg, seed):
    """c2c: uniform values; r2c: a normal field; c2r: the spectrum of a normal field."""
    g = _generator(seed)
    full, half = _shapes(cfg)
    if cfg.type == bb.transform_type.c2c:
        return _uniform_complex(full, cfg, g)
    field = _normal(full, _real_of(cfg), g)
    if cfg.type == bb.transform_type.r2c:
        return field
    dims = list(range(1, cfg.dim + 1))
    x = torch.fft.fftn(field.to(_complex_of(cfg)), dim=dims)
    x = x.narrow(cfg.dim, 0, half[-2]).contiguous()
    return x / math.sqrt(math.prod(cfg.shape[1:cfg.dim + 1]))


def _inverse(desc):
    """Descriptor of the unnormalised inverse of a forward or backward descriptor."""
    return desc[:2] + ("b" if desc[2] == "f" else "f") + desc[3:]


def _half_input(case, seed):
    cfg = bb.parse_fft_descriptor(case["desc"])
    dtype = torch.float16 if case["storage"] == "f16" else torch.bfloat16
    x = torch.empty(_shapes(cfg)[0] + [2], dtype=torch.float32, device="cuda")
    return x.uniform_(-1.0, 1.0, generator=_generator(seed)).to(dtype)


def _filter_inputs(case, seed):
    g = _generator(seed)
    shape = [case["batch"], case["n3"], case["n2"], case["n1"]]
    x = _normal(shape, torch.float32, g)
    gy = _normal(shape, torch.float32, g)
    h = torch.view_as_complex(_normal(shape[1:3] + [case["n1"] // 2 + 1, 2], torch.float32, g))
    return x, gy, h


def _jobs(case):
    return ragged.synthetic_serving_jobs(case["jobs"], case["seed"],
                                         tuple(int(n) for n in case["lengths"].split(",")),
                                         k_max=case["k_max"])


def _ragged_input(case, seed):
    n = ragged.total_elements(_jobs(case))
    x = torch.empty([n, 2], dtype=torch.float32, device="cuda")
    return torch.view_as_complex(x.uniform_(-1.0, 1.0, generator=_generator(seed)))


def prepare(case, seed):
    kind = case["kind"]
    if kind == "filter":
        x, gy, h = _filter_inputs(case, seed)
        return {"kind": kind, "x": x.requires_grad_(), "gy": gy, "h": h, "n1": case["n1"],
                "scale": 1.0 / (case["n1"] * case["n2"] * case["n3"])}
    if kind == "ragged":
        x = _ragged_input(case, seed)
        return {"kind": kind, "x": x, "y": torch.empty_like(x),
                "plan": ragged.make_ragged_plan(_jobs(case), cache=bb.default_cache())}
    cfg = bb.parse_fft_descriptor(case["desc"])
    full, half = _shapes(cfg)
    if kind == "half":
        return {"kind": kind, "x": _half_input(case, seed),
                "y": torch.empty(full, dtype=torch.complex64, device="cuda"),
                "plan": bb.make_half_input_plan(cfg, case["storage"], case["mfma"],
                                                cache=bb.default_cache())}
    if cfg.type == bb.transform_type.c2r:
        y = torch.empty(full, dtype=_real_of(cfg), device="cuda")
    else:
        y = torch.empty(full if cfg.type == bb.transform_type.c2c else half,
                        dtype=_complex_of(cfg), device="cuda")
    state = {"kind": kind, "x": _plan_input(cfg, seed), "y": y,
             "plan": bb.make_plan(cfg, cache=bb.default_cache())}
    if kind == "trip":
        state["z"] = torch.empty_like(state["x"])
        state["inverse"] = bb.make_plan(_inverse(case["desc"]), cache=bb.default_cache())
    return state


def run(state):
    if state["kind"] == "filter":
        x = state["x"]
        y = autograd.irfftn(autograd.rfftn(x, 3), state["n1"], 3, filter=state["h"],
                            scale=state["scale"])
        (gx,) = torch.autograd.grad(y, x, state["gy"])
        return {"y": y.detach(), "gx": gx}
    state["plan"].execute(state["x"], state["y"])
    if state["kind"] == "trip":
        state["inverse"].execute(state["y"], state["z"])
        return [state["y"], state["z"]]
    return state["y"]


# ---- compulsory work -----------------------------------------------------------------------
def work(case):
    """Every input read once and every output written once; 5 N log2 N flops per complex
    transform, half of that per real one."""
    kind = case["kind"]
    if kind == "filter":
        n = case["n1"] * case["n2"] * case["n3"]
        spec = n // case["n1"] * (case["n1"] // 2 + 1)
        return {"bytes": 4 * 4 * n * case["batch"] + 8 * spec,
                "flops": case["batch"] * (4 * 2.5 * n * math.log2(n) + 2 * 6 * spec)}
    if kind == "ragged":
        jobs = _jobs(case)
        return {"bytes": sum(16 * j.elements for j in jobs),
                "flops": sum(5 * math.log2(j.N) * j.elements for j in jobs)}
    cfg = bb.parse_fft_descriptor(case["desc"])
    full, half = (math.prod(s) for s in _shapes(cfg))
    flops = 5 * math.log2(math.prod(cfg.shape[1:cfg.dim + 1])) * full
    if kind == "half":
        return {"bytes": 12 * full, "flops": flops}
    if cfg.type == bb.transform_type.c2c:
        io = 2 * int(cfg.fp) * full, 2 * int(cfg.fp) * full
    else:
        io, flops = (int(cfg.fp) * full, 2 * int(cfg.fp) * half), flops / 2
    if kind == "trip":  # x is read, the spectrum y and the field z are written
        return {"bytes": 2 * io[0] + io[1], "flops": 2 * flops}
    return {"bytes": sum(io), "flops": flops}


# ---- 64-bit values -------------------------------------------------------------------------
def _dft64(x, dims, sign):
    if sign < 0:
        return torch.fft.fftn(x, dim=dims)
    return torch.fft.ifftn(x, dim=dims, norm="forward")


def _c2r64(x, ndim, n1):
    """Unnormalised c2r over dims ndim .. 1 (dim ndim is the half one): the imaginary part of
    the zero bin is ignored, that of bin n1 / 2 is subtracted from every sample."""
    if ndim > 1:
        x = _dft64(x, list(range(1, ndim)), 1)
    bins = x.shape[ndim]
    y = x.narrow(ndim, 0, 1).real.expand(*x.shape[:ndim], n1, *x.shape[ndim + 1:])
    rest = x.narrow(ndim, 1, bins - 1)
    pad = [*x.shape[:ndim], n1, *x.shape[ndim + 1:]]
    z = torch.zeros(pad, dtype=x.dtype, device=x.device)
    z.narrow(ndim, 1, bins - 1).copy_(rest)
    if n1 % 2 == 0:
        mid = x.narrow(ndim, bins - 1, 1)
        z.narrow(ndim, bins - 1, 1).copy_(torch.complex(mid.real / 2, torch.zeros_like(mid.real)))
        y = y - mid.imag
    return y + 2 * _dft64(z, [ndim], 1).real


def exact(case, seed):
    kind = case["kind"]
    if kind == "filter":
        x, gy, h = (t.to(torch.complex128 if t.is_complex() else torch.float64)
                    for t in _filter_inputs(case, seed))
        scale = 1.0 / (case["n1"] * case["n2"] * case["n3"])

        def filtered(t, w):
            return _c2r64(torch.fft.fftn(t, dim=[1, 2, 3])[..., :w.shape[-1]] * w, 3,
                          case["n1"]) * scale

        # gradient: the adjoint of each map, written as the gradient of the 64-bit graph
        xs = x.requires_grad_()
        y = filtered(xs, h)
        (gx,) = torch.autograd.grad(y, xs, gy)
        return {"y": y.detach(), "gx": gx}
    if kind == "ragged":
        x = _ragged_input(case, seed)
        y = torch.empty(x.shape, dtype=torch.complex128, device="cuda")
        for j in _jobs(case):
            v = x[j.in_offset:j.in_offset + j.elements].view(j.K, j.N, j.M)
            y[j.out_offset:j.out_offset + j.elements] = \
                _dft64(v.to(torch.complex128), [1], j.direction).reshape(-1)
        return y
    cfg = bb.parse_fft_descriptor(case["desc"])
    dims = list(range(1, cfg.dim + 1))
    if kind == "half":
        x = torch.view_as_complex(_half_input(case, seed).to(torch.float64))
        return _dft64(x, dims, int(cfg.dir))
    x = _plan_input(cfg, seed)
    if cfg.type == bb.transform_type.c2c:
        y = _dft64(x.to(torch.complex128), dims, int(cfg.dir))
        return [y, _dft64(y, dims, -int(cfg.dir))] if kind == "trip" else y
    if cfg.type == bb.transform_type.r2c:
        y = torch.fft.fftn(x.to(torch.float64).to(torch.complex128), dim=dims)
        y = y.narrow(cfg.dim, 0, cfg.shape[1] // 2 + 1).contiguous()
        return [y, _c2r64(y, cfg.dim, cfg.shape[1])] if kind == "trip" else y
    return _c2r64(x.to(torch.complex128), cfg.dim, cfg.shape[1])
