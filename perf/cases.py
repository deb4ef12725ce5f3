"""The calls whose speed this framework is judged by: what each stands for, its
inputs, one pass through the public entry points, and the bytes it must move.

    listed()            the fixed cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) inputs and the buffers a program keeps between calls
    run(state)          one pass
    work(case)          bytes a pass cannot do without
    exact(case, seed)   the decoded values in 64 bits, without this package

A case is a dict: "op" (below), "n" values of "dtype" ("f32" / "f64"), SZp block
size "B", team size "T", the reference's fastMode "mode", the bound ("err" =
"rel" or "abs", "eb") and the field's "kind".

    compress      DeviceCodec.compress into the caller's buffers ("index": with
                  the side index)
    decompress    DeviceCodec.decompress with the side index
    foreign       DeviceCodec.decompress of a bare stream (as the reference, or
                  a compress without the index, writes it)
    batch_compress, batch_decompress
                  one launch over "count" fields of "lo" .. "hi" bytes
    host          the drop-in C entry points on host memory, there and back
"""
import ctypes
import math

import numpy as np
import torch

import szp_amd
from szp_amd import ABS, REL, SZ_DOUBLE, SZ_FLOAT
from szp_amd.batch import CompressBatch, DecompressBatch

DEV = "cuda"


def _c(name, op, n, B=128, T=16, dtype="f32", mode=1, err="rel", eb=1e-4, kind="grf", **more):
    return dict(name=name, op=op, n=n, B=B, T=T, dtype=dtype, mode=mode, err=err, eb=eb, kind=kind,
                **more)


def listed():
    return [
        # The smallest requests a server gets (64 KB): launches and latency count.
        _c("small_compress", "compress", 1 << 14, eb=1e-3, kind="sinusoids", index=True),
        # A small stream from elsewhere, of an odd length.
        _c("small_foreign", "foreign", 100003, B=32, T=8, eb=1e-3, kind="zeroblocks"),
        # A medium field with a block size that is no multiple of 8 and an
        # absolute bound, as a caller of the bare format may choose.
        _c("odd_compress_abs", "compress", 16000001, B=100, T=7, err="abs", eb=1e-3, index=False),
        # The headline workload: a 512^3 simulation field held on the GPU,
        # compressed with its side index, ...
        _c("field_compress", "compress", 512 ** 3, index=True),
        # ... read back with it, ...
        _c("field_decompress", "decompress", 512 ** 3),
        # ... and read back from the bare stream, as a file written by the
        # reference is.
        _c("field_foreign", "foreign", 512 ** 3),
        # Double-precision fields, both ways.
        _c("double_compress", "compress", 384 ** 3, dtype="f64", index=True),
        _c("double_foreign", "foreign", 384 ** 3, B=64, dtype="f64", eb=1e-2),
        # The random-access format (units that restart the chain).
        _c("ra_foreign", "foreign", 384 ** 3, mode=2),
        # Many uneven fields at once (a checkpoint's arrays), both ways.
        _c("batch_compress", "batch_compress", 0, eb=1e-3, kind="mix", count=256, lo=64 << 10,
           hi=64 << 20),
        _c("batch_decompress", "batch_decompress", 0, eb=1e-3, kind="mix", count=256, lo=64 << 10,
           hi=64 << 20),
        # The drop-in C calls on host arrays, as an existing program makes them.
        _c("host_roundtrip", "host", 1 << 24, err="abs", eb=1e-3, kind="sinusoids"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["compress", "compress", "decompress", "decompress", "foreign", "foreign",
                     "foreign", "batch_compress", "batch_decompress", "host"])
    eb = 10.0 ** rng.uniform(-4.0, -2.0)
    B = rng.choice([8, 16, 32, 64, 128, 128, 256])
    if op.startswith("batch"):
        c = _c("", op, 0, B=B, T=rng.choice([1, 4, 8, 16]), eb=eb, kind="mix",
               count=_log_int(rng, 4, 128), lo=16 << 10, hi=_log_int(rng, 1 << 20, 32 << 20))
    elif op == "host":
        c = _c("", op, _log_int(rng, 1 << 12, 1 << 24), B=B, T=rng.choice([1, 4, 8, 16]),
               err="abs", eb=eb, kind=rng.choice(["sinusoids", "grf"]))
    else:
        dtype = rng.choice(["f32", "f32", "f32", "f64"])
        hi = 1 << (25 if dtype == "f64" else 26)
        if rng.random() < 0.2:  # a block size of no special form
            B, hi = _log_int(rng, 5, 2000), 1 << 24
        c = _c("", op, _log_int(rng, 1 << 12, hi), B=B, T=rng.choice([1, 3, 8, 16, 16, 40]),
               dtype=dtype, mode=rng.choice([1, 1, 1, 2]), err=rng.choice(["rel", "rel", "abs"]),
               eb=eb, kind=rng.choice(["grf", "grf", "sinusoids", "zeroblocks", "noise"]))
        if op == "compress":
            c["index"] = rng.random() < 0.6
    del c["name"]
    return c


# ---- inputs -----------------------------------------------------------------

def _grf(n, gen):
    """The first n values, in C order, of a cube with the isotropic spectrum
    k^-3 (edges 2^k and 3 * 2^k: few transform lengths)."""
    e = next(s for k in range(3, 12) for s in (1 << k, 3 << (k - 1)) if s ** 3 >= n)
    F = torch.fft.rfftn(torch.randn((e, e, e), generator=gen, device=DEV))
    k = torch.fft.fftfreq(e, device=DEV)
    kz = torch.fft.rfftfreq(e, device=DEV)
    k2 = k.view(e, 1, 1) ** 2 + k.view(1, e, 1) ** 2 + kz.view(1, 1, -1) ** 2
    k2[0, 0, 0] = 1.0
    F *= k2.pow(-0.75)
    F[0, 0, 0] = 0
    return torch.fft.irfftn(F, s=(e, e, e)).reshape(-1)[:n]


def _sinusoids(n, gen):
    """Eight sinusoids of 1e-6 .. 1e-3 cycles per value, and 1e-3 of noise."""
    f, a, ph = torch.rand(3, 8, generator=gen, device=DEV, dtype=torch.float64).tolist()
    i = torch.arange(n, device=DEV, dtype=torch.float64)
    x = torch.zeros(n, device=DEV, dtype=torch.float64)
    for s in range(8):
        x += (0.1 + 0.9 * a[s]) * torch.sin(i * (2 * math.pi * 10 ** (-6 + 3 * f[s]))
                                            + 2 * math.pi * ph[s])
    return x.float() + 1e-3 * torch.randn(n, generator=gen, device=DEV)


def _field(kind, n, gen):
    if kind == "noise":
        return torch.rand(n, generator=gen, device=DEV) * 2 - 1
    x = _sinusoids(n, gen) if kind == "sinusoids" else _grf(n, gen)
    mn, mx = torch.aminmax(x)
    x = (x - mn) / (mx - mn) * 2 - 1
    if kind == "zeroblocks":  # a fifth of it masked out, in runs of 128
        z = torch.rand((n + 127) // 128, generator=gen, device=DEV) < 0.2
        x = x.masked_fill(z.repeat_interleave(128)[:n], 0.0)
    return x.contiguous()


def _generator(seed):
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    return gen


def _sizes(case):
    """Values per field of a batch: the same for every seed, uneven."""
    u = np.random.default_rng(case["count"] * 1000003 + case["hi"]).uniform(
        math.log(case["lo"]), math.log(case["hi"]), case["count"])
    return [max(1, int(math.exp(v)) // 4) for v in u]


def _inputs(case, seed):
    gen = _generator(seed)
    if case["kind"] != "mix":
        x = _field(case["kind"], case["n"], gen)
        return x.double() if case["dtype"] == "f64" else x
    kinds = ("grf", "noise", "zeroblocks", "sinusoids")
    return [_field(kinds[k % 4], n, gen) for k, n in enumerate(_sizes(case))]


def _bound(case):
    return (REL, 0.0, case["eb"]) if case["err"] == "rel" else (ABS, case["eb"], 0.0)


def prepare(case, seed):
    op, B, T = case["op"], case["B"], case["T"]
    x = _inputs(case, seed)
    if op.startswith("batch"):
        cb = CompressBatch(x, _bound(case), block_size=B, threads=T)
        cb.out.zero_()
        cb.index.zero_()
        if op == "batch_compress":
            return {"op": op, "batch": cb}
        cb.launch()
        cb.check()
        ns = [v.numel() for v in x]
        at = np.concatenate([[0], np.cumsum([(n + 63) // 64 * 64 for n in ns])])
        flat = torch.zeros(int(at[-1]), device=DEV)
        outs = [flat[int(a):int(a) + n] for a, n in zip(at, ns)]
        sizes = cb.byte_sizes()
        db = DecompressBatch([cb.stream(k, s) for k, s in enumerate(sizes)], sizes, ns,
                             [cb.index_of(k) for k in range(len(ns))], block_size=B, threads=T,
                             outs=outs)
        return {"op": op, "batch": db, "flat": flat}
    n, dt = case["n"], SZ_DOUBLE if case["dtype"] == "f64" else SZ_FLOAT
    cap = szp_amd.compress_bound(n, B, T, dt, case["mode"])
    if op == "host":
        return {"op": op, "x": x.cpu().numpy(), "out": np.zeros(cap, np.uint8), "eb": case["eb"],
                "values": np.zeros(n, np.float32), "B": B, "T": T}
    codec = szp_amd.DeviceCodec(block_size=B, threads=T, fast_mode=case["mode"])
    out = torch.zeros(cap, dtype=torch.uint8, device=DEV)
    idx = None
    if case.get("index") or op == "decompress":
        idx = torch.zeros(codec.index_size(n), dtype=torch.uint8, device=DEV)
    state = {"op": op, "codec": codec, "x": x, "bound": _bound(case), "out": out, "index": idx}
    if op == "compress":
        return state
    em, ab, rel = _bound(case)
    size = codec.compress(x, em, ab, rel, out=out, index=idx)[1]
    codec.check()
    state.update(stream=out[:int(size.item())].clone(), n=n, values=torch.zeros_like(x), x=None,
                 out=None)
    return state


def run(state):
    op = state["op"]
    if op == "compress":
        em, ab, rel = state["bound"]
        return list(state["codec"].compress(state["x"], em, ab, rel, out=state["out"],
                                            index=state["index"]))
    if op in ("decompress", "foreign"):
        st = state["stream"]
        return state["codec"].decompress(st, st.numel(), state["n"], out=state["values"],
                                         index=state["index"])
    if op == "batch_compress":
        b = state["batch"]
        b.launch()
        return [b.out, b.sizes, b.index]
    if op == "batch_decompress":
        state["batch"].launch()
        return state["flat"]
    x, out, values, lib = state["x"], state["out"], state["values"], szp_amd.lib
    szp_amd.set_threads(state["T"])
    size = ctypes.c_size_t(0)
    lib.szp_float_openmp_threadblock_arg(out.ctypes.data, x.ctypes.data, ctypes.byref(size),
                                         state["eb"], x.size, state["B"])
    lib.szp_float_decompress_openmp_threadblock_arg(values.ctypes.data, x.size, state["eb"],
                                                    state["B"], out.ctypes.data + 4)
    return [out, int(size.value), values]


# ---- what a pass cannot do without ------------------------------------------

def _stream_bytes(kind, n, eb, B):
    """About what a stream of n values takes (from the entropy of the deltas
    at this bound, one sign bit each and a width byte per block)."""
    if kind == "mix":
        return sum(_stream_bytes(k, n, eb, B) for k in ("grf", "noise", "zeroblocks", "sinusoids")) / 4
    scale = {"grf": 0.4, "zeroblocks": 0.4, "noise": 2.0, "sinusoids": 0.002}[kind]
    bits = max(0.3, math.log2(max(scale / eb, 1.0)))
    return n * ((bits + 1) / 8 * (0.8 if kind == "zeroblocks" else 1.0) + 1.0 / B)


def work(case):
    B, op = case["B"], case["op"]
    n = sum(_sizes(case)) if case["kind"] == "mix" else case["n"]
    eb = case["eb"] * (2 if case["err"] == "rel" else 1)  # the fields span [-1, 1]
    field = n * (8 if case["dtype"] == "f64" else 4)
    b = field + _stream_bytes(case["kind"], n, eb, B)
    if case.get("index") or "decompress" in op or op == "batch_compress":
        b += 8 * n / B
    return {"bytes": float(b * (2 if op == "host" else 1)), "flops": 0.0}


# ---- the decoded values in 64 bits ------------------------------------------

def _values(x, case):
    """trunc(x * fl(1 / eb)) * eb, with eb and 1 / eb in the field's own type
    (the format's definition) and the rest in double."""
    if case["err"] == "rel":
        mn, mx = torch.aminmax(x)
        eb = (mx - mn) * torch.tensor(case["eb"], dtype=x.dtype, device=x.device)
    else:
        eb = torch.tensor(case["eb"], dtype=x.dtype, device=x.device)
    inv = torch.ones((), dtype=x.dtype, device=x.device) / eb
    return torch.trunc(x.double() * inv.double()) * eb.double()


def exact(case, seed):
    op = case["op"]
    if op in ("compress", "batch_compress"):
        return None  # bytes
    x = _inputs(case, seed)
    if op == "batch_decompress":
        parts = []
        for v in x:
            parts += [_values(v, case), torch.zeros(-v.numel() % 64, device=DEV, dtype=torch.float64)]
        return torch.cat(parts)
    y = _values(x, case)
    if op == "host":
        return [None, None, y.cpu().numpy()]
    if case["mode"] == 2 and case["B"] == 1:
        return None
    return y
