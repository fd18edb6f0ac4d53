"""Work that a program on this library has the GPU do, case by case: buffers
compressed, decompressed and summed while compressed, alone and in batches,
streams adopted from elsewhere, a staged allreduce, and 3-D volumes.

Sizes, fields and error bounds are those of bench.py, zccl_amd/workloads.py
and the GPU tests: FP32 buffers from 64 KiB (the smallest served request) to
8 x 512^3 values, blocks of 36 values (the reference's default) and the chunk
counts T its OpenMP team gives.  A program keeps its output buffers, index,
workspace and plans from call to call, and so do the states here.
"""
import math

import torch

L = 36

# Compressed bytes per value by field and bound (relative to the range of the
# values; absolute for "sines" and "velocity"), as the streams of these fields
# come out: for work() alone.
BYTES_PER_VALUE = {
    ("field", 1e-2): 0.70, ("field", 1e-3): 1.13, ("field", 1e-4): 1.55,
    ("sines", 1e-2): 0.37, ("sines", 1e-3): 0.69, ("sines", 1e-4): 1.10,
    ("gradient", 1e-2): 0.20, ("gradient", 1e-3): 0.63, ("gradient", 1e-4): 1.06,
    ("slabs", 1e-2): 0.23, ("slabs", 1e-3): 0.36, ("slabs", 1e-4): 0.49,
    ("velocity", 1e-2): 2.16, ("velocity", 1e-4): 2.98,
}
# Compressed bytes per value of a volume by block side, at relative 1e-3.
BYTES_PER_VALUE_3D = {4: 1.02, 8: 1.04}


# ---------------------------------------------------------------- fields

def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _grf(side, seed):
    """Gaussian random field on a side^3 grid, P(k) ~ k^-3, unit deviation."""
    w = torch.randn((side, side, side), generator=_generator(seed), device="cuda")
    f = torch.fft.rfftn(w)
    del w
    k1, kz = torch.fft.fftfreq(side, device="cuda"), torch.fft.rfftfreq(side, device="cuda")
    kk = k1[:, None, None] ** 2 + k1[None, :, None] ** 2 + kz[None, None, :] ** 2
    kk[0, 0, 0] = 1.0
    f *= kk.pow_(-0.75)
    f[0, 0, 0] = 0
    x = torch.fft.irfftn(f, s=(side, side, side))
    return x / x.std()


def _values(kind, n, seed):
    """n FP32 values of a kind of field, flat."""
    if kind == "sines":
        g = torch.Generator()
        g.manual_seed(int(seed))
        u = torch.rand((3, 16), generator=g, dtype=torch.float64)
        period = torch.exp(math.log(64) + u[0] * (math.log(65536) - math.log(64)))
        amp, phase = 0.1 + 0.9 * u[1], 2 * math.pi * u[2]
        i = torch.arange(n, device="cuda", dtype=torch.float64)
        x = 1e-3 * torch.randn(n, generator=_generator(seed), device="cuda", dtype=torch.float64)
        for p, a, ph in zip(period.tolist(), amp.tolist(), phase.tolist()):
            x += a * torch.sin(i * (2 * math.pi / p) + ph)
        return x.float()
    if kind == "gradient":
        g = _generator(seed)
        x = 1e-2 * torch.randn(n, generator=g, device="cuda")
        return torch.where(torch.rand(n, generator=g, device="cuda") < 0.01, 100 * x, x)
    side = 16
    while side ** 3 < n:
        side *= 2
    x = _grf(side, seed).reshape(-1)[:n].clone()
    if kind == "velocity":
        x *= 300.0
    elif kind == "slabs":
        # exact zeros over 70 % of the values, in contiguous runs
        run = max(n // 40, 1)
        keep = torch.rand(n // run + 1, generator=_generator(seed + 1), device="cuda") < 0.3
        x *= keep[torch.arange(n, device="cuda") // run]
    return x


def _perturbed(base, amount, seed):
    return base + amount * torch.randn(base.shape, generator=_generator(seed), device="cuda")


def _f32(v):
    return float(torch.tensor(v, dtype=torch.float32).item())


def _bound(kind, rel, x):
    """The absolute bound of a call: `rel` times the range of the values, or
    `rel` itself for the fields whose bound is given in their own unit."""
    if kind in ("sines", "velocity"):
        return _f32(rel)
    return _f32(_f32(float((x.max() - x.min()).item())) * _f32(rel)) or _f32(rel)


# ---------------------------------------------------------------- states

def _stream(n, T, data=None):
    """A stream with room for n values, its unused bytes zero."""
    from zccl_amd import codec

    if data is None:
        data = torch.zeros(codec.worst_case_bytes(n, L, T), dtype=torch.uint8, device="cuda")
    return codec.DeviceStream(data, torch.zeros(codec.index_bytes(n, L, T), dtype=torch.uint8, device="cuda"), n, L, T)


def _resident(s):
    """A finished stream, its buffer cut to its bytes."""
    from zccl_amd import codec

    return codec.DeviceStream(s.data[: s.size].clone(), s.index, s.n, s.L, s.T)


def _compressed(x, eb, T):
    from zccl_amd import codec

    return _resident(codec.compress(x, eb, L, T))


def _views(sizes, T):
    """Streams of these sizes over one flat buffer, and that buffer."""
    from zccl_amd import codec

    caps = [(codec.worst_case_bytes(n, L, T) + 255) // 256 * 256 for n in sizes]
    flat = torch.zeros(sum(caps), dtype=torch.uint8, device="cuda")
    outs, at = [], 0
    for n, cap in zip(sizes, caps):
        outs.append(_stream(n, T, flat[at: at + cap]))
        at += cap
    return outs, flat


def _bucket_sizes(case):
    """Log-uniform buffer sizes (values) between 4 KB and the case's largest."""
    g = torch.Generator()
    g.manual_seed(case["sizes"])
    u = torch.rand(case["buffers"], generator=g, dtype=torch.float64)
    lo, hi = math.log(4096), math.log(case["largest"])
    return [int(math.exp(lo + v * (hi - lo))) // 4 for v in u.tolist()]


def _ranks(case, seed):
    """Every rank's values of a staged allreduce."""
    n = case["n"]
    base = _values(case["kind"], n, seed)
    amount = 0.05 * float(base.std().item())
    return [_perturbed(base, amount, seed + 100 + r) for r in range(case["k"])]


def _volume(case, seed):
    d = (case["d1"], case["d2"], case["d3"])
    side = 16
    while side < max(d):
        side *= 2
    x = _grf(side, seed)[: d[0], : d[1], : d[2]].contiguous()
    return x, float((x.max() - x.min()).item()) * case["rel"]


def prepare(case, seed):
    from zccl_amd import allreduce, batch, codec, sz3d

    op, T = case["op"], case["T"]
    st = {"case": case}
    if op == "compress":
        st["x"] = _values(case["kind"], case["n"], seed)
        st["eb"] = _bound(case["kind"], case["rel"], st["x"])
        st["out"] = _stream(case["n"], T)
        st["ws"] = codec.Workspace(codec.num_tiles(case["n"], L, T))
    elif op == "decompress":
        x = _values(case["kind"], case["n"], seed)
        st["eb"] = _bound(case["kind"], case["rel"], x)
        st["s"] = _compressed(x, st["eb"], T)
        st["y"] = torch.empty(case["n"], device="cuda")
        st["ws"] = codec.Workspace(codec.num_tiles(case["n"], L, T))
    elif op == "adopt":
        x = _values(case["kind"], case["n"], seed)
        st["eb"] = _bound(case["kind"], case["rel"], x)
        st["bytes"] = _compressed(x, st["eb"], T).data
        st["y"] = torch.empty(case["n"], device="cuda")
    elif op == "sum":
        xs = _ranks(case, seed)
        eb = _bound(case["kind"], case["rel"], xs[0])
        st["ops"] = [_compressed(x, eb, T) for x in xs]
        st["out"] = _stream(case["n"], T)
        st["ws"] = codec.Workspace(codec.num_tiles(case["n"], L, T))
    elif op == "sums":
        # every rank's values in segments; segment j of all ranks is sum j
        n, jobs = case["n"], case["jobs"]
        base = _values(case["kind"], n * jobs, seed)
        amount = 0.05 * float(base.std().item())
        eb = _bound(case["kind"], case["rel"], base)
        outs, st["flat"] = _views([n] * jobs, T)
        streams = []
        for r in range(case["k"]):
            x = _perturbed(base, amount, seed + 100 + r)
            streams.append([_compressed(x[j * n: (j + 1) * n], eb, T) for j in range(jobs)])
        st["plan"] = batch.homsum_plan([[s[j] for s in streams] for j in range(jobs)], outs)
    elif op == "buckets":
        sizes, k = _bucket_sizes(case), case["k"]
        flat = _values("gradient", sum(sizes), seed)
        xs = list(flat.split(sizes))
        ebs = [_bound("gradient", case["rel"], x) for x in xs]
        outs, st["flat"] = _views(sizes, T)
        st["compress"] = batch.compress_plan(xs, ebs, outs)
        st["compress"].launch()
        # the other ranks' streams of the buffers this rank sums (distinct memory)
        owned = outs[::k]
        ops = [[codec.DeviceStream(o.data[: o.size].clone(), o.index.clone(), o.n, L, T) for _ in range(k - 1)] + [o]
               for o in owned]
        sums, st["sums"] = _views([o.n for o in owned], T)
        st["sum"] = batch.homsum_plan(ops, sums)
        st["ws"] = codec.Workspace(max(st["compress"].tiles, st["sum"].tiles))
    elif op == "allreduce":
        st["xs"] = _ranks(case, seed)
        st["eb"] = _bound(case["kind"], case["rel"], st["xs"][0])
        st["ar"] = allreduce.DeviceAllreduce(case["k"], case["n"], st["eb"], L, T)
        st["y"] = torch.empty(case["n"], device="cuda")
    else:
        x, st["eb"] = _volume(case, seed)
        worst, wsb = sz3d.sizes(x.shape, case["side"], T)
        st["ws"] = torch.zeros(wsb, dtype=torch.uint8, device="cuda")
        data = torch.zeros(worst, dtype=torch.uint8, device="cuda")
        if op == "volume-compress":
            st["x"], st["out"] = x, data
        else:
            s = sz3d.compress(x, case["side"], st["eb"], T, out=data, ws=st["ws"])
            st["s"] = sz3d.Stream3D(data[: s.size].clone(), st["ws"], s.dims, s.Bs, s.eb, T)
            st["y"] = torch.empty(x.shape, device="cuda")
    return st


def run(st):
    from zccl_amd import codec, sz3d

    case = st["case"]
    op, T = case["op"], case["T"]
    if op == "compress":
        s = codec.compress(st["x"], st["eb"], L, T, out=st["out"], ws=st["ws"])
        return {"bytes": s.data, "size": s.size_tensor(), "widths": s.widths()}
    if op == "decompress":
        return codec.decompress(st["s"], st["eb"], out=st["y"], ws=st["ws"])
    if op == "adopt":
        s = codec.from_bytes(st["bytes"], case["n"], L, T)
        y = codec.decompress(s, st["eb"], out=st["y"])
        return {"y": y, "size": s.size_tensor(), "widths": s.widths()}
    if op == "sum":
        s = codec.homsum(st["ops"], out=st["out"], ws=st["ws"])
        return {"bytes": s.data, "size": s.size_tensor(), "widths": s.widths()}
    if op == "sums":
        st["plan"].launch()
        return st["flat"]
    if op == "buckets":
        st["compress"].launch(st["ws"])
        st["sum"].launch(st["ws"])
        return {"streams": st["flat"], "sums": st["sums"]}
    if op == "allreduce":
        return st["ar"].run(st["xs"], out=st["y"])
    if op == "volume-compress":
        return sz3d.compress(st["x"], case["side"], st["eb"], T, out=st["out"], ws=st["ws"]).data
    return sz3d.decompress(st["s"], out=st["y"], ws=st["ws"])


# ---------------------------------------------------------------- cases

def listed():
    return [
        # the smallest served request, both ways: launches and latency
        {"name": "compress-64k", "op": "compress", "kind": "field", "n": 16384, "rel": 1e-3, "T": 16},
        {"name": "decompress-64k", "op": "decompress", "kind": "field", "n": 16411, "rel": 1e-3, "T": 16},
        # one large 1-D array, the plain compressor's workload, and back
        {"name": "compress-2p24", "op": "compress", "kind": "sines", "n": 1 << 24, "rel": 1e-4, "T": 16},
        {"name": "decompress-2p24", "op": "decompress", "kind": "field", "n": 1 << 24, "rel": 1e-3, "T": 16},
        # a ring step: two compressed operands of 1 MB added
        {"name": "add-1m", "op": "sum", "kind": "field", "n": 262147, "k": 2, "rel": 1e-3, "T": 8},
        # a gradient bucket of 8 MB summed over 16 ranks, short of a whole tile
        {"name": "sum-bucket", "op": "sum", "kind": "gradient", "n": 2000003, "k": 16, "rel": 1e-3, "T": 16},
        # the reduce-scatter of 8 ranks of 512^3 fields on one device
        {"name": "sums-8x8-2p24", "op": "sums", "kind": "field", "n": 1 << 24, "jobs": 8, "k": 8, "rel": 1e-3, "T": 16},
        # gradient buffers of uneven sizes: all compressed, this rank's summed over 16 ranks
        {"name": "buckets", "op": "buckets", "buffers": 256, "largest": 16 << 20, "sizes": 4096, "k": 16, "rel": 1e-3, "T": 16},
        # a stream that another program wrote: its bytes indexed, then decompressed
        {"name": "adopt-2p24", "op": "adopt", "kind": "field", "n": 1 << 24, "rel": 1e-3, "T": 16},
        # four ranks' velocities allreduced: wide blocks
        {"name": "allreduce-velocity", "op": "allreduce", "kind": "velocity", "n": 1 << 24, "k": 4, "rel": 1e-2, "T": 16},
        # a 512^3 volume through the 3-D codec, both ways
        {"name": "volume-compress-512", "op": "volume-compress", "d1": 512, "d2": 512, "d3": 512, "side": 4, "rel": 1e-3, "T": 16},
        {"name": "volume-decompress-512", "op": "volume-decompress", "d1": 512, "d2": 512, "d3": 512, "side": 4, "rel": 1e-3, "T": 16},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["compress", "decompress", "adopt", "sum", "sum", "sums", "buckets", "allreduce", "volume-compress",
                     "volume-decompress"])
    T = rng.choice([1, 4, 7, 8, 16, 16, 32])
    if op.startswith("volume"):
        d = [_log(rng, 24, 400) for _ in range(3)]
        return {"op": op, "d1": d[0], "d2": d[1], "d3": d[2], "side": rng.choice([4, 4, 8]),
                "rel": rng.choice([1e-2, 1e-3, 1e-4]), "T": rng.choice([1, 4, 8, 16])}
    rel = rng.choice([1e-2, 1e-3, 1e-4])
    if op == "buckets":
        return {"op": op, "buffers": rng.randint(32, 200), "largest": _log(rng, 1 << 20, 16 << 20),
                "sizes": rng.randrange(1 << 20), "k": rng.randint(4, 16), "rel": rel, "T": T}
    kind = rng.choice(["field", "field", "sines", "gradient", "slabs", "velocity"])
    case = {"op": op, "kind": kind, "rel": rng.choice([1e-2, 1e-4]) if kind == "velocity" else rel, "T": T}
    if op == "sum":
        case["k"] = rng.randint(2, 32)
        case["n"] = _log(rng, 16384, 1 << 22)
    elif op == "sums":
        case["jobs"], case["k"] = rng.randint(2, 8), rng.randint(2, 12)
        case["n"] = _log(rng, 16384, 1 << 21)
    elif op == "allreduce":
        case["k"] = rng.randint(2, 8)
        case["n"] = _log(rng, 1 << 17, 1 << 23)
    else:
        case["n"] = _log(rng, 16384, 1 << 24)
    return case


def work(case):
    op = case["op"]
    if op.startswith("volume"):
        n = case["d1"] * case["d2"] * case["d3"]
        return {"bytes": n * (4 + BYTES_PER_VALUE_3D[case["side"]]), "flops": 0}
    if op == "buckets":
        sizes = _bucket_sizes(case)
        b, k = BYTES_PER_VALUE[("gradient", case["rel"])], case["k"]
        return {"bytes": sum(sizes) * (4 + b) + sum(sizes[::k]) * b * (k + 1), "flops": 0}
    n, b = case["n"], BYTES_PER_VALUE[(case["kind"], case["rel"])]
    if op == "sum":
        return {"bytes": n * b * (case["k"] + 1), "flops": 0}
    if op == "sums":
        return {"bytes": n * b * (case["k"] + 1) * case["jobs"], "flops": 0}
    if op == "allreduce":
        # every rank's values read, their streams written and read, the sums
        # written and read, the result written
        return {"bytes": n * (case["k"] * (4 + 2 * b) + 2 * b + 4), "flops": 0}
    return {"bytes": n * (4 + b), "flops": 0}


def _quantized(x, eb):
    """The codec's integers: the bound's FP32 reciprocal, an exact product,
    truncation (in 64 bits)."""
    inv = (torch.tensor(1.0, dtype=torch.float32) / torch.tensor(eb, dtype=torch.float32)).item()
    return torch.trunc(x.double() * inv)


def exact(case, seed):
    op = case["op"]
    if op in ("decompress", "adopt"):
        x = _values(case["kind"], case["n"], seed)
        eb = _bound(case["kind"], case["rel"], x)
        y = _quantized(x, eb) * eb
        return y if op == "decompress" else {"y": y, "size": None, "widths": None}
    if op == "allreduce":
        xs = _ranks(case, seed)
        eb = _bound(case["kind"], case["rel"], xs[0])
        return sum(_quantized(x, eb) for x in xs) * eb
    if op == "volume-decompress":
        x, eb = _volume(case, seed)
        return torch.floor(x.double() * (0.5 / eb) + 0.5) * (2 * eb)
    return None
