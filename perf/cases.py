"""Performance cases of the library: the calls its users make, over their real ranges.

A case is a dict of plain values.  ``listed()`` are the standing ones, ``draw(rng)`` gives
more of the same ranges, ``prepare`` makes a case's inputs, plans and handles on the GPU,
``run`` is one pass through the public entry points, ``work`` what that pass cannot do
without, and ``exact`` its outputs in 64 bits by plain torch on the CPU.

Kinds:
  fft     batched complex64 transforms (``Plan``), 2^6 .. 2^26 points, both directions
  fft16   complex64 data packed to FP16 storage and transformed there
  fft2d   2-D transforms (``Plan2D``)
  uneven  one batch of transforms of many sizes (``UnevenBatch``)
  conv    real rows convolved with one filter (``Convolution``)
  conv16  the same on binary16 rows with per-row scales
  served  a burst of convolution requests through the ``Server``
"""
import math

import torch

import estl_amd
from estl_amd import workloads

DEVICE = "cuda"


def listed():
    return [
        # one transform by itself, as an interactive caller makes it: latency and launches
        {"name": "fft_one_64k", "kind": "fft", "n": 1 << 16, "batch": 1, "dir": -1, "normalize": False},
        # the headline batch: 4096 points, 16384 rows
        {"name": "fft_4096_batch", "kind": "fft", "n": 4096, "batch": 16384, "dir": -1, "normalize": False},
        # short rows, a ragged number of them, scaled inverse
        {"name": "fft_512_ragged", "kind": "fft", "n": 512, "batch": 50001, "dir": 1, "normalize": True},
        # rows too long for one launch, an odd batch, inverse
        {"name": "fft_1m_batch", "kind": "fft", "n": 1 << 20, "batch": 33, "dir": 1, "normalize": True},
        # one very large transform
        {"name": "fft_64m", "kind": "fft", "n": 1 << 26, "batch": 1, "dir": -1, "normalize": False},
        # half the bytes: rows packed to FP16 storage and transformed
        {"name": "fft16_256k", "kind": "fft16", "n": 1 << 18, "batch": 101, "dir": -1, "normalize": False},
        # an image-sized 2-D transform
        {"name": "fft2d_4096", "kind": "fft2d", "nx": 4096, "ny": 4096, "batch": 1, "dir": -1},
        # thousands of transforms of mixed sizes in one call
        {"name": "uneven_8192", "kind": "uneven", "count": 8192, "kmin": 8, "kmax": 18, "mix": 3, "dir": -1},
        # short real rows correlated with a short template, an odd number of rows
        {"name": "conv_1024_rows", "kind": "conv", "n": 1024, "rows": 30001, "k": 129, "corr": True, "center": False,
         "normalize": False, "new_filter": False},
        # long real rows and a long filter, the filter kept
        {"name": "conv_1m_rows", "kind": "conv", "n": 1 << 20, "rows": 63, "k": 2049, "corr": False, "center": False,
         "normalize": False, "new_filter": False},
        # binary16 rows, a longer filter that is new with each call
        {"name": "conv16_256k_rows", "kind": "conv16", "n": 1 << 18, "rows": 101, "k": 6001, "corr": False,
         "center": False, "normalize": False, "new_filter": True},
        # a burst of requests, each with rows, length and filter of its own
        {"name": "served_burst", "kind": "served", "count": 24, "mix": 4, "max_log2": 23},
    ]


def _log_uniform(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _rows(rng, n, lo_log2, hi_log2):
    """A number of rows of n values, the total log-uniform between 2^lo_log2 and 2^hi_log2."""
    return max(1, min(1 << hi_log2, int(2.0 ** rng.uniform(lo_log2, hi_log2))) // n)


def draw(rng):
    kind = rng.choice(["fft"] * 4 + ["fft16", "fft16", "fft2d", "uneven", "conv", "conv", "conv", "conv16", "served"])
    sign = rng.choice([-1, 1])
    if kind in ("fft", "fft16"):
        n = 1 << (rng.randint(6, 26) if kind == "fft" else rng.randint(8, 24))
        return {"kind": kind, "n": n, "batch": _rows(rng, n, 16, 26), "dir": sign, "normalize": rng.random() < 0.4}
    if kind == "fft2d":
        nx, ny = 1 << rng.randint(6, 13), 1 << rng.randint(6, 13)
        return {"kind": kind, "nx": nx, "ny": ny, "batch": _rows(rng, nx * ny, 16, 25), "dir": sign}
    if kind == "uneven":
        kmin = rng.randint(6, 12)
        kmax = rng.randint(kmin + 2, 18)
        most = max(16, min(8192, (1 << 28) >> (kmax - 1)))
        return {"kind": kind, "count": _log_uniform(rng, 16, most), "kmin": kmin, "kmax": kmax,
                "mix": rng.randint(1, 1 << 20), "dir": sign}
    if kind == "served":
        return {"kind": kind, "count": rng.randint(4, 32), "mix": rng.randint(1, 1 << 20), "max_log2": rng.randint(20, 23)}
    n = 1 << rng.randint(10, 22)
    center = rng.random() < 0.25
    return {"kind": kind, "n": n, "rows": _rows(rng, n, 16, 26), "k": rng.randint(16, 8192), "corr": rng.random() < 0.25,
            "center": center, "normalize": center, "new_filter": rng.random() < 0.5}


# ---------------------------------------------------------------- inputs

def _uniform(seed, *shape):
    """uniform [-1, 1) float32 on the GPU, from the seed alone"""
    g = torch.Generator(device=DEVICE).manual_seed(int(seed))
    return torch.rand(*shape, generator=g, device=DEVICE, dtype=torch.float32).mul_(2.0).sub_(1.0)


def _complex(seed, *shape):
    return torch.view_as_complex(_uniform(seed, *shape, 2))


def _taps(seed, k, normalize):
    """A filter: random taps, or, where it is divided by its sum, a positive (smoothing) one."""
    h = _uniform(seed ^ 0x5A5A5A, k)
    return h.mul_(0.5).add_(1.0) if normalize else h


def _conv_flags(case):
    return ((estl_amd.CONV_CORRELATE if case["corr"] else 0) | (estl_amd.CONV_CENTER if case["center"] else 0)
            | (estl_amd.CONV_NORMALIZE_KERNEL if case["normalize"] else 0))


def _uneven_sizes(case):
    return workloads.uneven_batch(case["count"], case["mix"], case["kmin"], case["kmax"])


def _requests(case):
    """The requests of a burst: lengths 2^U{10..22}, rows U{1..256} as far as max_log2
    values a request allow, filters of U{16..8192} taps, a quarter of them correlations."""
    r = workloads.conv_requests(case["count"], case["mix"], log2n=(10, min(22, case["max_log2"])),
                                max_values=1 << case["max_log2"])
    return [(int(n), int(rows), int(k), int(f)) for n, rows, k, f in zip(r.n, r.rows, r.k, r.flags)]


def _served_inputs(case, seed):
    reqs = _requests(case)
    x = _uniform(seed, sum(n * rows for n, rows, _, _ in reqs))
    h = _uniform(seed ^ 0x5A5A5A, sum(k for _, _, k, _ in reqs))
    out, xo, ho = [], 0, 0
    for n, rows, k, flags in reqs:
        out.append((n, rows, flags, x[xo:xo + n * rows], h[ho:ho + k]))
        xo, ho = xo + n * rows, ho + k
    return out


def prepare(case, seed):
    estl_amd.init(0)
    kind = case["kind"]
    if kind in ("fft", "fft16"):
        n, batch = case["n"], case["batch"]
        flags = estl_amd.FLAG_NORMALIZE if case["normalize"] else 0
        s = {"kind": kind, "x": _complex(seed, batch, n), "n": n, "batch": batch}
        if kind == "fft":
            s["plan"] = estl_amd.Plan(n, batch, case["dir"], flags=flags)
            s["y"] = torch.empty_like(s["x"])
        else:
            s["plan"] = estl_amd.Plan(n, batch, case["dir"], precision=estl_amd.FP16, flags=flags)
            s["x16"] = torch.empty(batch, n, 2, dtype=torch.float16, device=DEVICE)
            s["y16"] = torch.empty_like(s["x16"])
            s["sx"] = torch.empty(batch, dtype=torch.float32, device=DEVICE)
            s["sy"] = torch.empty_like(s["sx"])
        return s
    if kind == "fft2d":
        x = _complex(seed, case["batch"], case["ny"], case["nx"])
        return {"kind": kind, "x": x, "y": torch.empty_like(x),
                "plan": estl_amd.Plan2D(case["nx"], case["ny"], case["batch"], case["dir"])}
    if kind == "uneven":
        b = _uneven_sizes(case)
        x = _complex(seed, b.total)
        return {"kind": kind, "x": x, "y": torch.empty_like(x),
                "plan": estl_amd.UnevenBatch(b.sizes.tolist(), b.offsets.tolist(), case["dir"])}
    if kind == "served":
        return {"kind": kind, "server": estl_amd.Server(4 << 30, streams=8), "requests": _served_inputs(case, seed)}
    n, rows = case["n"], case["rows"]
    x, h = _uniform(seed, rows, n), _taps(seed, case["k"], case["normalize"])
    s = {"kind": kind, "h": h, "new_filter": case["new_filter"]}
    if kind == "conv":
        s.update(conv=estl_amd.Convolution(n, rows, _conv_flags(case)), x=x, y=torch.empty_like(x))
    else:
        s["conv"] = estl_amd.Convolution(n, rows, _conv_flags(case), precision=estl_amd.FP16)
        s["x16"] = torch.empty(rows, n, dtype=torch.float16, device=DEVICE)
        s["y16"] = torch.empty_like(s["x16"])
        s["sx"] = torch.empty(rows, dtype=torch.float32, device=DEVICE)
        s["sy"] = torch.empty_like(s["sx"])
        estl_amd.pack_fp16(x, s["x16"], s["sx"], n // 2, rows)
    s["conv"].set_filter(h)
    return s


def run(state):
    kind = state["kind"]
    if kind in ("fft", "fft2d", "uneven"):
        state["plan"].execute(state["x"], state["y"])
        return state["y"]
    if kind == "fft16":
        estl_amd.pack_fp16(state["x"], state["x16"], state["sx"], state["n"], state["batch"])
        state["plan"].execute_fp16(state["x16"], state["sx"], state["y16"], state["sy"])
        return {"y16": state["y16"], "scale": state["sy"]}
    if kind == "served":
        srv = state["server"]
        ids = [srv.submit_conv(n, rows, x, h, flags=flags) for n, rows, flags, x, h in state["requests"]]
        out = []
        for rid, (n, rows, _, _, _) in zip(ids, state["requests"]):
            srv.wait(rid)
            out.append(srv.output(rid, (rows, n), torch.float32))
            srv.release(rid)
        return out
    if state["new_filter"]:
        state["conv"].set_filter(state["h"])
    if kind == "conv":
        state["conv"].execute(state["x"], state["y"])
        return state["y"]
    state["conv"].execute_fp16(state["x16"], state["sx"], state["y16"], state["sy"])
    return {"y16": state["y16"], "scale": state["sy"]}


# ---------------------------------------------------------------- work

def _fft_flops(n, count=1):
    return 5.0 * count * n * math.log2(n)


def _conv_work(n, rows, k, bytes_per_value, taps_bytes):
    """Rows in and out once and the taps once; two real transforms (each half a complex
    one) and a multiply, of whole rows or of the window length that costs least."""
    per_value = 5.0 * math.log2(n) + 3.0
    for log2l in range(int(math.log2(n))):
        length = 1 << log2l
        if length >= k:
            per_value = min(per_value, length / (length - k + 1) * (5.0 * log2l + 3.0))
    return {"bytes": rows * n * 2.0 * bytes_per_value + taps_bytes, "flops": rows * n * per_value}


def work(case):
    kind = case["kind"]
    if kind == "fft":
        v = case["n"] * case["batch"]
        return {"bytes": 16.0 * v, "flops": _fft_flops(case["n"], case["batch"])}
    if kind == "fft16":  # complex64 in, binary16 pairs out
        v = case["n"] * case["batch"]
        return {"bytes": 12.0 * v + 4.0 * case["batch"], "flops": _fft_flops(case["n"], case["batch"])}
    if kind == "fft2d":
        v = case["nx"] * case["ny"] * case["batch"]
        return {"bytes": 16.0 * v, "flops": 5.0 * v * math.log2(case["nx"] * case["ny"])}
    if kind == "uneven":
        sizes = _uneven_sizes(case).sizes
        return {"bytes": 16.0 * float(sizes.sum()), "flops": float(sum(_fft_flops(int(n)) for n in sizes))}
    if kind == "served":
        parts = [_conv_work(n, rows, k, 4.0, 4.0 * k) for n, rows, k, _ in _requests(case)]
        return {key: sum(p[key] for p in parts) for key in ("bytes", "flops")}
    taps = 4.0 * case["k"] if case["new_filter"] else 0.0
    return _conv_work(case["n"], case["rows"], case["k"], 4.0 if kind == "conv" else 2.0, taps)


# ---------------------------------------------------------------- 64-bit results

def _exact_fft(x, sign, normalize=False):
    """x: complex128 [..., n] on the CPU; unnormalised in both directions unless asked"""
    n = x.shape[-1]
    y = torch.fft.fft(x) if sign < 0 else torch.fft.ifft(x, norm="forward")
    return y / n if normalize else y


def _exact_conv(x, h, corr, center, normalize):
    """x: float64 [rows, n], h: float64 [k], on the CPU; circular in n"""
    n, k = x.shape[-1], h.numel()
    folded = torch.zeros(n, dtype=torch.float64).index_add_(0, torch.arange(k) % n, h)
    if center:
        folded = torch.roll(folded, -((k + 1) // 2))
    if normalize:
        folded = folded / h.sum()
    spec = torch.fft.rfft(folded)
    return torch.fft.irfft(torch.fft.rfft(x) * (spec.conj() if corr else spec), n)


def exact(case, seed):
    kind = case["kind"]
    if kind == "fft":
        x = _complex(seed, case["batch"], case["n"]).cpu().to(torch.complex128)
        return _exact_fft(x, case["dir"], case["normalize"])
    if kind == "fft16":
        n = case["n"]
        x = _complex(seed, case["batch"], n).cpu().to(torch.complex128)
        peak = torch.view_as_real(x).abs().amax(dim=(1, 2))
        scale = peak * (math.sqrt(n) / n if case["normalize"] else math.sqrt(n))
        y = _exact_fft(x, case["dir"], case["normalize"]) / scale[:, None]
        return {"y16": torch.view_as_real(y), "scale": scale}
    if kind == "fft2d":
        x = _complex(seed, case["batch"], case["ny"], case["nx"]).cpu().to(torch.complex128)
        return torch.fft.fft2(x) if case["dir"] < 0 else torch.fft.ifft2(x, norm="forward")
    if kind == "uneven":
        b = _uneven_sizes(case)
        x = _complex(seed, b.total).cpu()
        y = torch.empty(b.total, dtype=torch.complex128)
        sizes, offsets = torch.from_numpy(b.sizes), torch.from_numpy(b.offsets)
        for n in sorted(set(b.sizes.tolist())):
            at = offsets[sizes == n].tolist()
            rows = _exact_fft(torch.stack([x[o:o + n] for o in at]).to(torch.complex128), case["dir"])
            for o, r in zip(at, rows):
                y[o:o + n] = r
        return y
    if kind == "served":
        corr = estl_amd.CONV_CORRELATE
        return [_exact_conv(x.cpu().double().view(rows, n), h.cpu().double(), bool(flags & corr), False, False)
                for n, rows, flags, x, h in _served_inputs(case, seed)]
    h = _taps(seed, case["k"], case["normalize"]).cpu().double()
    x = _uniform(seed, case["rows"], case["n"]).cpu().double()
    y = _exact_conv(x, h, case["corr"], case["center"], case["normalize"])
    if kind == "conv":
        return y
    gain = h.abs().sum() / (h.sum().abs() if case["normalize"] else 1.0)
    scale = x.abs().amax(dim=1) * gain
    return {"y16": y / scale[:, None], "scale": scale}
