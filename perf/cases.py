"""The calls whose speed matters, as a program that uses this package makes them.

A case is a dict of plain values. `listed()` holds the ones that are always measured, `draw(rng)`
gives another of the same ranges, `prepare(case, seed)` builds what a program has in hand before
the call (inputs on the GPU, a plan, an operator, a running server), `run(state)` makes one pass
through the public entry points and returns its outputs, `work(case)` says what a pass cannot do
without, and `exact(case, seed)` gives the same outputs in 64 bits.

Kinds of case:
  fft1d  Plan((n,), batch).exec: batched 1D transforms, powers of two from 2^8 to 2^20 and lengths
         with factors 3, 5 and 17; natural or digit-reversed input; every precision
  fft2d  Plan((nx, ny), batch).exec: batched 2D transforms, sides 64 to 2176
  conv   Conv2d.forward with resident filters: one channel, image sides 64 to 2048, filters 3 to 63
  layer  one training step of a convolution layer: new filters in, forward, both gradients
  queue  the work-queue batcher: uneven lengths and counts in one launch
  serve  a burst of mixed 1D and 2D requests on a running server
"""
import ctypes
import math
import random

import torch

import fft_demo_amd as F
from fft_demo_amd import _lib as L
from fft_demo_amd.conv import Conv2d, good_size
from fft_demo_amd.plan import Plan
from fft_demo_amd.serve import KIND_1D, KIND_2D, Server

DTYPE = {"split_fp16": torch.float16, "fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
CONV_OPTIONS = {"default": {}, "mid_fp16": {"mid_fp16": True}, "spec_fp16": {"spec_fp16": True}}
ODD_PARTS = (3, 5, 9, 15, 17)


def _smooth(n):
    for p in (2, 3, 5, 17):
        while n % p == 0:
            n //= p
    return n == 1


SMOOTH = [n for n in range(48, 4097) if n & (n - 1) and _smooth(n)]


def listed():
    return [
        # a single short signal block per call: latency
        {"name": "fft1d_1024x4", "op": "fft1d", "n": 1024, "batch": 4, "precision": "split_fp16", "mid": "",
         "inverse": False, "reversed": False},
        # the plain batched configuration, 256 points x 4096
        {"name": "fft1d_256x4096", "op": "fft1d", "n": 256, "batch": 4096, "precision": "split_fp16", "mid": "",
         "inverse": False, "reversed": False},
        # a block of medium lines back to the time domain, bf16
        {"name": "fft1d_16384x96_bf16_inv", "op": "fft1d", "n": 16384, "batch": 96, "precision": "bf16", "mid": "",
         "inverse": True, "reversed": False},
        # the headline configuration, 65536 points x 256, 16-bit words between the passes
        {"name": "fft1d_65536x256", "op": "fft1d", "n": 65536, "batch": 256, "precision": "split_fp16", "mid": "c16",
         "inverse": False, "reversed": False},
        # the longest 1D requests of the serving mix, the inverse direction
        {"name": "fft1d_2p20x16_inv", "op": "fft1d", "n": 1 << 20, "batch": 16, "precision": "split_fp16",
         "mid": "c16", "inverse": True, "reversed": False},
        # a mixed-radix length (16 * 3 * 5 * 5) and a ragged batch: frames of audio or radar data
        {"name": "fft1d_1200x3001", "op": "fft1d", "n": 1200, "batch": 3001, "precision": "split_fp16", "mid": "",
         "inverse": False, "reversed": False},
        # the 2D configuration, 1024 x 1024 x 64, 10% of the entries x 100
        {"name": "fft2d_1024x64", "op": "fft2d", "nx": 1024, "ny": 1024, "batch": 64, "precision": "split_fp16",
         "mid": "c16", "inverse": False},
        # video frames (480 = 15 * 32, 640 = 5 * 128) in plain fp32, inverse
        {"name": "fft2d_480x640x18_fp32_inv", "op": "fft2d", "nx": 480, "ny": 640, "batch": 18, "precision": "fp32",
         "mid": "", "inverse": True},
        # the convolution configuration: 2048 x 2048 images x 16, a 31 x 31 filter, padded to 2176
        {"name": "conv_2048x16_f31", "op": "conv", "h": 2048, "w": 2048, "batch": 16, "fsize": 31, "pad": 2176,
         "option": "mid_fp16"},
        # one training step of the reference's accuracy shape as a layer: 256 x 256, 16 filters of 13 x 13
        {"name": "layer_256_c3_f16_k13", "op": "layer", "h": 256, "w": 256, "batch": 8, "channels": 3, "filters": 16,
         "fsize": 13},
        # uneven transforms that arrived together, one launch
        {"name": "queue_48", "op": "queue", "items": 48, "mix": 7, "precision": "split_fp16"},
        # a burst of the serving mix's 1D and 2D requests
        {"name": "serve_32", "op": "serve", "requests": 32, "mix": 11},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _side(rng, hi):
    while True:
        s = rng.choice((1,) * 5 + ODD_PARTS) << rng.randint(4, 11)
        if 64 <= s <= hi:
            return s


def draw(rng):
    op = rng.choice(("fft1d", "fft1d", "fft1d", "fft2d", "fft2d", "conv", "layer", "queue", "serve"))
    precision = rng.choice(("split_fp16", "split_fp16", "split_fp16", "fp16", "bf16", "fp32"))
    mid = rng.choice(("", "c16")) if precision == "split_fp16" else ""
    if op == "fft1d":
        rev = precision in ("split_fp16", "fp16") and rng.random() < 0.2
        kind = rng.random()
        if rev:
            n = 1 << rng.choice((8, 9, 10, 11, 12, 16, 17, 18, 19))
        elif kind < 0.55:
            n = 1 << rng.randint(8, 20)
        elif kind < 0.8:
            n = rng.choice(SMOOTH)
        else:
            n = rng.choice(ODD_PARTS) << rng.randint(5, 12)
        return {"op": op, "n": n, "batch": _log(rng, 1, max(1, min(8192, (1 << 25) // n))), "precision": precision,
                "mid": mid, "inverse": rng.random() < 0.4, "reversed": rev}
    if op == "fft2d":
        nx, ny = _side(rng, 2176), _side(rng, 2176)
        return {"op": op, "nx": nx, "ny": ny, "batch": _log(rng, 1, max(1, min(64, (1 << 25) // (nx * ny)))),
                "precision": precision, "mid": mid, "inverse": rng.random() < 0.4}
    if op == "conv":
        h, w = _log(rng, 64, 2048), _log(rng, 64, 2048)
        return {"op": op, "h": h, "w": w, "batch": rng.randint(1, 16), "fsize": 2 * rng.randint(1, 31) + 1, "pad": 0,
                "option": rng.choice(("default", "mid_fp16", "spec_fp16"))}
    if op == "layer":
        return {"op": op, "h": _log(rng, 32, 300), "w": _log(rng, 32, 300), "batch": rng.randint(1, 8),
                "channels": rng.randint(1, 8), "filters": rng.randint(1, 16), "fsize": rng.randint(2, 13)}
    if op == "queue":
        return {"op": op, "items": rng.randint(2, 60), "mix": rng.randint(0, 10 ** 6),
                "precision": rng.choice(("split_fp16", "fp16", "bf16", "fp32"))}
    return {"op": op, "requests": rng.randint(4, 32), "mix": rng.randint(0, 10 ** 6)}


# ---------------------------------------------------------------- shapes of the composite cases
def _queue_items(case):
    """(length, count) of each item: powers of two 2^4..2^12, some mixed-radix lengths."""
    rng = random.Random(case["mix"])
    out = []
    for _ in range(case["items"]):
        n = 1 << rng.randint(4, 12) if rng.random() < 0.75 else rng.choice(SMOOTH)
        out.append((n, _log(rng, 1, max(1, min(256, (1 << 16) // n)))))
    return out


def _requests(case):
    """(nx, ny, batch) of each request, ny = 0 for 1D: the serving mix's shapes, at most 2^22 points each."""
    rng = random.Random(case["mix"])
    out = []
    for _ in range(case["requests"]):
        if rng.random() < 60 / 85:
            n = 1 << rng.randint(8, 20)
            out.append((n, 0, min(rng.randint(1, 64), (1 << 22) // n)))
        else:
            s = rng.choice((256, 512, 1024, 2048))
            out.append((s, s, max(1, min(rng.randint(1, 16), (1 << 22) // (s * s)))))
    return out


# ---------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _uniform(shape, dtype, g, lo=-1.0, hi=1.0):
    return (torch.rand(shape, generator=g, device="cuda", dtype=torch.float32) * (hi - lo) + lo).to(dtype)


def _signal(shape, dtype, g):
    """Interleaved complex, real and imaginary parts uniform in [-1, 1]."""
    return _uniform((*shape, 2), dtype, g)


def _fft2d_input(case, seed):
    """Uniform entries, 10% of them x 100 (the dynamic-range stress of the 2D configuration)."""
    g = _gen(seed)
    shape = (case["batch"], case["nx"], case["ny"])
    x = _signal(shape, torch.float32, g)
    x *= torch.where(torch.rand(shape, generator=g, device="cuda") < 0.1, 100.0, 1.0).unsqueeze(-1)
    if case["precision"] != "split_fp16":
        x *= 2.0 ** -6  # unscaled 16-bit transforms: the largest outputs stay below 65504
    return x.to(DTYPE[case["precision"]])


def _fft1d_input(case, seed):
    return _signal((case["batch"], case["n"]), DTYPE[case["precision"]], _gen(seed))


def _conv_inputs(case, seed):
    g = _gen(seed)
    k = case["fsize"]
    x = _uniform((case["batch"], 1, case["h"], case["w"]), torch.float32, g, 0.0, 1.0)
    r = torch.arange(k, device="cuda", dtype=torch.float64) - (k - 1) / 2
    w = torch.exp(-(r[:, None] ** 2 + r[None, :] ** 2) / 50.0)
    w = (w / w.sum()).float() * (1 + _uniform((k, k), torch.float32, g, -0.01, 0.01))
    return x, w.reshape(1, 1, k, k).contiguous()


def _layer_inputs(case, seed):
    g = _gen(seed)
    k, c, f = case["fsize"], case["channels"], case["filters"]
    x = _uniform((case["batch"], c, case["h"], case["w"]), torch.float32, g, 0.0, 1.0)
    w = torch.randn((f, c, k, k), generator=g, device="cuda") / math.sqrt(c * k * k)
    d = torch.randn((case["batch"], f, case["h"] - k + 1, case["w"] - k + 1), generator=g, device="cuda")
    return x, w, d


def _queue_inputs(case, seed):
    g = _gen(seed)
    return [_signal((c, n), DTYPE[case["precision"]], g) for n, c in _queue_items(case)]


def _serve_inputs(case, seed):
    g = _gen(seed)
    return [_signal((b, nx, ny) if ny else (b, nx), torch.float16, g) for nx, ny, b in _requests(case)]


# ---------------------------------------------------------------- states
class _Batcher:
    def __init__(self, case, xs):
        lib = L.load()
        desc = F.make_desc(precision=case["precision"])
        self.handle = ctypes.c_void_p()
        L.check(lib.mfft_batcher_create(ctypes.byref(self.handle), ctypes.byref(desc), len(xs)), "batcher")
        self.xs, self.outs = xs, [torch.empty_like(x) for x in xs]
        self.items = (L.BatchItem * len(xs))()
        for it, x, y in zip(self.items, self.xs, self.outs):
            it.in_, it.out, it.n, it.count = x.data_ptr(), y.data_ptr(), x.shape[1], x.shape[0]

    def run(self):
        s = torch.cuda.current_stream()
        L.check(L.load().mfft_batcher_exec(self.handle, self.items, len(self.xs), ctypes.c_void_p(s.cuda_stream)),
                "mfft_batcher_exec")
        return self.outs

    def __del__(self):
        torch.cuda.synchronize()
        L.load().mfft_batcher_destroy(self.handle)


class _Serving:
    def __init__(self, case, xs):
        self.xs, self.outs = xs, [torch.empty_like(x) for x in xs]
        self.server = Server(precision="split", mid_fmt="c16")
        self.reqs = []
        for i, ((nx, ny, b), x, y) in enumerate(zip(_requests(case), xs, self.outs)):
            shape = {"nx": nx, "ny": ny} if ny else {"n": nx}
            self.reqs.append(((KIND_2D if ny else KIND_1D, x.data_ptr(), y.data_ptr(), i), dict(batch=b, **shape)))
        torch.cuda.synchronize()  # the server reads the inputs on streams of its own

    def run(self):
        for args, kw in self.reqs:
            self.server.submit(*args, **kw)
        self.server.wait_idle()
        for c in self.server.poll():
            if c.status != 0:
                raise RuntimeError("request %d: status %d" % (c.tag, c.status))
        return self.outs

    def __del__(self):
        self.server.close()


class _Fft:
    def __init__(self, case, shape, x, in_order=F.ORDER_NATURAL):
        self.plan = Plan(shape, case["batch"], precision=case["precision"],
                         direction=F.INVERSE if case["inverse"] else F.FORWARD, in_order=in_order,
                         mid_fmt=case["mid"] or None)
        if in_order == F.ORDER_DIGIT_REVERSED:
            x = x[:, torch.from_numpy(self.plan.input_permutation()).long().to(x.device)]
        self.x = x.contiguous()
        self.out = self.plan.empty_out()

    def run(self):
        return self.plan.exec(self.x, out=self.out)


class _Conv:
    def __init__(self, case, x, w):
        k = case["fsize"]
        self.op = Conv2d(case["batch"], 1, 1, case["h"], case["w"], k, k, mode="same", pad=case["pad"] or None,
                         **CONV_OPTIONS[case["option"]])
        self.op.set_filters(w)
        self.x, self.w = x, w
        self.out = torch.empty(self.op.out_shape, dtype=torch.float32, device="cuda")

    def run(self):
        return self.op.forward(self.x, out=self.out)


class _Layer:
    def __init__(self, case, x, w, d):
        k = case["fsize"]
        self.op = Conv2d(case["batch"], case["channels"], case["filters"], case["h"], case["w"], k, k,
                         mode="valid_corr")
        self.x, self.w, self.d = x, w, d

    def run(self):
        self.op.set_filters(self.w)
        out = self.op.forward(self.x)
        grad_in, grad_w = self.op.backward(self.d, self.x)
        return {"out": out, "grad_in": grad_in, "grad_w": grad_w}


def prepare(case, seed):
    op = case["op"]
    if op == "fft1d":
        return _Fft(case, (case["n"],), _fft1d_input(case, seed),
                    F.ORDER_DIGIT_REVERSED if case["reversed"] else F.ORDER_NATURAL)
    if op == "fft2d":
        return _Fft(case, (case["nx"], case["ny"]), _fft2d_input(case, seed))
    if op == "conv":
        return _Conv(case, *_conv_inputs(case, seed))
    if op == "layer":
        return _Layer(case, *_layer_inputs(case, seed))
    if op == "queue":
        return _Batcher(case, _queue_inputs(case, seed))
    return _Serving(case, _serve_inputs(case, seed))


def run(state):
    return state.run()


# ---------------------------------------------------------------- work and exact results
def _fft_work(points, n, elem):
    return {"bytes": 2 * points * elem, "flops": 5 * points * math.log2(n)}


def work(case):
    op = case["op"]
    if op == "fft1d":
        return _fft_work(case["n"] * case["batch"], case["n"], 8 if case["precision"] == "fp32" else 4)
    if op == "fft2d":
        p = case["nx"] * case["ny"]
        return _fft_work(p * case["batch"], p, 8 if case["precision"] == "fp32" else 4)
    if op == "conv":
        # two images share a transform of P points each way; the filter's spectrum is resident
        b, h, w, k = case["batch"], case["h"], case["w"], case["fsize"]
        p = case["pad"] ** 2 if case["pad"] else good_size(h + k - 1) * good_size(w + k - 1)
        pairs = (b + 1) // 2
        return {"bytes": 2 * b * h * w * 4 + p * 8, "flops": pairs * (10 * p * math.log2(p) + 8 * p)}
    if op == "layer":
        # transforms: images, filters, delta forward; outputs, both gradients inverse
        b, c, f, h, w, k = (case[x] for x in ("batch", "channels", "filters", "h", "w", "fsize"))
        p, pairs = good_size(h) * good_size(w), (b + 1) // 2
        o = (h - k + 1) * (w - k + 1)
        return {"bytes": 4 * (2 * b * c * h * w + 2 * b * f * o + 2 * f * c * k * k),
                "flops": (2 * pairs * c + 2 * f * c + 2 * pairs * f) * 5 * p * math.log2(p) + 3 * 8 * p * pairs * c * f}
    parts = []
    if op == "queue":
        elem = 8 if case["precision"] == "fp32" else 4
        parts = [_fft_work(n * c, n, elem) for n, c in _queue_items(case)]
    else:
        parts = [_fft_work(nx * max(1, ny) * b, nx * max(1, ny), 4) for nx, ny, b in _requests(case)]
    return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}


def _dft(x, dims, inverse, scaled):
    """Interleaved result of the unnormalised transform, times 1/n when scaled."""
    z = torch.view_as_complex(x.double())
    y = torch.fft.ifftn(z, dim=dims, norm="forward") if inverse else torch.fft.fftn(z, dim=dims)
    if scaled:
        y = y / math.prod(z.shape[d] for d in dims)
    return torch.view_as_real(y)


def exact(case, seed):
    op = case["op"]
    if op in ("fft1d", "fft2d"):
        x, dims = (_fft1d_input(case, seed), (1,)) if op == "fft1d" else (_fft2d_input(case, seed), (1, 2))
        return _dft(x, dims, case["inverse"], case["precision"] == "split_fp16")
    if op == "queue":
        return [_dft(x, (1,), False, case["precision"] == "split_fp16") for x in _queue_inputs(case, seed)]
    if op == "serve":
        return [_dft(x, tuple(range(1, x.dim() - 1)), False, True) for x in _serve_inputs(case, seed)]
    k = case["fsize"]
    s = (case["h"] + k - 1, case["w"] + k - 1)
    if op == "conv":
        x, w = (t.double() for t in _conv_inputs(case, seed))
        o = (k - 1) // 2
        full = torch.fft.irfft2(torch.fft.rfft2(x, s) * torch.fft.rfft2(w, s), s)
        return full[..., o:o + case["h"], o:o + case["w"]].contiguous()
    x, w, d = (t.double() for t in _layer_inputs(case, seed))
    X, W, D = (torch.fft.rfft2(t, s) for t in (x, w, d))
    out = torch.stack([(X * W[f].conj()).sum(1) for f in range(case["filters"])], 1)
    gin = torch.stack([(D * W[:, c]).sum(1) for c in range(case["channels"])], 1)
    gw = torch.stack([(X * D[:, f:f + 1].conj()).sum(0) for f in range(case["filters"])])
    out, gin, gw = (torch.fft.irfft2(t, s) for t in (out, gin, gw))
    return {"out": out[..., :d.shape[2], :d.shape[3]].contiguous(),
            "grad_in": gin[..., :case["h"], :case["w"]].contiguous(), "grad_w": gw[..., :k, :k].contiguous()}
