"""Performance cases: optimizer steps as a training program takes them.

Each case is one ``optimizer.step()`` of one of the library's optimizers over a
set of params whose gradients and state are resident on the GPU, in the middle
of a training run (the second moment and the momentum are those of a run with
gradients of the same size).  ``listed()`` holds the cases that are measured,
``draw()`` gives others of the same ranges, ``prepare()`` builds a case's
params, gradients, state and optimizer, ``run()`` takes the step and returns
everything it wrote, and ``exact()`` computes the same step in 64 bits.

Param sets (``case["set"]``):
  bag       ``count`` matrices of ``rows`` x ``cols``: adapters of one small layer
  adapters  a rank-``rank`` pair [rank, in], [out, rank] for each linear of the
            UNet-shaped set (``share`` of them)
  unet      the SDXL-UNet-shaped set: ``share`` of each shape's count, the dims
            scaled by ``width`` / 320
  dense     a transformer: ``layers`` blocks of width ``dim`` with an inner width
            ``inner``, an embedding of ``vocab`` rows, biases and norms
All tensors of one role live in one buffer, each at a 512-byte boundary (where
the caching allocator would put it), so a step's whole output is a few tensors.
"""
from __future__ import annotations

import math
import os
import sys

import torch

# imported with the repository's root as the working folder
sys.path.insert(0, os.path.abspath("k-optimizers_amd"))

DEV = "cuda:0"
_DT = {"bf16": torch.bfloat16, "fp32": torch.float32}
_MOM = {"bf16": "bfloat16", "fp32": "float32", "int8": "int8", "4bit": "4bit"}

# the SDXL-UNet-shaped set: (shape, count); 1,678 tensors, 2.664 G params
_UNET = [
    ((1280, 1280), 368), ((1280, 2048), 130), ((5120, 1280), 120), ((1280, 5120), 60),
    ((5120, 640), 20), ((2048, 640), 20), ((1280, 640), 40),
    ((1280, 1280, 3, 3), 22), ((640, 640, 3, 3), 10), ((320, 320, 3, 3), 8), ((1280, 640, 3, 3), 2),
    ((640, 1280, 3, 3), 3), ((640, 320, 3, 3), 2), ((320, 640, 3, 3), 3),
    ((1280,), 580), ((5120,), 140), ((640,), 120), ((320,), 30),
]


def listed() -> list[dict]:
    return [
        # adapter training of a small layer set in fp32: a launch-bound step
        dict(name="adakaon_bag_fp32", opt="adakaon", set="bag", count=512, rows=8, cols=16, dtype="fp32", mom="bf16",
             method="sr", fused=True),
        # LoRA training of a diffusion UNet's linears, bf16 adapters: 1,516 thin matrices
        dict(name="adakaon_adapters_int8", opt="adakaon", set="adapters", rank=16, share=1.0, dtype="bf16",
             mom="int8", method="sr", fused=False),
        # full fine-tune of the UNet, the library's headline configuration
        dict(name="adakaon_unet_int8", opt="adakaon", set="unet", width=320, share=1.0, dtype="bf16", mom="int8",
             method="sr", fused=True),
        # the same with Lion, which leaves the gradient centralized
        dict(name="lion_unet_int8", opt="lion", set="unet", width=320, share=1.0, dtype="bf16", mom="int8",
             method="sr"),
        # lookahead training in little memory: 4-bit momentum, removal and climb of the lookahead, weight decay
        dict(name="nekaon_unet_4bit", opt="nekaon", set="unet", width=320, share=0.25, dtype="bf16", mom="4bit",
             block=64, method="sr", wd=0.1, fused=True),
        # orthogonalized updates: two Newton-Schulz iterations per matrix
        dict(name="adamuon_unet_int8", opt="adamuon", set="unet", width=320, share=0.25, dtype="bf16", mom="int8",
             method="sr"),
        # the positive-negative momentum pair at its default bf16 storage
        dict(name="adapnm_unet_bf16", opt="adapnm", set="unet", width=320, share=0.25, dtype="bf16", mom="bf16",
             method="sr", fused=False),
        # learning-rate-free training at its defaults: fp32 second moment and distance statistics
        dict(name="kprodigy_unet_bf16", opt="kprodigy", set="unet", width=320, share=0.25, dtype="bf16", mom="bf16",
             method="sr"),
        # sharpness-aware climb with a norm over the whole net
        dict(name="msam_unet_int8", opt="msam", set="unet", width=320, share=0.25, dtype="bf16", mom="int8",
             method="sr", fused=True),
        # a transformer trained in full fp32 (params and gradients), its vocabulary an odd number
        dict(name="adakaon_dense_fp32", opt="adakaon", set="dense", layers=12, dim=768, inner=3072, vocab=50257,
             dtype="fp32", mom="bf16", method="sr", fused=False),
        # the same net in bf16 with compensated (kahan) writes and weight decay
        dict(name="adakaon_dense_kahan", opt="adakaon", set="dense", layers=12, dim=768, inner=3072, vocab=50257,
             dtype="bf16", mom="bf16", method="kahan", wd=0.01, fused=False),
        # dims that are no multiple of a vector: rows that start at any alignment
        dict(name="adakaon_odd_int8", opt="adakaon", set="dense", layers=8, dim=771, inner=2057, vocab=10007,
             dtype="bf16", mom="int8", method="sr", fused=False),
    ]


def _log(rng, lo: float, hi: float) -> float:
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng) -> dict:
    kind = rng.choice(["bag", "adapters", "unet", "unet", "unet", "dense", "dense", "dense"])
    c: dict = dict(set=kind, method="sr", dtype="bf16")
    if kind == "bag":
        c.update(opt=rng.choice(["adakaon", "lion"]), dtype=rng.choice(["fp32", "bf16"]),
                 mom=rng.choice(["bf16", "int8"]), count=int(_log(rng, 16, 2048)), rows=int(_log(rng, 4, 65)),
                 cols=int(_log(rng, 8, 257)))
    elif kind == "adapters":
        c.update(opt=rng.choice(["adakaon", "lion", "adapnm"]), dtype=rng.choice(["bf16", "bf16", "fp32"]),
                 mom=rng.choice(["bf16", "int8"]), rank=int(_log(rng, 4, 129)),
                 share=round(_log(rng, 0.02, 1.0), 4))
    elif kind == "unet":
        c.update(opt=rng.choice(["adakaon", "lion", "nekaon", "adamuon", "adapnm", "kprodigy", "msam"]),
                 width=rng.choice([rng.randint(32, 320), 8 * rng.randint(4, 40), 320]),
                 share=round(_log(rng, 0.01, 0.25), 4))
        c["mom"] = rng.choice(["bf16", "int8"] if c["opt"] == "kprodigy" else ["bf16", "int8", "4bit"])
    else:
        c.update(opt=rng.choice(["adakaon", "adakaon", "lion", "adapnm", "kprodigy"]),
                 dtype=rng.choice(["fp32", "bf16"]), method=rng.choice(["sr", "kahan", "rn"]),
                 mom=rng.choice(["bf16", "int8", "fp32"]), layers=rng.randint(2, 12),
                 dim=int(_log(rng, 128, 1281)), vocab=int(_log(rng, 1000, 50258)))
        if rng.random() < 0.5:
            c["dim"] = max(128, c["dim"] // 64 * 64)
        c["inner"] = int(c["dim"] * rng.choice([4, 2.667, 3.5]))
    if c["mom"] == "4bit":
        c["block"] = rng.choice([64, 128, 256])
    if c["opt"] in ("adakaon", "lion", "nekaon", "adapnm") and rng.random() < 0.5:
        c["wd"] = 0.01
    if c["opt"] in ("adakaon", "adapnm", "nekaon", "msam"):
        c["fused"] = rng.random() < 0.5
    return c


# ------------------------------------------------------------------ shapes
def _shapes(case: dict) -> list[tuple[int, ...]]:
    if case["set"] == "bag":
        return [(case["rows"], case["cols"])] * case["count"]
    if case["set"] == "dense":
        d, f = case["dim"], case["inner"]
        out: list[tuple[int, ...]] = [(case["vocab"], d)]
        for _ in range(case["layers"]):
            out += [(3 * d, d), (3 * d,), (d, d), (d,), (f, d), (f,), (d, f), (d,), (d,), (d,)]
        return out
    out = []
    for shape, count in _UNET:
        n = max(1, round(count * case["share"]))
        if case["set"] == "adapters":
            if len(shape) == 2:
                out += [(case["rank"], shape[1]), (shape[0], case["rank"])] * n
        else:
            s = case["width"] / 320
            out += [tuple(x if x == 3 else max(1, round(x * s)) for x in shape)] * n
    return out


def _rc(shape: tuple[int, ...]) -> tuple[int, int]:
    n = math.prod(shape)
    return (shape[0], n // shape[0]) if len(shape) > 1 else (1, n)


class _Flat:
    """One buffer holding a view per tensor, each at a 512-byte boundary."""

    def __init__(self, sizes: list[int], dtype: torch.dtype) -> None:
        self.step = 512 // torch.empty(0, dtype=dtype).element_size()
        self.sizes, self.at, n = sizes, [], 0
        for s in sizes:
            self.at.append(n)
            n += -(-s // self.step) * self.step
        self.buf = torch.zeros(max(n, 1), dtype=dtype, device=DEV)

    def view(self, i: int, shape: tuple[int, ...]) -> torch.Tensor:
        return self.buf[self.at[i]:self.at[i] + self.sizes[i]].view(shape)

    def like(self, dtype: torch.dtype) -> "_Flat":
        """The same layout in another type (64-bit results beside the step's own)."""
        f = object.__new__(_Flat)
        f.step, f.sizes, f.at = self.step, self.sizes, self.at
        f.buf = torch.zeros(self.buf.numel(), dtype=dtype, device=DEV)
        return f


# ------------------------------------------------------------ hyper-parameters
def _hyper(case: dict) -> dict:
    """Constructor keywords of the case's optimizer."""
    opt = case["opt"]
    kw = {"adakaon": dict(lr=1e-4, betas=(0.9, 0.999)), "lion": dict(lr=2e-4, betas=(0.95, 0.98)),
          "nekaon": dict(lr=1e-4, betas=(0.2, 0.999), k=1.5), "adamuon": dict(lr=2e-2, betas=(0.95, 0.999), ns_steps=2),
          "adapnm": dict(lr=1e-4, betas=(0.8, 0.999)), "kprodigy": dict(lr=1.0, betas=(0.9, 0.999)),
          "msam": dict(lr=1e-4, betas=(0.9, 0.999), rho=0.3, norm="global")}[opt]
    kw.update(momentum_dtype=_MOM[case["mom"]], weight_decay=case.get("wd", 0.0),
              bf16_method={"sr": "stochastic_rounding", "kahan": "kahan", "rn": "none"}[case["method"]])
    if case["mom"] == "4bit":
        kw["momentum_4bit_block"] = case["block"]
    if "fused" in case:
        kw["fused"] = case["fused"]
    return kw


# KProdigy in the middle of a run: its distance estimate and initial estimate
_D, _D0 = 2e-5, 1e-6
# AdaPNM: steps taken before this one
_PNM_STEP = 20


def _codec_sizes(case: dict, n: int, R: int, dims: int) -> tuple[int, int, int]:
    """(stored momentum values, scales, 4-bit block) of a tensor of n values."""
    if case["mom"] == "int8":
        return n, (R if dims > 1 else 1), 0
    if case["mom"] == "4bit":
        b = min(case["block"], n)
        return (n + 1) // 2, -(-n // b), b
    return n, 0, 0


_MOM_DT = {"bf16": torch.bfloat16, "fp32": torch.float32, "int8": torch.int8, "4bit": torch.uint8}


@torch.no_grad()
def _build(case: dict, seed: int) -> dict:
    """Params, gradients and mid-run state of a case, from the seed alone."""
    shapes = _shapes(case)
    rc = [_rc(s) for s in shapes]
    ns = [r * c for r, c in rc]
    opt, kw = case["opt"], _hyper(case)
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    # one gradient size per tensor, log-uniform over three decades
    sig = (10.0 ** (torch.rand(len(shapes), generator=gen, device=DEV, dtype=torch.float64) * 3 - 5)).tolist()
    dt = _DT[case["dtype"]]
    pn = opt == "adapnm"
    pd = opt == "kprodigy"
    cs = [_codec_sizes(case, n, r, len(s)) for n, (r, _), s in zip(ns, rc, shapes)]
    f = {"p": _Flat(ns, dt), "g": _Flat(ns, dt)}
    for key in ("m_pos", "m_neg") if pn else ("m",):
        f[key] = _Flat([c[0] for c in cs], _MOM_DT[case["mom"]])
        if case["mom"] in ("int8", "4bit"):
            f[key + "_scale"] = _Flat([c[1] for c in cs], torch.float32)
    if opt != "lion":
        if not pd:
            f["row"] = _Flat([r if len(s) > 1 else 0 for (r, _), s in zip(rc, shapes)], torch.float32)
            f["col"] = _Flat([c if len(s) > 1 else 0 for (_, c), s in zip(rc, shapes)], torch.float32)
        f["v"] = _Flat([n if pd or len(s) < 2 else 0 for n, s in zip(ns, shapes)], torch.float32)
    if pd:
        f["s"], f["p0"] = _Flat(ns, torch.float32), _Flat(ns, torch.float32)
    if case["method"] == "kahan" and dt == torch.bfloat16:
        f["shift"] = _Flat(ns, dt)

    b1 = kw["betas"][0]
    ema = math.sqrt((1 - b1) / (1 + b1))
    alpha_s = _D / _D0 * _D  # KProdigy's weight of a gradient in s (lr 1)
    states, den = [], 0.0
    for i, (shape, (R, C), n) in enumerate(zip(shapes, rc, ns)):
        sg = sig[i]
        f["p"].view(i, shape).normal_(0.0, 0.02, generator=gen)
        f["g"].view(i, shape).normal_(0.0, sg, generator=gen)
        st: dict = {}
        # the momentum holds updates of about lr (Adakaon's family) or gradients (the rest)
        std = ema * (kw["lr"] if opt in ("adakaon", "nekaon", "msam") else sg * (_D if pd else 1.0))
        if opt == "adamuon" and len(shape) < 2:
            std = ema * 0.2 * kw["lr"]
        for key in ("m_pos", "m_neg") if pn else ("m",):
            numel, nsc, block = cs[i]
            m = f[key].view(i, (numel,) if case["mom"] == "4bit" else shape)
            if case["mom"] in ("bf16", "fp32"):
                m.normal_(0.0, std, generator=gen)
            else:
                top, wide = (127.0, 4.2) if case["mom"] == "int8" else (7.0, 2.7)
                q = torch.empty(n + n % 2, device=DEV).normal_(0.0, top / wide, generator=gen)
                q.round_().clamp_(-top, top)
                if case["mom"] == "int8":
                    m.copy_(q[:n].view(shape))
                else:
                    q = (q + 8.0).to(torch.uint8)
                    m.copy_(q[0::2] | (q[1::2] << 4))
                sc = f[key + "_scale"].view(i, (nsc,))
                sc.uniform_(0.8 * std * wide / top, 1.2 * std * wide / top, generator=gen)
                if case["mom"] == "int8":
                    sc = sc.view((R,) + (1,) * (len(shape) - 1) if len(shape) > 1 else ())
                else:
                    st[key + "_numel"], st[key + "_block"] = n, block
                st[key + "_scale"] = sc
            st[key] = m
        q = sg * sg + (1e-8 if pn else 0.0)
        if opt == "adamuon" and len(shape) > 1:
            q = 1.0 / max(R, C)  # the orthogonal factor's mean square
        if "row" in f and len(shape) > 1:
            st["row"] = f["row"].view(i, (R,)).uniform_(0.9 * q, 1.1 * q, generator=gen)
            st["col"] = f["col"].view(i, (C,)).uniform_(0.9 * q, 1.1 * q, generator=gen)
        elif opt != "lion":
            q *= _D * _D if pd else 1.0
            st["v"] = f["v"].view(i, shape).uniform_(0.5 * q, 1.5 * q, generator=gen)
        if pd:
            st["step"] = 100
            wide = alpha_s * sg * 22.0
            st["s"] = f["s"].view(i, (n,)).normal_(0.0, wide, generator=gen)
            st["p0"] = f["p0"].view(i, (n,))
            st["p0"].normal_(0.0, 1e-3, generator=gen).add_(f["p"].view(i, (n,)).float())
            den += n * 0.8 * wide
        if "shift" in f:
            st["shift"] = f["shift"].view(i, shape).normal_(0.0, 2e-5, generator=gen)
        states.append(st)
    return dict(shapes=shapes, rc=rc, f=f, states=states, den=den)


def prepare(case: dict, seed: int) -> dict:
    import kaon_amd

    b = _build(case, seed)
    cls = {"adakaon": kaon_amd.Adakaon, "lion": kaon_amd.Lion, "nekaon": kaon_amd.Nekaon, "adamuon": kaon_amd.AdaMuon,
           "adapnm": kaon_amd.AdaPNM, "kprodigy": kaon_amd.KProdigy, "msam": kaon_amd.MSAM}[case["opt"]]
    params = []
    for i, shape in enumerate(b["shapes"]):
        p = torch.nn.Parameter(b["f"]["p"].view(i, shape))
        p.grad = b["f"]["g"].view(i, shape)
        params.append(p)
    opt = cls(params, **_hyper(case))
    inner = getattr(opt, "inner", opt)
    inner.sr_seed = seed & 0x7FFFFFFF
    for p, st in zip(params, b["states"]):
        inner.state[p] = st
    if case["opt"] == "kprodigy":
        opt.param_groups[0].update(d=_D, d0=_D0, d_max=_D, k=100, d_numerator=_D * b["den"])
    if case["opt"] == "adapnm":
        opt.param_groups[0]["step"] = _PNM_STEP
    out = {k: v.buf for k, v in b["f"].items() if k != "p0" and v.buf.numel() > 1}
    return dict(opt=opt, out=out, d=case["opt"] == "kprodigy")


def run(state: dict) -> dict:
    state["opt"].step()
    if state["d"]:
        return dict(state["out"], d=state["opt"].get_d())
    return state["out"]


# ------------------------------------------------------------------- work
def _writes_grad(case: dict, shape: tuple[int, ...]) -> bool:
    """Which gradients the step leaves centralized: all matrices' by default; with
    ``fused`` only those of convolutions with quantized momentum, of bf16 params not
    written by stochastic rounding, and of 4-bit matrices of odd width up to 2**17
    padded elements; AdaMuon centers none and AdaPNM's ``fused`` writes none."""
    if case["opt"] == "adamuon" or len(shape) < 2:
        return False
    if not case.get("fused"):
        return True
    if case["opt"] == "adapnm":
        return False
    if case["dtype"] == "bf16" and case["method"] != "sr":
        return True
    if len(shape) > 2 and case["mom"] in ("int8", "4bit"):
        return True
    R, C = _rc(shape)
    pad = (1 << (R - 1).bit_length()) * (1 << (C - 1).bit_length())
    return pad <= 1 << 17 and case["mom"] == "4bit" and C % 2 == 1


def work(case: dict) -> dict:
    """Bytes: the gradient, the param and every state tensor read once, and what the step
    changes written once.  FLOPs: AdaMuon's Newton-Schulz products."""
    eb = 2 if case["dtype"] == "bf16" else 4
    mb = {"bf16": 2.0, "fp32": 4.0, "int8": 1.0, "4bit": 0.5}[case["mom"]]
    b = fl = 0.0
    for shape in _shapes(case):
        R, C = _rc(shape)
        n = R * C
        b += n * (eb + 2 * eb + 2 * mb)
        if _writes_grad(case, shape):
            b += n * eb
        if case["opt"] == "adapnm":
            b += n * mb
        b += 8 * _codec_sizes(case, n, R, len(shape))[1]
        if case["opt"] == "kprodigy":
            b += n * (8 + 8 + 4)  # v and s read and written, p0 read
        elif case["opt"] != "lion":
            b += 8 * (R + C if len(shape) > 1 else n)
        if case["method"] == "kahan" and eb == 2:
            b += 4 * n
        if case["opt"] == "adamuon" and len(shape) > 1:
            m, k = min(R, C), max(R, C)
            fl += 2 * (4.0 * m * m * k + 2.0 * m * m * m)
    return dict(bytes=b, flops=fl)


def tolerance(case: dict):
    """The library fixes the order of every sum it takes, so a step's results are the same
    bits on every correct build; only the Newton-Schulz products (bf16 matrix products,
    whose order is the hardware's) are held to a tolerance."""
    if case["opt"] == "adamuon":
        # 16-bit products: a sum order of another tile moves single bf16 roundings of the
        # orthogonal factor and with them some stochastically rounded weights by one bf16
        # step.  Against 64 bits the row / column statistics are 4e-7 off and the weights
        # 1.9e-3, the rounding of their write; two such writes differ by 2.7e-3 at most.
        return {"rel": 4e-3, "max": 0.05, "differ": 0.0}
    return "exact"


# ------------------------------------------------------------------ 64 bits
def _deq(case: dict, st: dict, key: str, shape: tuple[int, ...], R: int, C: int) -> torch.Tensor:
    m = st[key]
    if case["mom"] == "int8":
        return m.view(R, C).double() * st[key + "_scale"].view(-1, 1).double()
    if case["mom"] == "4bit":
        q = torch.stack((m & 15, m >> 4), dim=1).view(-1)[:R * C].double() - 8.0
        sc = st[key + "_scale"].double().repeat_interleave(st[key + "_block"])[:R * C]
        return (q * sc).view(R, C)
    return m.view(R, C).double()


def _requant(case: dict, st: dict, key: str, m: torch.Tensor, dims: int) -> tuple[torch.Tensor, torch.Tensor | None]:
    """(stored value, scales) of a new momentum; float momenta stay unrounded."""
    if case["mom"] == "int8":
        sc = (m.abs().amax(dim=1, keepdim=True)).clamp_min(1e-12) / 127.0
        return (m / sc).round().clamp(-127, 127) * sc, sc.view(-1)
    if case["mom"] == "4bit":
        b, n = st[key + "_block"], m.numel()
        nb = -(-n // b)
        x = torch.zeros(nb * b, dtype=torch.float64, device=DEV)
        x[:n] = m.view(-1)
        x = x.view(nb, b)
        sc = x.abs().amax(dim=1, keepdim=True).clamp_min(1e-12) / 7.0
        return ((x / sc).round().clamp(-7, 7) * sc).view(-1)[:n].view(m.shape), sc.view(-1)
    return m, None


def _newton_schulz(x: torch.Tensor, steps: int) -> torch.Tensor:
    a, b, c = 3.4445, -4.7750, 2.0315
    tr = x.shape[0] > x.shape[1]
    x = x.t().contiguous() if tr else x
    x = x / (x.norm() + 1e-7)
    for _ in range(steps):
        A = x @ x.t().contiguous()
        x = a * x + (b * A + c * (A @ A)) @ x
    return x.t().contiguous() if tr else x


@torch.no_grad()
def exact(case: dict, seed: int) -> dict | None:
    """One step in 64 bits from ``prepare``'s inputs.  The gradient's centering keeps the
    gradient's type (its definition); weights come without the rounding of their write."""
    b = _build(case, seed)
    f, kw, opt = b["f"], _hyper(case), case["opt"]
    b1, b2 = kw["betas"]
    lr, wd = kw["lr"], kw["weight_decay"]
    dt = _DT[case["dtype"]]
    names = [k for k in f if k != "p0" and f[k].buf.numel() > 1]
    out = {k: f[k].like(torch.float64) for k in names if f[k].buf.is_floating_point() and k != "shift"}
    cautious = opt != "kprodigy"
    gc = opt != "adamuon"
    t = _PNM_STEP + 1
    kept = []  # MSAM: (param, 64-bit weights, stored momentum); KProdigy: (param, ...)
    sq = num = den = 0.0
    for i, (shape, (R, C)) in enumerate(zip(b["shapes"], b["rc"])):
        st, mat = b["states"][i], len(shape) > 1
        put = lambda k, v: out[k].view(i, (v.numel(),)).copy_(v.reshape(-1)) if k in out else None  # noqa: E731
        p = f["p"].view(i, (R, C)).double()
        if "shift" in f:
            p = p + f["shift"].view(i, (R, C)).double()  # the compensated weight
        g0 = f["g"].view(i, (R, C))
        g = g0.double()
        if gc and mat:
            g = (g - g.mean(dim=1, keepdim=True).to(dt).double()).to(dt).double()
        put("g", g if _writes_grad(case, shape) else g0.double())
        key = ("m_pos" if t % 2 else "m_neg") if opt == "adapnm" else "m"
        m = _deq(case, st, key, shape, R, C)
        if opt == "adapnm":
            other = "m_neg" if key == "m_pos" else "m_pos"
            neg = _deq(case, st, other, shape, R, C)
            put(other, neg)
            if other + "_scale" in st:
                put(other + "_scale", st[other + "_scale"].double())
        new = None
        if opt == "lion":
            d = torch.sign((1 - b1) * g + b1 * m) + wd * p
            new = (1 - b2) * g + b2 * m
        elif opt == "kprodigy":
            dlr, b3 = _D * lr, math.sqrt(b2)
            flat = g.reshape(-1)
            num += float((flat * (st["p0"].double() - p.reshape(-1))).sum())
            s = b3 * st["s"].double() + (_D / _D0 * dlr) * flat
            put("s", s)
            den += float(s.abs().sum())
            new = b1 * m + _D * (1 - b1) * g
            v = b2 * st["v"].view(R, C).double() + _D * _D * (1 - b2) * g * g
            put("v", v)
            stored, sc = _requant(case, st, key, new, len(shape))
            kept.append((i, (R, C), p, stored, v))
            if sc is not None:
                put("m_scale", sc)
            else:
                put("m", new)
            continue
        else:
            x, eps = g, 1e-8 if opt == "adapnm" else 1e-30
            if opt == "adamuon" and mat:
                new = m + (1 - b1) * (g - m)
                x = _newton_schulz(new, kw["ns_steps"])
            w2 = 1 - b2
            if mat:
                row = st["row"].double() + w2 * ((x * x).mean(dim=1) + eps - st["row"].double())
                col = st["col"].double() + w2 * ((x * x).mean(dim=0) + eps - st["col"].double())
                put("row", row)
                put("col", col)
                inv = (row / row.mean()).rsqrt().view(-1, 1) * col.rsqrt().view(1, -1)
            elif opt == "adapnm":
                v = b2 * st["v"].view(R, C).double() + w2 * g * g
                put("v", v)
                inv = 1.0 / (((v + 1e-15).sqrt() + eps))
            else:
                v = st["v"].view(R, C).double() + w2 * (g * g + eps - st["v"].view(R, C).double())
                put("v", v)
                inv = v.rsqrt()
            if opt == "adapnm":
                beta0 = 0.5
                new = b1 * b1 * m + (1 - b1 * b1) * g
                u = ((1 + beta0) * new - beta0 * neg) / math.sqrt((1 + beta0) ** 2 + beta0 ** 2)
                u = u * inv * math.sqrt(1 - b2 ** t)
                scale = lr / (1 - b1 ** t)
                p = p * (1 - lr * wd)
            else:
                u, scale = x * inv, lr * (0.2 if opt == "adamuon" else 1.0)
            d = u / max(float(u.square().mean().sqrt()), 1.0) * scale
            if opt in ("adakaon", "nekaon", "msam") or (opt == "adamuon" and not mat):
                d = new = m + (1 - b1) * (d - m)
            if opt != "adapnm":
                d = d + lr * wd * p
        if cautious:
            mask = (d * g > 0).double()
            d = d * mask / max(float(mask.mean()), 1e-8)
        p = p - (lr * d if opt == "lion" else d)
        stored, sc = _requant(case, st, key, new, len(shape))
        if sc is not None:
            put(key + "_scale", sc)
        else:
            put(key, new)
        if opt == "nekaon":
            e = kw["k"] * lr
            p = p + (-kw["k"] * stored).clamp(-e, e)
        if opt == "msam":
            sq += float(stored.square().sum())
            kept.append((i, (R, C), p, stored, None))
        else:
            put("p", p)
    if opt == "msam":
        e = kw["rho"] / (math.sqrt(sq) + 1e-12)
        for i, rc, p, stored, _ in kept:
            out["p"].view(i, rc).copy_(p + e * stored)
    res: dict = {k: out[k].buf if k in out else None for k in names}
    if opt == "kprodigy":
        glob = _D * b["den"] * math.sqrt(b2) + _D / _D0 * _D * lr * num
        d_new = max(_D, glob / den)
        for i, rc, p, stored, v in kept:
            out["p"].view(i, rc).copy_(p - _D * lr * stored / v.sqrt().clamp_min(d_new * 1e-8))
        res["d"] = d_new
    if "shift" in f:
        res["p"] = None  # the weight and its compensation share the value: neither has one of its own
    return res
