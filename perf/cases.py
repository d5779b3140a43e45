"""The calls that this framework's speed is measured on, through its public entry points.

Six kinds of call, each over the sizes, data types and options it is used with:

* ``module``   -- ``SPARCMixer.forward`` on a whole sequence, with its backward
                  (training) or without gradients and with the cache (prefill)
* ``block``    -- one ``SPARCBlock`` of the block stack, forward and backward
* ``p1``       -- the P1 scan operators: ``sparc_chunk_scan`` with and without
                  its relu output, ``sparc_tiled_serial_scan`` on packed sequences
* ``grouped``  -- ``polar_chunk_scan`` / ``grouped_real_scan``, gates shared by
                  the states of a channel
* ``elementwise`` -- ``complex_scan`` / ``real_scan``, a transition per element
* ``decode``   -- ``SPARCMixer.step`` after ``prepare_inference``

Every scan call but prefill and decode is a training pass: the forward, then the
gradients of every input for an incoming gradient ~ N(0, 1).
"""
from __future__ import annotations

import math

import torch

import sparc_amd
from sparc_amd.stack import SPARCBlock

DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16}
PARAMS = ("phase_direction", "radial_direction", "nu_log", "theta_log", "write_log_gain",
          "write_phase_response", "write_radial_response")


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the layer's training step at the size the scan is quoted at: d_model
        # 1024 with 16 states a channel, the controls on
        dict(name="module_train_large", kind="module", train=True, B=8, T=4096, W=32768, dtype="bf16"),
        # the smallest training step in use: d_model 64 with 16 states, where
        # the host and the launches are most of the time
        dict(name="module_train_small", kind="module", train=True, B=2, T=256, W=2048, dtype="fp32"),
        # one long document through a narrow layer: few chains, much time
        dict(name="module_train_long", kind="module", train=True, B=1, T=65536, W=2048, dtype="bf16"),
        # prompts of an odd length into the cache that decoding starts from
        dict(name="module_prefill", kind="module", train=False, B=3, T=1237, W=24576, dtype="bf16"),
        # one layer of the 12-layer stack (d_model 768, 16 states), a smaller batch
        dict(name="block_train", kind="block", B=4, T=2048, D=768, N=16, dtype="bf16"),
        # the scan operator as the layer itself calls it: relu(cat) output
        dict(name="p1_relu", kind="p1", op="relu", B=4, T=2048, M=8192, dtype="bf16"),
        # packed documents with a carried state, in full precision and at odd sizes
        dict(name="p1_packed", kind="p1", op="packed", B=3, T=4001, M=3000, dtype="fp32"),
        # the headline scan: bf16 throughout, gates shared by a channel's 16 states
        dict(name="polar_train", kind="grouped", op="polar", B=8, T=4096, G=1024, N=16, dtype="bf16", gates="bf16"),
        # the same scan as mixed-precision training feeds it: gates kept in fp32
        dict(name="polar_fp32_gates", kind="grouped", op="polar", B=4, T=4096, G=512, N=16, dtype="bf16",
             gates="fp32"),
        # a transition per element, full precision
        dict(name="complex_elementwise", kind="elementwise", op="complex", B=4, T=2048, M=4096, dtype="fp32"),
        # the gated real recurrence of a linear RNN layer
        dict(name="real_elementwise", kind="elementwise", op="real", B=8, T=4096, M=4096, dtype="bf16"),
        # one token for each of 256 streams, d_model 2048 with 16 states
        dict(name="decode_batch", kind="decode", B=256, W=65536, dtype="bf16"),
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, evenly spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _sizes(rng, most, width):
    """B and T for rows of ``width``: B * T * width up to ``most``."""
    b = _log(rng, 1, 16)
    t = _log(rng, 24, 65536)
    while b * t * width > most:
        if t > 64:
            t = t * 2 // 3
        else:
            b = max(1, b // 2)
    return b, t


def draw(rng):
    kind = rng.choice(("module", "module", "module", "block", "p1", "p1", "grouped", "grouped", "elementwise",
                       "decode"))
    dtype = rng.choice(("fp32", "bf16"))
    if kind == "module":
        modes = _log(rng, 32, 16384)
        if rng.random() < 0.8:
            modes = max(32, modes // 16 * 16)
        b, t = _sizes(rng, 1 << (27 if modes % 4 == 0 else 25), 2 * modes)
        return dict(kind=kind, train=rng.random() < 0.7, B=b, T=t, W=2 * modes, dtype=dtype)
    if kind == "block":
        d, n = 64 * rng.randint(2, 16), rng.choice((4, 8, 16))
        b, t = _sizes(rng, 1 << 25, 2 * d * n)
        return dict(kind=kind, B=b, T=t, D=d, N=n, dtype=dtype)
    if kind == "p1":
        op = rng.choice(("plain", "relu", "packed"))
        m = _log(rng, 64, 8192)
        if rng.random() < 0.8:
            m = m // 8 * 8
        b, t = _sizes(rng, 1 << 25, m)
        if op != "packed":  # these operators take whole chunks of 32 steps
            t = max(32, t // 32 * 32)
        return dict(kind=kind, op=op, B=b, T=t, M=m, dtype=dtype)
    if kind == "grouped":
        n = rng.choice((4, 8, 16, 32))
        g = _log(rng, 16, 16384 // n)
        b, t = _sizes(rng, 1 << 27, g * n)
        return dict(kind=kind, op=rng.choice(("polar", "real")), B=b, T=t, G=g, N=n, dtype=dtype,
                    gates=rng.choice(("fp32", "bf16")) if dtype == "bf16" else "fp32")
    if kind == "elementwise":
        m = _log(rng, 64, 8192)
        b, t = _sizes(rng, 1 << 26, m)
        return dict(kind=kind, op=rng.choice(("complex", "real")), B=b, T=t, M=m, dtype=dtype)
    return dict(kind="decode", B=_log(rng, 1, 256), W=2 * 16 * _log(rng, 8, 2048), dtype=dtype)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
class _Inputs:
    """Random tensors on the GPU, from the seed alone."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed))

    def randn(self, *shape, dtype=torch.float32, scale=1.0):
        return (torch.randn(*shape, device="cuda", generator=self.g) * scale).to(dtype)

    def rand(self, *shape, lo=0.0, hi=1.0, dtype=torch.float32):
        return (lo + (hi - lo) * torch.rand(*shape, device="cuda", generator=self.g)).to(dtype)

    def integers(self, lo, hi, *shape):
        return torch.randint(lo, hi, shape, device="cuda", generator=self.g)


def _spectrum(r, modes):
    """nu_log, theta_log of a freshly initialised layer (radius^2 and phase uniform)."""
    nu = -0.5 * torch.log(r.rand(modes, lo=1e-6, hi=1.0 - 1e-6))
    return torch.log(nu), torch.log(r.rand(modes, lo=1e-6, hi=2.0 * math.pi))


def _fill_mixer(m, r):
    """A layer that has trained a little: the initial spectrum, the controls on."""
    with torch.no_grad():
        nu_log, theta_log = _spectrum(r, m.modes)
        m.nu_log.copy_(nu_log)
        m.theta_log.copy_(theta_log)
        gain = torch.log(torch.sqrt(1.0 - torch.exp(-2.0 * torch.exp(nu_log))) + 1.0e-8)
        m.write_log_gain.copy_(gain)
        scale = 0.5 / math.sqrt(m.width)
        m.phase_direction.copy_(r.randn(m.width + 1, scale=scale))
        m.radial_direction.copy_(r.randn(m.width + 1, scale=scale))
        m.write_phase_response.copy_(r.randn(m.modes, scale=0.3))
        m.write_radial_response.copy_(r.randn(m.modes, scale=0.3))


def _segments(r, b, t):
    """Positions inside packed documents of about 500 steps; the first of a row
    goes on from an earlier batch."""
    starts = r.rand(b, t) < 1.0 / 500.0
    starts[:, 0] = False
    step = torch.arange(t, device="cuda").expand(b, t)
    last = torch.where(starts, step, torch.full_like(step, -(t + 1))).cummax(dim=1).values
    return torch.where(last < 0, step + 1 + r.integers(0, 1000, b, 1), step - last).to(torch.int32)


def _leaf(t):
    return t.detach().requires_grad_()


def prepare(case, seed):
    r, dt, kind = _Inputs(seed), DTYPES[case["dtype"]], case["kind"]
    s = {"case": case}
    if kind in ("module", "decode"):
        m = sparc_amd.SPARCMixer(case["W"]).cuda()
        _fill_mixer(m, r)
        s["module"] = m
        if kind == "decode":
            m.requires_grad_(False)
            m.prepare_inference()
            s["x"] = r.randn(case["B"], case["W"], dtype=dt)
            s["state"] = (r.randn(case["B"], m.modes, scale=0.1), r.randn(case["B"], m.modes, scale=0.1))
            return s
        s["x"] = r.randn(case["B"], case["T"], case["W"], dtype=dt)
        if case["train"]:
            s["x"] = _leaf(s["x"])
            s["dy"] = r.randn(case["B"], case["T"], case["W"], dtype=dt)
            s["inputs"] = [s["x"], *[getattr(m, n) for n in PARAMS]]
    elif kind == "block":
        blk = SPARCBlock(case["D"], case["N"]).cuda()
        with torch.no_grad():
            width = 2 * case["D"] * case["N"]
            blk.norm.weight.copy_(1.0 + r.randn(case["D"], scale=0.1))
            blk.in_proj.weight.copy_(r.randn(width, case["D"], scale=case["D"] ** -0.5))
            blk.out_proj.weight.copy_(r.randn(case["D"], width, scale=width ** -0.5))
        _fill_mixer(blk.mixer, r)
        s["block"] = blk = blk.to(dt)
        s["x"] = _leaf(r.randn(case["B"], case["T"], case["D"], dtype=dt))
        s["dy"] = r.randn(case["B"], case["T"], case["D"], dtype=dt)
        s["inputs"] = [s["x"], blk.norm.weight, blk.in_proj.weight, blk.out_proj.weight,
                       *[getattr(blk.mixer, n) for n in PARAMS]]
    elif kind == "p1":
        b, t, m = case["B"], case["T"], case["M"]
        nu_log, theta_log = _spectrum(r, m)
        eta = math.log(16.0) * torch.tanh(r.randn(b, t, scale=0.5))
        delta = 0.5 * math.pi * torch.tanh(r.randn(b, t, scale=0.5))
        w = [r.randn(b, t, m, dtype=dt) for _ in range(2)]
        s["inputs"] = [_leaf(v) for v in (eta, delta, nu_log, theta_log, *w)]
        if case["op"] == "relu":
            s["dy"] = [r.randn(b, t, 2 * m, dtype=dt)]
        else:
            s["dy"] = [r.randn(b, t, m, dtype=dt) for _ in range(2)]
        if case["op"] == "packed":
            s["segment_pos"] = _segments(r, b, t)
            s["inputs"] += [_leaf(r.randn(b, m)) for _ in range(2)]
            s["dy"] += [r.randn(b, m) for _ in range(2)]
    elif kind == "grouped":
        b, t, g, m = case["B"], case["T"], case["G"], case["G"] * case["N"]
        gdt = DTYPES[case["gates"]]
        if case["op"] == "polar":
            gates = [torch.sigmoid(2.0 + r.randn(b, t, g)).to(gdt), r.rand(b, t, g, lo=-math.pi, hi=math.pi, dtype=gdt)]
        else:
            gates = [r.rand(b, t, g, lo=0.95, hi=0.9999, dtype=gdt)]
        n = len(gates)
        s["inputs"] = [_leaf(v) for v in (*gates, *[r.randn(b, t, m, dtype=dt) for _ in range(n)])]
        s["dy"] = [r.randn(b, t, m, dtype=dt) for _ in range(n)]
    else:
        b, t, m = case["B"], case["T"], case["M"]
        if case["op"] == "complex":
            rad, phi = r.rand(b, t, m, lo=0.9, hi=0.999), r.rand(b, t, m, lo=-math.pi, hi=math.pi)
            gates = [(rad * torch.cos(phi)).to(dt), (rad * torch.sin(phi)).to(dt)]
        else:
            gates = [torch.sigmoid(2.0 + r.randn(b, t, m)).to(dt)]
        n = len(gates)
        s["inputs"] = [_leaf(v) for v in (*gates, *[r.randn(b, t, m, dtype=dt) for _ in range(n)])]
        s["dy"] = [r.randn(b, t, m, dtype=dt) for _ in range(n)]
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "decode":
        return state["module"].step(state["x"], state["state"], None)
    if kind == "module" and not case["train"]:
        with torch.no_grad():
            return state["module"](state["x"], return_cache=True)
    if kind == "module":
        y, _ = state["module"](state["x"])
        outs, dys = [y], [state["dy"]]
    elif kind == "block":
        outs, dys = [state["block"](state["x"])], [state["dy"]]
    else:
        i, dys = state["inputs"], state["dy"]
        if kind == "p1" and case["op"] == "packed":
            outs = sparc_amd.sparc_tiled_serial_scan(*i[:6], segment_pos=state["segment_pos"],
                                                     initial_state=(i[6], i[7]))
        elif kind == "p1":
            outs = sparc_amd.sparc_chunk_scan(*i, fused_output_relu=case["op"] == "relu")
        elif kind == "grouped" and case["op"] == "polar":
            outs, _ = sparc_amd.polar_chunk_scan(*i)
        elif kind == "grouped":
            outs, _ = sparc_amd.grouped_real_scan(*i)
        else:
            outs = (sparc_amd.complex_scan if case["op"] == "complex" else sparc_amd.real_scan)(*i)
        outs = [outs] if torch.is_tensor(outs) else list(outs)
    return [o.detach() for o in outs], list(torch.autograd.grad(outs, state["inputs"], dys))


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    """Inputs read once, outputs and gradients written once; the operations of
    the recurrence (8 a complex multiply-add, forward; twice that and the
    transition's gradient backward) and of the products beside it."""
    kind, es = case["kind"], 2 if case["dtype"] == "bf16" else 4
    if kind == "decode":
        bw = case["B"] * case["W"]
        return {"bytes": bw * (2 * es + 8) + 14 * case["W"], "flops": bw * 10}
    rows = case["B"] * case["T"]
    if kind == "module":
        el = rows * case["W"]
        if case["train"]:  # x, dy in; y, dx out
            return {"bytes": 4 * el * es, "flops": el * 22}
        return {"bytes": 2 * el * es, "flops": el * 8}
    if kind == "block":
        d, w = case["D"], 2 * case["D"] * case["N"]
        # six products; x, dy in, y, dx out; the weights in, their gradients out
        return {"bytes": 4 * rows * d * es + 4 * d * w * es, "flops": 12 * rows * d * w + rows * w * 22}
    if kind == "p1":
        el = rows * case["M"]
        return {"bytes": 8 * el * es + 16 * rows, "flops": el * 32}
    planes, per = (2, 32) if case["op"] in ("polar", "complex") else (1, 6)
    if kind == "grouped":
        el, gs = rows * case["G"] * case["N"], 2 if case["gates"] == "bf16" else 4
        return {"bytes": planes * (4 * el * es + 2 * rows * case["G"] * gs), "flops": el * per}
    el = rows * case["M"]
    return {"bytes": planes * 6 * el * es, "flops": el * per}


def tolerance(case):
    """About four times what a pass is off its 64-bit values by.  Where a relu
    stands behind the scan, a state within its own rounding of zero may fall on
    either side, and the gradients of the steps before it take or leave the whole
    incoming gradient there: in bf16, with the write rounded, one state in a
    thousand does (gradients 0.02 - 0.05 off), in fp32 one in some millions
    (up to 3e-3 over long sequences)."""
    kind, bf16 = case["kind"], case["dtype"] == "bf16"
    if kind == "block" or (kind == "module" and case["train"]):
        return {"rel": 3e-2 if bf16 else 1e-2, "max": 0.99}
    if kind == "p1" and case["op"] == "relu":
        return {"rel": 1e-2, "max": 0.99}
    if bf16:  # each output and gradient is rounded to 8 bits once: 1.6e-3 - 2.3e-3
        return {"rel": 1e-2}
    if kind == "decode":  # sums over the width, then a step: 1.2e-7 - 5e-7
        return {"rel": 2e-6}
    if kind == "elementwise":  # a recurrence that forgets within some 1000 steps: 1e-7 - 2e-7
        return {"rel": 2e-6}
    # the phase and decay of slow modes add up over the steps they remember:
    # 1e-6 - 2e-5, more the longer the sequence
    return {"rel": 1e-4}


# ---------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# ---------------------------------------------------------------------------
class _Scan64(torch.autograd.Function):
    """h_t = a_t h_{t-1} + w_t over [B, T, M], complex or real."""

    @staticmethod
    def forward(ctx, a, w, h0):
        h, prev = torch.empty_like(w), h0
        for at, wt, ht in zip(a.unbind(1), w.unbind(1), h.unbind(1)):
            torch.addcmul(wt, at, prev, out=ht)
            prev = ht
        ctx.save_for_backward(a, h, h0)
        return h

    @staticmethod
    def backward(ctx, dh):
        a, h, h0 = ctx.saved_tensors
        ac, lam = a.conj().resolve_conj(), torch.empty_like(dh)
        adj = torch.zeros_like(h0)
        for at, dt, lt in zip(ac.unbind(1)[::-1], dh.unbind(1)[::-1], lam.unbind(1)[::-1]):
            lt.copy_(dt).add_(adj)
            adj = at * lt
        before = torch.cat((h0[:, None], h[:, :-1]), dim=1)
        return lam * before.conj(), lam, adj


def _p1_transition(eta, delta, nu_log, theta_log):
    em = torch.expm1(-torch.exp(nu_log) * torch.exp(eta)[..., None])
    phase = torch.exp(theta_log) - em * delta[..., None]
    return (1.0 + em) * torch.complex(torch.cos(phase), torch.sin(phase))


def _mixer64(x, pd, rd, nu_log, theta_log, log_gain, phase_response, radial_response, scan):
    modes = nu_log.numel()
    phase, radial = torch.tanh(x @ pd[:-1] + pd[-1]), torch.tanh(x @ rd[:-1] + rd[-1])
    eta, delta = math.log(16.0) * radial, 0.5 * math.pi * phase
    nu = torch.exp(nu_log)
    ratio = torch.sqrt(torch.expm1(-2.0 * nu * torch.exp(eta)[..., None]) / torch.expm1(-2.0 * nu))
    gate = 2.0 * torch.sigmoid(phase[..., None] * phase_response + radial[..., None] * radial_response)
    gain = torch.exp(log_gain) * ratio * gate
    w = torch.complex(gain * torch.tanh(x[..., :modes]), gain * torch.tanh(x[..., modes:]))
    h = scan(_p1_transition(eta, delta, nu_log, theta_log), w,
             torch.zeros(x.shape[0], modes, dtype=w.dtype, device=x.device))
    return torch.cat((h.real, h.imag), dim=-1).relu(), h[:, -1]


def _block64(x, norm, w_in, w_out, *params, scan):
    xn = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * norm
    y, _ = _mixer64(xn @ w_in.t(), *params, scan)
    return x + y @ w_out.t()


def _expand(g, n):
    return g.repeat_interleave(n, dim=-1)


def exact(case, seed):
    s = prepare(case, seed)
    kind, scan = case["kind"], _Scan64.apply
    if kind == "decode":
        m, x = s["module"], s["x"].double()
        p = [getattr(m, n).detach().double() for n in PARAMS]
        h0 = torch.complex(*[v.double() for v in s["state"]])
        y, h = _mixer64(x[:, None], *p, lambda a, w, _: a * h0[:, None] + w)
        return y[:, 0], (h.real, h.imag)
    b, t = case["B"], case["T"]
    width = {"module": lambda: case["W"] // 2, "block": lambda: case["D"] * case["N"], "p1": lambda: case["M"],
             "grouped": lambda: case["G"] * case["N"], "elementwise": lambda: case["M"]}[kind]()
    rows = max(1, (1 << 27) // (t * width))  # batch rows at a time: they meet in the parameters' gradients only
    if -(-b // rows) * t > 150000:
        return None
    if kind == "module" and not case["train"]:
        with torch.no_grad():
            p = [getattr(s["module"], n).detach().double() for n in PARAMS]
            got = [_mixer64(s["x"][k:k + rows].double(), *p, scan) for k in range(0, b, rows)]
        y, last = torch.cat([g[0] for g in got]), torch.cat([g[1] for g in got])
        return y, (last.real, last.imag)
    dys = s["dy"] if isinstance(s["dy"], list) else [s["dy"]]
    shared = [i.dim() < 3 and not (kind == "p1" and i.dim() == 2) for i in s["inputs"]]
    if kind == "block":
        shared = [k > 0 for k in range(len(s["inputs"]))]
    whole = [_leaf(i.double()) if sh else None for i, sh in zip(s["inputs"], shared)]
    outs, grads = [], []
    for k in range(0, b, rows):
        cut = slice(k, k + rows)
        i = [w if sh else _leaf(v[cut].double()) for v, w, sh in zip(s["inputs"], whole, shared)]
        if kind == "module":
            o = [_mixer64(*i, scan)[0]]
        elif kind == "block":
            o = [_block64(*i, scan=scan)]
        else:
            if kind == "p1":
                a, w = _p1_transition(*i[:4]), torch.complex(i[4], i[5])
                if case["op"] == "packed":
                    a = a * (s["segment_pos"][cut] != 0)[..., None]
            elif case["op"] == "polar":
                r, phi = i[:2]
                a, w = torch.complex(r * torch.cos(phi), r * torch.sin(phi)), torch.complex(i[2], i[3])
                a = _expand(a, case["N"])
            elif case["op"] == "complex":
                a, w = torch.complex(i[0], i[1]), torch.complex(i[2], i[3])
            else:
                a, w = (_expand(i[0], case["N"]) if kind == "grouped" else i[0]), i[1]
            packed = kind == "p1" and case["op"] == "packed"
            h0 = torch.complex(i[6], i[7]) if packed else torch.zeros_like(w[:, 0])
            h = scan(a, w, h0)
            if not w.is_complex():
                o = [h]
            elif kind == "p1" and case["op"] == "relu":
                o = [torch.cat((h.real, h.imag), dim=-1).relu()]
            else:
                o = [h.real, h.imag]
            if packed:
                o += [h[:, -1].real, h[:, -1].imag]
        g = torch.autograd.grad(o, i, [d[cut].double() for d in dys])
        outs.append([v.detach() for v in o])
        grads.append(g)
    return ([torch.cat(v) for v in zip(*outs)],
            [sum(v) if sh else torch.cat(v) for v, sh in zip(zip(*grads), shared)])
