"""fp32 gates beside bf16 writes on the kernels for lane-shared gates (serial
with 4 modes per lane, the 8-wave chain kernels, time segments), which the
automatic plan takes for them as for bf16 gates: every output and gradient
against the look-back kernels, which form each lane's transition by itself.

The states are fp32 recurrences in both and round to bf16 once, so an output or
write gradient whose last fp32 bits differ may round to the neighbouring bf16
value: with 8 significant bits that is at most 2^-7 of the value.  A gate
gradient is an fp32 sum over a group's modes of products with states read back
in bf16, whose rounding is the same in both unless that happens."""
import pytest
import torch

from sparc_amd import ops
from test_gpu_scan import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("transition,B,T,G,N,plan", [
    ("polar", 8, 70, 1024, 16, "serial, 4 modes per lane"),
    ("cartesian", 9, 65, 1022, 16, "serial, lanes past M"),
    ("polar", 4, 130, 512, 16, "chain"),
    ("polar", 1, 1023, 2304, 16, "chain, 288 workgroups"),
    ("real", 1, 1024, 4224, 16, "look-back, 264 chains"),
    ("real", 4, 130, 2048, 8, "chain"),
    ("real", 16, 129, 2048, 8, "serial"),
    ("polar", 1, 1100, 64, 16, "look-back"),
    ("cartesian", 2, 640, 33, 8, "look-back, lanes past M"),
    ("real", 1, 777, 48, 32, "look-back"),
    ("polar", 8, 1100, 240, 16, "backward in time segments"),
    ("cartesian", 1, 33000, 17, 16, "time segments, lanes past M"),
    ("real", 1, 33000, 16, 16, "time segments"),
])
@pytest.mark.parametrize("reset", [False, True])
def test_fp32_gates_lane_shared(transition, B, T, G, N, plan, reset):
    print(f"[case] fp32 gates {transition} B={B} T={T} G={G} N={N}: {plan} reset={reset}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(T + G)
    M = G * N
    cplx = transition != "real"
    r = torch.sigmoid(2.0 + torch.randn(B, T, G, device="cuda", generator=g))
    phi = (torch.rand(B, T, G, device="cuda", generator=g) * 2 - 1) * 3.14159
    gates = {"polar": (r, phi), "cartesian": (r * torch.cos(phi), r * torch.sin(phi)), "real": (r, None)}[transition]
    n = 2 if cplx else 1
    w = [torch.randn(B, T, M, device="cuda", generator=g).bfloat16() for _ in range(n)]
    h0 = [torch.randn(B, M, device="cuda", generator=g) for _ in range(n)]
    dy = [torch.randn(B, T, M, device="cuda", generator=g).bfloat16() for _ in range(n)]
    dl = [torch.randn(B, M, device="cuda", generator=g) for _ in range(n)]
    seg = torch.randint(0, 40, (B, T), device="cuda", generator=g, dtype=torch.int32) if reset else None
    got = {}
    for algo in ("lookback", "auto"):
        ops.set_algorithm(algo)
        try:
            leaves = [t.clone().requires_grad_() for t in (*gates[:n], *w, *h0)]
            gl, wl, hl = leaves[:n], leaves[n:2 * n], leaves[2 * n:]
            y, last = ops.chunk_scan(transition, gl[0], gl[1] if cplx else None, wl[0], wl[1] if cplx else None,
                                     initial_state=tuple(hl) if cplx else hl[0], segment_pos=seg)
            outs = [*(y if cplx else [y]), *(last if cplx else [last])]
            grads = torch.autograd.grad(outs, leaves, [*dy, *dl])
            got[algo] = [*outs, *grads]
            assert grads[0].dtype == torch.float32 and grads[n].dtype == torch.bfloat16
        finally:
            ops.set_algorithm("auto")
    for k, (a, b) in enumerate(zip(got["auto"], got["lookback"])):
        assert rel_err(a, b) <= 2.0 ** -7, f"tensor {k}: {rel_err(a, b):.3g}"


def _gate_gradients_64(gates, w, dy, N):
    """d gates of h_t = a_t h_{t-1} + w_t (polar, or real with one gate) in float64."""
    gates = [t.double().requires_grad_() for t in gates]
    w, dy = [t.double() for t in w], [t.double() for t in dy]
    a = torch.polar(*gates) if len(gates) == 2 else gates[0]
    a = a.repeat_interleave(N, dim=-1)
    w, dy = (torch.complex(*t) if len(t) == 2 else t[0] for t in (w, dy))
    h, hs = torch.zeros_like(w[:, 0]), []
    for t in range(w.shape[1]):
        h = a[:, t] * h + w[:, t]
        hs.append(h)
    loss = (torch.stack(hs, 1) * dy.conj()).real.sum()
    return torch.autograd.grad(loss, gates)


@pytest.mark.parametrize("transition,B,T,G,N,algo", [
    ("polar", 8, 70, 1024, 16, "auto"),     # 1024 chains of 128 modes
    ("polar", 8, 70, 512, 16, "auto"),      # 512 chains, the fewest whose states are recomputed
    ("real", 8, 70, 1024, 16, "auto"),      # 512 chains of 256 modes
    ("polar", 2, 130, 16, 16, "chain"),
    ("real", 2, 130, 16, 16, "serial"),
])
def test_fp32_gate_gradients_from_fp32_states(transition, B, T, G, N, algo):
    """fp32 gates get fp32 gradients: from states recomputed in fp32, not from
    the saved bf16 output, which is 2^-9 off.  A state is a sum of products
    that fades within some 20 steps, each rounded to 2^-24 of its value, as are
    the adjoint and the transition: 2e-6 is some thirty such roundings, and a
    thousandth of what one bf16 rounding of the states costs."""
    print(f"[case] fp32 gate gradients {transition} B={B} T={T} G={G} N={N} {algo}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(T + G)
    r = torch.sigmoid(2.0 + torch.randn(B, T, G, device="cuda", generator=g))
    phi = (torch.rand(B, T, G, device="cuda", generator=g) * 2 - 1) * 3.14159
    gates = [r, phi] if transition == "polar" else [r]
    w, dy = ([torch.randn(B, T, G * N, device="cuda", generator=g).bfloat16() for _ in gates] for _ in range(2))
    want = _gate_gradients_64(gates, w, dy, N)
    ops.set_algorithm(algo)
    try:
        leaves = [t.clone().requires_grad_() for t in gates]
        y, _ = ops.chunk_scan(transition, leaves[0], leaves[1] if len(leaves) == 2 else None, w[0],
                              w[1] if len(leaves) == 2 else None)
        got = torch.autograd.grad(list(y) if len(leaves) == 2 else [y], leaves, dy)
    finally:
        ops.set_algorithm("auto")
    for a, b in zip(got, want):
        err = ((a.double() - b).norm() / b.norm()).item()
        print(f"[case] off by {err:.3g}", flush=True)
        assert err <= 2e-6
