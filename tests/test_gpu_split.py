"""The split-chain kernels (a chain's time shared by the waves of a workgroup)
at the sizes where they can go wrong: one round and its remainders, rounds
that end on and off the 64-step chunks, lanes past M, every number of waves
per chain, and the chain modes (states or relu out, an initial state, resets,
a gradient through the last state).

Few chains are held against the float64 oracle; the shapes with enough chains
for 16, 8 and 4 waves each against the general chain kernels, whose per-step
recurrence is the same: both are fp32 recurrences with relative error about
2^-24 per remembered step, so 1e-5 of max |reference| over 300 steps (bf16
I/O: values that differ in their last fp32 bits may round to neighbouring bf16
values, at most 2^-7 apart)."""
import pytest
import torch

import sparc_amd
from sparc_amd import ops
from test_gpu_module import _masked_dy, oracle_params
from test_gpu_scan import BF16, F32, check_case, make_case, rel_err

pytestmark = pytest.mark.gpu

FEW = [  # few chains: T from 16 to 768 steps is split
    ("one_round_f32", 2, 16, 256, F32, {}),
    ("one_past_f32", 2, 17, 132, F32, dict(h0=True, dlast=True)),
    ("chunk_less_one_bf16", 1, 63, 256, BF16, dict(h0=True)),
    ("chunk_plus_one_f32", 1, 65, 128, F32, dict(h0=True, dlast=True, seg=True)),
    ("round_plus_one_bf16", 2, 129, 260, BF16, dict(dlast=True)),
    ("resets_bf16", 2, 200, 128, BF16, dict(h0=True, dlast=True, seg=True, reset_first=True)),
    ("relu_f32", 2, 257, 132, F32, dict(relu=True, h0=True, dlast=True)),
    ("relu_resets_bf16", 2, 150, 256, BF16, dict(relu=True, seg=True)),
    ("longest_f32", 1, 768, 64, F32, dict(h0=True, dlast=True)),
    ("relu_longest_f32", 2, 288, 132, F32, dict(relu=True, h0=True, dlast=True)),
    ("relu_past_bf16", 2, 289, 132, BF16, dict(relu=True, dlast=True, seg=True)),  # the look-back's backward
    ("relu_36_chains_f32", 3, 290, 1500, F32, dict(relu=True, dlast=True)),
]


@pytest.mark.parametrize("cid,B,T,M,dtype,extra", FEW, ids=[c[0] for c in FEW])
def test_split_few_chains(cid, B, T, M, dtype, extra):
    print(f"[case] split {cid} B={B} T={T} M={M} {dtype}", flush=True)
    ops.set_algorithm("auto")
    check_case(make_case("p1", B, T, M, 1, dtype, seed=sum(map(ord, cid)) % 1000, **extra))


def _run(case, algorithm, want_grads):
    ops.set_algorithm(algorithm)
    try:
        names = ("g0", "g1", "nu_log", "theta_log", "w_re", "w_im")
        leaves = [case[n].cuda().requires_grad_(want_grads) for n in names]
        init = None if case["init"] is None else tuple(t.cuda().requires_grad_(want_grads) for t in case["init"])
        segpos = None if case["segpos"] is None else case["segpos"].cuda()
        y, last = ops.chunk_scan("p1", *leaves[:2], *leaves[4:], *leaves[2:4], initial_state=init, segment_pos=segpos,
                                 reset_first=case["reset_first"], relu_output=case["relu"])
        outs = [*([y] if case["relu"] else y), *last]
        if not want_grads:
            return outs
        dys = [case["dy_re"].cuda()] + ([] if case["relu"] else [case["dy_im"].cuda()]) + [d.cuda() for d in case["dlast"]]
        return outs + list(torch.autograd.grad(outs, leaves + list(init or ()), dys))
    finally:
        ops.set_algorithm("auto")


@pytest.mark.parametrize("B,M,dtype,extra", [
    (2, 8188, F32, dict(h0=True, dlast=True)),                            # 128 chains: 16 waves each
    (3, 8192, BF16, dict(dlast=True, relu=True)),                         # 192 chains: 8 waves
    (3, 8192, F32, dict(h0=True, dlast=True, seg=True)),
    (8, 8188, BF16, dict(h0=True, dlast=True, reset_first=True)),         # 512 chains: 4 waves
    (8, 8192, F32, dict(dlast=True, relu=True, h0=True)),
], ids=["waves16_f32", "waves8_relu_bf16", "waves8_resets_f32", "waves4_bf16", "waves4_relu_f32"])
@pytest.mark.parametrize("T", [256, 300])
def test_split_many_chains(B, M, dtype, extra, T):
    print(f"[case] split B={B} T={T} M={M} {dtype} {extra}", flush=True)
    case = make_case("p1", B, T, M, 1, dtype, seed=B + T, **extra)
    tol = 1e-5 if dtype == F32 else 2.0 ** -7
    n_out = 3 if extra.get("relu") else 4
    for k, (a, b) in enumerate(zip(_run(case, "auto", True), _run(case, "chain", True))):
        if k < n_out:
            assert rel_err(a, b) <= tol, f"output {k}: {rel_err(a, b):.3g}"
        elif extra.get("relu"):
            # a state within its rounding of zero may pass the relu in one form
            # and not in the other; its dy (of order 1) then moves the gradients
            # of the steps before it: in the 2-norm a few such states of some
            # millions
            e = ((a.float() - b.float()).norm() / b.float().norm().clamp_min(1e-30)).item()
            assert e <= (2e-3 if dtype == F32 else 1e-2), f"gradient {k - n_out}: {e:.3g}"
        else:
            # the transition gradients sum over the modes and steps
            assert rel_err(a, b) <= max(4 * tol, 5e-5), f"gradient {k - n_out}: {rel_err(a, b):.3g}"


@pytest.mark.parametrize("B,L,width,dtype", [
    (2, 20, 264, torch.float32), (1, 129, 2048, torch.bfloat16), (2, 300, 16376, torch.float32),
    (3, 256, 16384, torch.bfloat16), (8, 259, 16384, torch.bfloat16),
])
def test_split_module_forward(B, L, width, dtype):
    """The module's forward (few chains; 16, 8 and 4 waves per chain) against
    the composed path, whose scan runs the general kernels."""
    print(f"[case] split module B={B} L={L} width={width} {dtype}", flush=True)
    torch.manual_seed(L)
    m = sparc_amd.SPARCMixer(width).cuda()
    with torch.no_grad():
        for p in (m.phase_direction, m.radial_direction):
            p.copy_(torch.randn_like(p) * 0.5 / width ** 0.5)
        for p in (m.write_phase_response, m.write_radial_response):
            p.copy_(torch.randn_like(p) * 0.3)
        x = torch.randn(B, L, width, device="cuda").to(dtype)
        got = {}
        for path in ("fused", "composed"):
            sparc_amd.set_mixer_path(path)
            try:
                y, last = m(x, return_cache=True)
            finally:
                sparc_amd.set_mixer_path("auto")
            got[path] = [y, *last]
    # bf16: the write's rounding meets the states at other places when its last fp32 bit differs
    tol = 2e-5 if dtype == torch.float32 else 2.0 ** -7
    for a, b in zip(got["fused"], got["composed"]):
        assert rel_err(a, b) <= tol, rel_err(a, b)


@pytest.mark.parametrize("B,L,width,dtype", [
    (1, 1500, 256, torch.float32),          # time segments
    (2, 40, 512, torch.bfloat16),           # split chains
    (8, 70, 32768, torch.bfloat16),         # the wide kernel
    (1, 100, 32768, torch.float32),         # one wave per chain
])
def test_forward_without_gradients_matches(B, L, width, dtype):
    """The forward that keeps no states gives the same bits as the one that
    does, with gradients switched off and with nothing that requires them."""
    print(f"[case] no-gradient forward B={B} L={L} width={width} {dtype}", flush=True)
    torch.manual_seed(L)
    m = sparc_amd.SPARCMixer(width).cuda()
    x = torch.randn(B, L, width, device="cuda").to(dtype)
    y, last = m(x, return_cache=True)
    assert y.requires_grad
    with torch.no_grad():
        y1, last1 = m(x, return_cache=True)
    m.requires_grad_(False)
    y2, last2 = m(x, return_cache=True)
    for a, b, c in zip((y, *last), (y1, *last1), (y2, *last2)):
        assert torch.equal(a, b) and torch.equal(a, c) and not b.requires_grad


@pytest.mark.parametrize("B,L,width,dtype", [
    (1, 33, 264, torch.float32), (2, 257, 2048, torch.bfloat16),   # few chains
    (3, 259, 16384, torch.bfloat16),   # 192 chains of 128: 8 waves, 2 modes per lane
    (5, 260, 16376, torch.bfloat16),   # 320: 4 waves, 1 mode per lane
    (7, 256, 16384, torch.bfloat16),   # 448: 4 waves, 2 modes per lane
    (2, 300, 16376, torch.float32),    # 128, fp32
])
def test_split_module_backward(B, L, width, dtype):
    """Every gradient of the module's split backward against the composed path
    (separate operators on the general kernels).  The incoming gradient is
    masked where the state before the relu is near its edge and nowhere else:
    it reaches the kernel at clearly negative states, whose relu has to stop
    it."""
    print(f"[case] split module backward B={B} L={L} width={width} {dtype}", flush=True)
    torch.manual_seed(L + B)
    m = sparc_amd.SPARCMixer(width).cuda()
    with torch.no_grad():
        for p in (m.phase_direction, m.radial_direction):
            p.copy_(torch.randn_like(p) * 0.5 / width ** 0.5)
        for p in (m.write_phase_response, m.write_radial_response):
            p.copy_(torch.randn_like(p) * 0.3)
    x = torch.randn(B, L, width, device="cuda").to(dtype)
    dy = torch.randn(B, L, width, device="cuda").to(dtype)
    dl = torch.randn(B, width // 2, device="cuda")
    params = [m.phase_direction, m.radial_direction, m.nu_log, m.theta_log, m.write_log_gain,
              m.write_phase_response, m.write_radial_response]
    p = oracle_params(m, requires_grad=False)
    masked = _masked_dy(p, x.double().cpu(), dy.double().cpu(), band=1e-3 if dtype == torch.float32 else 2e-2)
    dy = masked.to(dtype).cuda()
    got = {}
    for path in ("composed", "fused"):
        sparc_amd.set_mixer_path(path)
        try:
            xx = x.clone().requires_grad_()
            y, last = m(xx, return_cache=True)
            got[path] = torch.autograd.grad([y, last[0]], [xx, *params], [dy, dl])
            assert (dy[y == 0] != 0).float().mean().item() > 0.5  # stopped states with a gradient coming in
        finally:
            sparc_amd.set_mixer_path("auto")
    tol = 1e-4 if dtype == torch.float32 else 2e-2
    for k, (a, b) in enumerate(zip(got["fused"], got["composed"])):
        assert rel_err(a, b) <= tol, f"gradient {k}: {rel_err(a, b):.3g}"


@pytest.mark.parametrize("B,L,M,dtype", [(2, 100, 260, torch.bfloat16), (3, 77, 132, torch.float32)])
def test_split_module_states_aligned_for_one_mode(B, L, M, dtype):
    """Through the C entry points with h_re, h_im on odd elements: where the
    split kernels hold two modes per lane the calls take the forms of one
    mode, and give the results of aligned states up to the order of the sums."""
    from sparc_amd import _lib
    print(f"[case] states off alignment B={B} L={L} M={M} {dtype}", flush=True)
    lib, P = _lib.load(), _lib.ptr
    g = torch.Generator(device="cuda").manual_seed(L)
    rn = lambda *s: torch.randn(*s, device="cuda", generator=g)
    x, dy = rn(B, L, 2 * M).to(dtype), rn(B, L, 2 * M).to(dtype)
    dirs = [rn(2 * M + 1) * 0.5 / (2 * M) ** 0.5 for _ in range(2)]
    modes = [torch.log(torch.rand(M, device="cuda", generator=g) + 0.01), rn(M), *(0.3 * rn(M) for _ in range(3))]
    st, io = _lib.stream_of(x.device), _lib.io_code(dtype)
    got = {}
    for off in (0, 1):
        controls = torch.empty(2, B * L, device="cuda")
        y = torch.empty_like(x)
        h = [torch.empty(B * L * M + 8, dtype=dtype, device="cuda")[off:off + B * L * M] for _ in range(2)]
        last = [torch.empty(B, M, device="cuda") for _ in range(2)]
        ws = torch.empty(lib.sparc_mixer_workspace_bytes(B, L, M, 0), dtype=torch.uint8, device="cuda")
        _lib.check(lib.sparc_mixer_forward(B, L, M, io, P(x), *map(P, dirs), *map(P, modes), P(controls[0]), P(controls[1]),
                                           P(y), *map(P, h), *map(P, last), P(ws), ws.numel(), st), "forward")
        dx = torch.empty_like(x)
        grads = [torch.empty(n, device="cuda") for n in (2 * M + 1, 2 * M + 1, M, M, M, M, M)]
        ws = torch.empty(lib.sparc_mixer_workspace_bytes(B, L, M, 1), dtype=torch.uint8, device="cuda")
        hs = h
        if off:  # the backward from the same states, moved
            hs = [torch.cat((t[:1], t))[1:] for t in got[0][1:3]]
            assert all(t.data_ptr() % (2 * t.element_size()) for t in (*h, *hs))
        _lib.check(lib.sparc_mixer_backward(B, L, M, io, P(x), *map(P, dirs), *map(P, modes), P(controls[0]), P(controls[1]),
                                            *map(P, hs), P(dy), None, None, P(dx), *map(P, grads), P(ws), ws.numel(), st),
                   "backward")
        got[off] = [y, *h, *last, dx, *grads]
    tol = 1e-5 if dtype == torch.float32 else 2.0 ** -7  # fp32 sums in another order, then one rounding
    for k, (a, b) in enumerate(zip(got[1], got[0])):
        assert rel_err(a, b) <= (tol if k < 6 else 5 * tol), f"tensor {k}: {rel_err(a, b):.3g}"
