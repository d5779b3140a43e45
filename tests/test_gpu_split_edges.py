"""The P1 scan on both sides of the chain counts and lengths where its split
chains give way to time segments or to one wave per chain: against the general
chain kernels (tolerances as for the split chains)."""
import math

import pytest
import torch

from test_gpu_scan import BF16, F32, rel_err
from test_gpu_split import _run

pytestmark = pytest.mark.gpu


def _case(B, T, M, dtype, seg):
    """test_gpu_scan.make_case's P1 inputs, drawn on the GPU (they are large)."""
    g = torch.Generator(device="cuda").manual_seed(T + M)
    rn = lambda *s: torch.randn(*s, device="cuda", generator=g)
    ru = lambda *s: torch.rand(*s, device="cuda", generator=g).clamp(1e-6, 1 - 1e-6)
    return dict(g0=math.log(16.0) * torch.tanh(0.5 * rn(B, T, 1)), g1=0.5 * math.pi * torch.tanh(rn(B, T, 1)),
                nu_log=torch.log(-0.5 * torch.log(ru(M))), theta_log=torch.log(2 * math.pi * ru(M)),
                w_re=rn(B, T, M).to(dtype), w_im=rn(B, T, M).to(dtype), init=(rn(B, M), rn(B, M)),
                segpos=(ru(B, T) > 0.002).int() if seg else None, reset_first=False, relu=False,
                dy_re=rn(B, T, M).to(dtype), dy_im=rn(B, T, M).to(dtype), dlast=(rn(B, M), rn(B, M)))


@pytest.mark.parametrize("B,T,M,dtype,seg", [
    (5, 256, 16384, F32, False),   # 640 chains: the forward not split
    (5, 256, 16260, F32, True),    # lanes past M
    (2, 3073, 8192, BF16, True),   # 128 chains: the forward in segments
    (2, 1537, 17280, BF16, False),  # 270 chains: the backward in segments
    (2, 1537, 21500, BF16, True),  # 336 chains, with resets only
    (2, 3073, 8640, F32, False),   # 136 chains, fp32
    (4, 257, 50000, BF16, True),   # 1564 chains with resets: one wave per chain
])
def test_p1_split_edges(B, T, M, dtype, seg):
    print(f"[case] split edges B={B} T={T} M={M} {dtype} resets={seg}", flush=True)
    case = _case(B, T, M, dtype, seg)
    # T steps of a recurrence that may remember all of them, in another order
    tol = 1e-5 * max(1.0, T / 300) if dtype == F32 else 2.0 ** -7
    for k, (a, b) in enumerate(zip(_run(case, "auto", True), _run(case, "chain", True))):
        assert rel_err(a, b) <= (tol if k < 4 else max(4 * tol, 5e-5)), f"tensor {k}: {rel_err(a, b):.3g}"
