"""The controls kernels over every number of rows per workgroup that their
launches choose (forward 4 or 16 in fp32; backward 16 to 128 rows per row block, 4 to 128 inside the module),
at the first and last row counts of each and with partial last blocks,
against float64.

Tolerances: eta and delta are tanh of an fp32 sum of W products, whose
rounding error stays below sqrt(W) units of 2^-24 of the sum of absolute
products for random signs; dx is one fused multiply-add pair per element; a
direction gradient is a sum over the rows."""
import math

import pytest
import torch

import sparc_amd
from sparc_amd.control import make_controls

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,width", [(1, 64), (3, 1024), (4, 1032), (5, 2056), (4095, 2048), (4097, 2048), (8191, 64),
                                        (8192, 1032), (8193, 2056), (16383, 64), (16385, 1032)])
def test_controls_rows(rows, width):
    print(f"[case] controls rows={rows} width={width}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(rows + width)
    m = sparc_amd.SPARCMixer(width).cuda()
    with torch.no_grad():
        for p in (m.phase_direction, m.radial_direction):
            p.copy_(torch.randn(width + 1, device="cuda", generator=g) * 0.5 / math.sqrt(width))
    x = torch.randn(1, rows, width, device="cuda", generator=g).requires_grad_()
    params = (m.phase_direction, m.radial_direction)
    eta, delta = make_controls(m, x)
    d_eta, d_delta = (torch.randn(1, rows, device="cuda", generator=g) for _ in range(2))
    got = torch.autograd.grad((eta, delta), (x, *params), (d_eta, d_delta))
    x64 = x.detach().double().requires_grad_()
    p64 = [p.detach().double().requires_grad_() for p in params]
    eta64 = math.log(16.0) * torch.tanh(x64 @ p64[1][:-1] + p64[1][-1])
    delta64 = 0.5 * math.pi * torch.tanh(x64 @ p64[0][:-1] + p64[0][-1])
    want = torch.autograd.grad((eta64, delta64), (x64, *p64), (d_eta.double(), d_delta.double()))
    # |x.u| sums to about 0.4 sqrt(W) 0.5 in absolute products; log16 scales eta
    tol = 3.0 * math.log(16.0) * 0.2 * math.sqrt(width) * math.sqrt(width) * 2.0 ** -24
    for a, b in ((eta, eta64), (delta, delta64)):
        assert (a.double() - b).abs().max().item() <= max(tol, 2e-6)
    assert (got[0].double() - want[0]).abs().max().item() <= 1e-5 * want[0].abs().max().item()
    for a, b in zip(got[1:], want[1:]):
        # a sum of `rows` terms in fp32, each carrying eta's or delta's error
        assert (a.double() - b).abs().max().item() <= 1e-5 * math.sqrt(rows) + 1e-5 * b.abs().max().item()
