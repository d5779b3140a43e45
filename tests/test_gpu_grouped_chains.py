"""The backward with four chains per workgroup, which grids of about one wave
per SIMD (961 to 1024 chains, the bf16 P1 scan without resets from 513) take: the P1 scan and the module's one-launch
form, at a number of chains that leaves three waves of the last workgroup
without one, with lanes past M."""
import pytest
import torch

import sparc_amd
from test_gpu_module import test_mixer_forward_backward_parity as module_parity
from test_gpu_scan import BF16, F32, make_case, rel_err
from test_gpu_split import _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,T,dtype,extra", [
    (17, 70, BF16, dict(h0=True, dlast=True)),
    (17, 70, BF16, dict(h0=True, dlast=True, seg=True)),
    (17, 3, F32, dict(h0=True, dlast=True)),
    (17, 70, F32, dict(dlast=True, reset_first=True)),
    (17, 260, BF16, dict(dlast=True)),  # from 256 steps on fewer chains split their time
    (9, 70, BF16, dict(h0=True, dlast=True)),  # 513 chains: the fewest, without resets in bf16
], ids=["bf16", "resets_bf16", "short_f32", "reset_first_f32", "long_bf16", "half_bf16"])
def test_p1_backward_grouped(B, T, dtype, extra):
    """969 = 17 x 57 and 513 = 9 x 57 chains of 128 modes against the general
    chain kernels (tolerances as for the split chains)."""
    M = 57 * 128 - 4
    print(f"[case] grouped P1 B={B} T={T} M={M} {dtype} {extra}", flush=True)
    case = make_case("p1", B, T, M, 1, dtype, seed=T, **extra)
    tol = 1e-5 if dtype == F32 else 2.0 ** -7
    for k, (a, b) in enumerate(zip(_run(case, "auto", True), _run(case, "chain", True))):
        assert rel_err(a, b) <= (tol if k < 4 else max(4 * tol, 5e-5)), f"tensor {k}: {rel_err(a, b):.3g}"


@pytest.mark.parametrize("L", [1, 10, 33])
@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-4), (torch.bfloat16, 2e-2)])
def test_one_launch_backward_grouped(L, dtype, tol):
    """969 = 17 x 57 chains of 64 modes in one launch, against the float64 oracle."""
    B, width = 17, 2 * (57 * 64 - 4)
    sparc_amd.set_mixer_path("fused")
    try:
        assert sparc_amd.backward_form(B, L, width // 2, dtype) == "one_launch"
        module_parity(dtype, tol, B, L, width, "fused")
    finally:
        sparc_amd.set_mixer_path("auto")
