"""What a caller may do with the gradients that the module's backward returns,
and with the tensors it keeps: each gradient is a tensor of its own."""
import pytest
import torch

import sparc_amd
from test_gpu_module import NAMES, make_module

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,L,width,dtype", [(2, 33, 264, torch.float32), (1, 300, 128, torch.bfloat16)])
def test_gradients_are_tensors_of_their_own(B, L, width, dtype):
    """No storage, version counter or view relation is shared: a gradient can
    be detached in place, scaled by a tensor that requires a gradient, and
    changed while another is saved for a backward; each starts on 16 bytes."""
    print(f"[case] module gradients B={B} L={L} width={width} {dtype}", flush=True)
    m = make_module(width, seed=5).cuda()
    x = torch.randn(B, L, width, device="cuda").to(dtype).requires_grad_()
    y, _ = m(x)
    params = [getattr(m, n) for n in NAMES]
    grads = torch.autograd.grad(y.float().square().sum(), [x, *params])
    for g in grads[1:]:
        assert g._base is None and g.data_ptr() % 16 == 0
        assert g.untyped_storage().nbytes() == g.numel() * g.element_size()
    scale = torch.ones((), device="cuda", requires_grad=True)
    saved = (grads[1] * scale).sum()  # keeps grads[1] for its backward
    for g in grads[2:]:
        g.detach_()
        g.mul_(scale)
    saved.backward()
    assert torch.isfinite(scale.grad)
