"""The gated delta rule over many tokens (hif8_gated_delta) against its
token-by-token definition in float64."""

from __future__ import annotations

import pytest
import torch

from hif8_rocm import synthetic_model

pytestmark = pytest.mark.gpu


def _inputs(b, h, t, dk, dv, layout, device):
    g = torch.Generator().manual_seed(1000 * t + dk + dv)

    def rand(*shape):
        return torch.randn(*shape, generator=g)

    norm = torch.nn.functional.normalize
    q, k, v = norm(rand(b, h, t, dk), dim=-1) * dk ** -0.5, norm(rand(b, h, t, dk), dim=-1), rand(b, h, t, dv)
    decay, beta = -torch.rand(b, h, t, generator=g) * 0.5, torch.rand(b, h, t, generator=g)
    state = rand(b, h, dk, dv) * 0.1
    tensors = [x.to(device) for x in (q, k, v, decay, beta)]
    if layout == "tokens_first":  # as a layer holds them
        tensors = [x.transpose(1, 2).contiguous().transpose(1, 2) for x in tensors]
    elif layout == "unaligned":  # rows that start on 4-byte addresses, gates with a stride
        tensors = [torch.cat([x[..., :1], x], dim=-1)[..., 1:] if x.ndim == 4 else
                   torch.stack([x, -x], dim=-1)[..., 0] for x in tensors]
    elif layout == "dims_strided":
        tensors = [x.transpose(-1, -2).contiguous().transpose(-1, -2) if x.ndim == 4 else x for x in tensors]
    return tensors, state.to(device)


@pytest.mark.parametrize("b,h,t,dk,dv,layout", [
    (1, 1, 1, 64, 16, "contiguous"), (1, 3, 63, 128, 128, "tokens_first"), (2, 2, 64, 128, 48, "unaligned"),
    (1, 9, 65, 64, 128, "dims_strided"), (2, 5, 200, 128, 256, "tokens_first"), (1, 2, 449, 64, 64, "unaligned"),
])
def test_gated_delta_matches_the_recurrence(native_ops, device, b, h, t, dk, dv, layout):
    tensors, state = _inputs(b, h, t, dk, dv, layout, device)
    want_state = state.double()
    want = torch.empty(b, h, t, dv, dtype=torch.float64, device=device)
    q, k, v, g, beta = (x.double() for x in tensors)
    for i in range(t):
        want[:, :, i] = synthetic_model.gated_delta_step(want_state, q[:, :, i], k[:, :, i], v[:, :, i], g[:, :, i],
                                                         beta[:, :, i])
    assert synthetic_model._delta_kernel_takes(*tensors, state, 64)
    got = synthetic_model.gated_delta_chunked(*tensors, state)
    torch.cuda.synchronize()
    # FP32 sums of up to 128 products per term, a few terms deep: ~2^-24 sqrt(128) each.
    for x, y in ((got, want), (state, want_state)):
        assert x.dtype == torch.float32 and float((x.double() - y).norm() / y.norm()) < 1e-6


def test_gated_delta_leaves_autograd_and_other_types_to_torch(native_ops, device):
    tensors, state = _inputs(1, 1, 70, 64, 16, "contiguous", device)
    takes = synthetic_model._delta_kernel_takes
    assert takes(*tensors, state, 64)
    assert not takes(*tensors, state, 32)
    assert not takes(*[x.double() for x in tensors], state.double(), 64)
    assert not takes(*[x.cpu() for x in tensors], state.cpu(), 64)
    assert not takes(*tensors[:2], tensors[2].requires_grad_(), *tensors[3:], state, 64)
    with torch.no_grad():
        assert takes(*tensors, state, 64)
