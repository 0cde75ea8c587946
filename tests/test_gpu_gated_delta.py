"""The gated delta rule over many tokens (hif8_gated_delta) against its
token-by-token definition in float64."""

from __future__ import annotations

import ctypes

import pytest
import torch

from conftest import PKG_ROOT
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


@pytest.mark.parametrize("b,kh,rep,t,dk,dv", [(2, 3, 2, 70, 64, 32), (1, 2, 4, 130, 128, 128)])
def test_gated_delta_of_fewer_key_heads(native_ops, device, b, kh, rep, t, dk, dv):
    """The C entry with k_heads < heads, q and k [B, T, k_heads, dk] as a layer holds
    them: value head h reads key head h / rep, bit for bit as if they were repeated."""
    i64, ptr = ctypes.c_int64, ctypes.c_void_p
    lib = ctypes.CDLL(str(PKG_ROOT / "hif8_rocm" / "libhif8_rocm.so"))
    lib.hif8_last_error.restype = ctypes.c_char_p
    lib.hif8_gated_delta_workspace_size.argtypes, lib.hif8_gated_delta_workspace_size.restype = [i64] * 5, ctypes.c_size_t
    lib.hif8_gated_delta.argtypes = [ptr] * 8 + [i64] * 6 + [ptr, ctypes.c_size_t, ptr]
    h = kh * rep
    (q, k, _, _, _), _ = _inputs(b, kh, t, dk, dv, "tokens_first", device)
    (_, _, v, g, beta), state = _inputs(b, h, t, dk, dv, "tokens_first", device)
    want_state = state.clone()
    want = torch.ops.vllm_ascend_hif8.hif8_gated_delta(q.repeat_interleave(rep, dim=1), k.repeat_interleave(rep, dim=1),
                                                       v, g, beta, want_state)
    out = torch.empty(b, t, h, dv, device=device).transpose(1, 2)
    strides = (i64 * 18)(*[x.stride(i) for x in (q, k, v, g, beta, out) for i in range(3)])
    need = lib.hif8_gated_delta_workspace_size(b, h, t, dk, dv)
    ws = torch.empty(need, dtype=torch.uint8, device=device)
    torch.cuda.synchronize()
    pointers = [ptr(x.data_ptr()) for x in (q, k, v, g, beta)]
    assert lib.hif8_gated_delta(*pointers, strides, ptr(state.data_ptr()), ptr(out.data_ptr()), b, h, kh, t, dk, dv,
                                ptr(ws.data_ptr()), need, None) == 0, lib.hif8_last_error()
    torch.cuda.synchronize()
    assert torch.equal(out, want) and torch.equal(state, want_state)


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


def test_gated_delta_change_of_the_state_is_seen_by_autograd(native_ops, device):
    """A backward that needs the state as it was before the call is refused."""
    tensors, state = _inputs(1, 1, 70, 64, 16, "contiguous", device)
    scale = torch.ones_like(state, requires_grad=True)
    loss = (state * scale).sum()
    with torch.no_grad():
        assert synthetic_model._delta_kernel_takes(*tensors, state, 64)
        synthetic_model.gated_delta_chunked(*tensors, state)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        loss.backward()
    with torch.inference_mode():
        inference = state.clone()
    with pytest.raises(RuntimeError, match="[Ii]nference tensor"):
        synthetic_model.gated_delta_chunked(*tensors, inference)


@pytest.mark.parametrize("b,t,channels,width,ld", [(1, 1, 64, 4, 80), (2, 2, 64, 3, 70), (3, 3, 66, 4, 66),
                                                   (2, 16, 514, 2, 520), (1, 49, 1026, 4, 1030)])
def test_conv_tokens_equals_the_elementwise_form(native_ops, device, b, t, channels, width, ld):
    """Bit for bit, with fewer tokens than the state is long, run edges and a padded row pitch."""
    g = torch.Generator().manual_seed(t + channels)
    x = torch.randn(b, t, ld, generator=g).to(torch.bfloat16).to(device)
    w = torch.randn(channels, width, generator=g).to(torch.bfloat16).to(device)
    state = torch.randn(b, channels, width - 1, generator=g).to(torch.bfloat16).to(device)
    seq = torch.cat([state, x[..., :channels].transpose(1, 2)], dim=-1)
    acc = sum(seq[..., j:j + t].float() * w.float()[:, j:j + 1] for j in range(width))
    got = torch.ops.vllm_ascend_hif8.hif8_conv_tokens(x, w, state)
    torch.cuda.synchronize()
    assert torch.equal(got, torch.nn.functional.silu(acc).transpose(1, 2))
    assert torch.equal(state, seq[..., -(width - 1):])


@pytest.mark.parametrize("b,t,h,dv,offset", [(1, 1, 1, 2, 0), (2, 5, 3, 128, 6), (1, 4, 2, 130, 2), (1, 3, 2, 256, 0)])
def test_gated_rms_norm_matches_torch(native_ops, device, b, t, h, dv, offset):
    g = torch.Generator().manual_seed(dv + h)
    o = torch.randn(b, h, t, dv, generator=g).to(device).transpose(1, 2)
    mixed = torch.randn(b, t, offset + h * dv + 2, generator=g).to(torch.bfloat16).to(device)
    w = torch.randn(dv, generator=g).to(torch.bfloat16).to(device)
    z = mixed[..., offset:offset + h * dv].reshape(b, t, h, dv).double()
    want = synthetic_model.rms_norm(o, w, 1e-6).double() * torch.nn.functional.silu(z)
    got = torch.ops.vllm_ascend_hif8.hif8_gated_rms_norm(o, mixed, offset, w, 1e-6)
    torch.cuda.synchronize()
    # One rounding to bf16: eight significant bits, so at most 2^-8 of the value
    # (ulp 2^-7 at 1, half of it), plus FP32 terms of ~1e-6.
    torch.testing.assert_close(got.double(), want.reshape(b, t, -1), rtol=2 ** -8 + 1e-5, atol=1e-30)


def test_norms_of_more_rows_than_one_launch_holds(native_ops, device):
    """Rows past the 2^32 threads of one launch: the last ones equal a call of their own."""
    ops, g = torch.ops.vllm_ascend_hif8, torch.Generator(device=device).manual_seed(5)
    bf, rows, n = torch.bfloat16, 2 ** 23 + 9, 8
    h = torch.randn(rows, n, generator=g, device=device).to(bf)
    w = torch.rand(n, generator=g, device=device).to(bf)
    tail_h, delta = h[-40:].clone(), h.flip(0).contiguous()
    want, got = (ops.hif8_add_rms_norm(x, d, w, 1e-6) for x, d in ((tail_h, delta[-40:].contiguous()), (h, delta)))
    assert torch.equal(got[-40:], want) and torch.equal(h[-40:], tail_h)
    tokens = 2 ** 26 + 9
    o = torch.randn(1, tokens, 1, 2, generator=g, device=device)
    mixed = torch.randn(1, tokens, 2, generator=g, device=device).to(bf)
    got = ops.hif8_gated_rms_norm(o, mixed, 0, w[:2].contiguous(), 1e-6)
    want = ops.hif8_gated_rms_norm(o[:, -40:].contiguous(), mixed[:, -40:].contiguous(), 0, w[:2].contiguous(), 1e-6)
    assert torch.equal(got[:, -40:], want)


@pytest.mark.parametrize("rows,n", [(1, 8), (3, 24), (5, 6), (300, 1024)])
def test_silu_mul_equals_torch(native_ops, device, rows, n):
    g = torch.Generator().manual_seed(n)
    gu = (torch.randn(rows, 2 * n, generator=g) * 4).to(torch.bfloat16).to(device)
    gate, up = gu.float().split([n, n], dim=-1)
    assert torch.equal(torch.ops.vllm_ascend_hif8.hif8_silu_mul(gu),
                       (torch.nn.functional.silu(gate) * up).to(torch.bfloat16))
