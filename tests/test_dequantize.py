"""dequantize on the GPU: the HIP pass against the torch formulation, bit for bit,
and the calls that stay with torch."""

from __future__ import annotations

import pytest
import torch

from decode_kernel import dequantize
from decode_kernel.quantize import _plain_gpu, dequantize_torch

pytestmark = pytest.mark.gpu


def _case(m: int, k: int, seed: int):
    g = torch.Generator(device="cuda").manual_seed(seed)
    packed = torch.randint(-2**31, 2**31, (m, k // 8), device="cuda", generator=g,
                           dtype=torch.int64).to(torch.int32)
    # Every fp16 pattern: subnormals, infinities, NaN and both signs.
    scales = torch.randint(0, 65536, (m, k // 128), device="cuda", generator=g)
    return packed, scales.to(torch.int16).view(torch.float16)


# One group; a last workgroup that is nearly empty (fp32: 1024 pieces of four
# weights, fp16: of eight); one past and one short of whole workgroups.
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("m,k", [(1, 128), (3, 128), (32, 128), (33, 128), (63, 128), (64, 128),
                                 (65, 128), (1000, 4224), (4096, 1152)])
def test_bits(m, k, dtype):
    packed, scales = _case(m, k, seed=m + k)
    assert _plain_gpu(packed, scales) is not None
    got, ref = dequantize(packed, scales, dtype=dtype), dequantize_torch(packed, scales, dtype=dtype)
    assert got.dtype == dtype and got.shape == (m, k) and got.is_contiguous()
    assert torch.equal(got.isnan(), ref.isnan())
    bits = torch.int32 if dtype == torch.float32 else torch.int16
    keep = ~ref.isnan()
    assert torch.equal(got.view(bits)[keep], ref.view(bits)[keep])
    # Words and scales that start anywhere their types may.
    pool = torch.cat([packed.reshape(-1)[:1], packed.reshape(-1)])[1:].view(m, -1)
    spool = torch.cat([scales.reshape(-1)[:1], scales.reshape(-1)])[1:].view(m, -1)
    again = dequantize(pool, spool, dtype=dtype)
    assert torch.equal(again.view(bits)[keep], ref.view(bits)[keep])


def test_calls_that_stay_with_torch():
    packed, scales = _case(16, 256, seed=1)
    scales = torch.rand_like(scales)
    ref = dequantize_torch(packed, scales)
    assert _plain_gpu(packed[:, ::2], scales) is None and _plain_gpu(packed.cpu(), scales) is None
    assert _plain_gpu(packed, scales.float()) is None
    assert torch.equal(dequantize(packed, scales.float()), ref)
    assert torch.equal(dequantize(packed, scales.t().contiguous().t()), ref)
    assert torch.equal(dequantize(packed, scales.reshape(-1)), ref)
    assert dequantize(packed, scales, dtype=torch.bfloat16).dtype == torch.bfloat16
    assert dequantize(packed, torch.rand(16, 4, device="cuda").half(), group_size=64).shape == (16, 256)
    s = scales.clone().requires_grad_()
    dequantize(packed, s).sum().backward()
    assert s.grad is not None
    _, tangent = torch.func.jvp(lambda t: dequantize(packed, t), (scales,), (scales,))
    assert torch.equal(tangent, ref)
    both = torch.func.vmap(lambda t: dequantize(packed, t))(torch.stack([scales, scales]))
    assert torch.equal(both[1], ref)
    with torch.no_grad():
        assert torch.equal(dequantize(packed, s), ref)
    param = torch.nn.Parameter(scales, requires_grad=False)
    assert _plain_gpu(packed, param) is not None and torch.equal(dequantize(packed, param), ref)


def test_under_a_default_device():
    """torch.set_default_device leaves a function mode on the stack for the whole
    process: it keeps the HIP pass; any other mode sees torch's operations."""
    packed, scales = _case(16, 256, seed=2)
    scales = torch.rand_like(scales)
    ref = dequantize_torch(packed, scales)
    for device in ("cuda", "cpu"):
        with torch.device(device):
            assert _plain_gpu(packed, scales) is not None
            assert torch.equal(dequantize(packed, scales), ref)
    seen = []

    class Watch(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    with torch.device("cuda"), Watch():
        assert _plain_gpu(packed, scales) is None
        out = dequantize(packed, scales)
    assert seen and torch.equal(out, ref)


def test_rows_past_int32():
    """K = 2^31, one more than the C ABI's int holds: torch's formulation, as
    before the kernel, with the bits that the kernel gives for each half."""
    words = 2**28
    g = torch.Generator(device="cuda").manual_seed(5)
    packed = torch.randint(-2**31, 2**31 - 1, (1, words), device="cuda", generator=g, dtype=torch.int32)
    scales = torch.rand(1, words // 16, device="cuda", generator=g).half()
    assert _plain_gpu(packed, scales) is None
    w = dequantize(packed, scales, dtype=torch.float16)
    assert w.shape == (1, 2**31)
    for p, s, half in zip(packed.chunk(2, 1), scales.chunk(2, 1), w.chunk(2, 1)):
        p, s = p.contiguous(), s.contiguous()
        assert _plain_gpu(p, s) is not None
        assert torch.equal(dequantize(p, s, dtype=torch.float16), half)
