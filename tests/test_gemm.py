"""The many-batch kernel (dk_w4a16_linear, dk_gate_up_silu above 16 batch rows).

On the CPU, where the dispatch draws its lines (the describe entry points
launch nothing): which calls stay on the kernels they had, and which take
gemm_w4. On the GPU, every launch shape of the kernel at the sizes where it can
go wrong: rows and batches one past and one short of a tile, K parts without a
group, one group, odd group counts, operands aligned to no more than the ABI
asks, against a float64 product of the dequantized weight within half an fp16
step + 1e-3 (fp16 rounding of y, plus the fp32 sums).
"""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from decode_kernel import _abi
from oracle import oracle


@pytest.fixture(scope="module")
def lib():
    return _abi.load()


@pytest.mark.parametrize("m,k,b,kernel,blocks", [
    # Scales in pairs, rows of over 1024 weights: over 256 tiles of 32 x 32;
    # over 8192 rows and up to 3 2^16 activations up to 32 batch rows.
    (8192, 8192, 17, "gemv_reuse", None),
    (8193, 8192, 17, "gemm_w4<1, 8, 1, 2, false>", 129),
    (8193, 6144, 32, "gemm_w4<1, 8, 1, 2, false>", 129),
    (8193, 6400, 32, "gemv_reuse", None),
    (12288, 28672, 17, "gemv_reuse", None),
    (4096, 4096, 64, "gemv_reuse", None),
    (4096, 4096, 65, "gemm_w4<1, 8, 2, 1, false>", 256),
    (4097, 4096, 33, "gemm_w4<1, 8, 2, 1, false>", 129),
    (4096, 4096, 129, "gemm_w4<1, 8, 2, 2, false>", 192),
    (4096, 4096, 1000, "gemm_w4<2, 4, 4, 2, false>", 256),
    (1024, 8192, 256, "gemv_reuse", None),
    (1024, 8192, 257, "gemm_w4<1, 8, 2, 1, false>", 160),
    (28672, 8192, 2048, "gemm_w4<4, 1, 4, 2, false>", 1792),
    # At 129 to 304 rows of over 1536 weights not from 321 tiles up to 128 of
    # 64 x 64.
    (256, 1536, 1409, "gemm_w4<", None),
    (227, 3584, 1432, "gemv_reuse_pfb<", None),
    (129, 4096, 2100, "gemv_reuse", None),
    (128, 4096, 2700, "gemm_w4<", None),
    (256, 4096, 1280, "gemm_w4<", None),
    (304, 4096, 1600, "gemv_reuse", None),
    (304, 4096, 1601, "gemm_w4<", None),
    (305, 4096, 1500, "gemm_w4<", None),
    (4096, 1024, 1000, "gemv_reuse_pfb<", None),
    # Odd group counts: over 512 tiles of 16 x 16, 384 at 1025 to 2048 rows
    # above 32 batch rows.
    (4096, 4224, 32, "gemv_reuse_lds<", None),
    (4097, 4224, 32, "gemm_w4<1, 8, 1, 1, false>", 129),
    (2032, 4224, 33, "gemv_reuse", None),
    (2033, 4224, 33, "gemm_w4<1, 8, 1, 1, false>", 128),
    (2048, 4224, 48, "gemm_w4<1, 8, 1, 1, false>", 128),
    (2049, 4224, 33, "gemv_reuse", None),
    (2736, 4224, 48, "gemm_w4<1, 8, 1, 1, false>", 172),
    (1024, 4224, 128, "gemv_reuse", None),
    (1024, 4224, 129, "gemm_w4<1, 8, 1, 1, false>", 160),
    (5000, 4224, 20, "gemm_w4<1, 8, 1, 1, false>", 157),
    # Short rows, odd group counts: up to 32 batch rows gemm_w4 from two thirds
    # of a round of its launch shape on; from 33 to 48 the 16-row tiles over
    # 4096 rows up to 10880 (5440 on rows of over 1024 weights), to 72 up to
    # 6144; with one group but for one round of 32 x 32 tiles, over 352 tiles of
    # 64 x 64 (296 from 33 to 64 batch rows) or over 192 batch rows.
    (4161, 384, 17, "gemv_reuse_lds<", None),
    (12288, 640, 32, "gemv_reuse_lds<", None),
    (12289, 640, 32, "gemm_w4<1, 8, 1, 2, false>", 193),
    (16385, 640, 32, "gemv_reuse_lds<", None),
    (21504, 640, 32, "gemv_reuse_lds<", None),
    (21505, 640, 32, "gemm_w4<2, 4, 2, 2, false>", 169),
    (32768, 640, 17, "gemm_w4<2, 4, 2, 2, false>", 256),
    (32769, 640, 17, "gemv_reuse_lds<", None),
    (45056, 384, 24, "gemv_reuse_lds<", None),
    (45057, 384, 24, "gemm_w4<", None),
    (4096, 896, 48, "gemm_w4<", None),
    (4097, 896, 48, "gemv_reuse", None),
    (10880, 896, 48, "gemv_reuse_lds<", None),
    (10881, 896, 48, "gemm_w4<", None),
    (4096, 640, 49, "gemm_w4<", None),
    (4097, 640, 72, "gemv_reuse", None),
    (4097, 640, 73, "gemm_w4<", None),
    (4864, 640, 72, "gemv_reuse", None),
    (4865, 640, 65, "gemm_w4<1, 8, 1, 2, false>", 231),
    (5440, 640, 72, "gemm_w4<1, 8, 1, 2, false>", 255),
    (5441, 640, 65, "gemv_reuse", None),
    (5000, 640, 64, "gemv_reuse", None),
    (6144, 640, 72, "gemv_reuse", None),
    (6145, 640, 72, "gemm_w4<", None),
    (4861, 1152, 38, "gemv_reuse", None),
    (5440, 1408, 38, "gemv_reuse_lds<", None),
    (5441, 1408, 38, "gemm_w4<", None),
    (5376, 1920, 48, "gemv_reuse_lds<", None),
    (5376, 2176, 48, "gemm_w4<", None),
    (5364, 128, 41, "gemv_reuse_lds<", None),
    (16392, 128, 64, "gemv_reuse", None),
    (18944, 128, 64, "gemv_reuse", None),
    (18945, 128, 64, "gemm_w4<", None),
    (22528, 128, 32, "gemv_reuse", None),
    (22529, 128, 32, "gemm_w4<", None),
    (16392, 128, 129, "gemm_w4<4, 1, 4, 2, false>", 130),
    (2704, 128, 81, "gemm_w4<1, 8, 1, 1, false>", 255),
    (114, 128, 2012, "gemm_w4<1, 8, 1, 1, false>", 252),
    (256, 1024, 300, "gemv_reuse", None),
    (1024, 28672, 33, "gemv_reuse_pf<", None),
    (4096, 1 << 21, 65, "gemm_w4<", None),
    (4096, (1 << 21) + 256, 65, "gemv_reuse_pfb<", None),  # beyond the 32-bit offsets
])
def test_linear_routes(lib, m, k, b, kernel, blocks):
    d = _abi.describe_linear(lib, m, k, b)
    assert d["kernel"].startswith("void dk::" + kernel), d
    assert d["launches"] == 1 and (blocks is None or d["grid"] == [blocks, 1, 1]), d
    if "gemm_w4" not in kernel:
        assert d == _abi.describe(lib, m, k, b, reuse_weights=1)


@pytest.mark.parametrize("i,h,b,kernel", [
    (11008, 4096, 16, "gate_up_silu_tiles_lds"),
    (11008, 4096, 17, "gemm_w4<1, 8, 1, 2, true>"),
    (2048, 4096, 64, "gate_up_silu_tiles_lds"),  # 128 x 4 tiles
    (2048, 4096, 65, "gemm_w4<1, 8, 1, 2, true>"),
    (11008, 4096, 1000, "gemm_w4<4, 1, 4, 2, true>"),
    (512, 4096, 20, "gate_up_silu_"),
    # Short rows: up to 1024 weights over 1536 tiles of 16 x 16, or over 768 in
    # one round of 32 x 32; up to 2048 over 144 or 176 of 32 x 32; one group
    # over 216 of 64 x 64 or 640 of 32 x 32.
    (4100, 256, 17, "gate_up_silu_tiles_lds"),
    (4096, 1024, 96, "gate_up_silu_tiles_lds"),
    (4097, 1024, 96, "gemm_w4"),
    (4096, 512, 64, "gemm_w4"),
    (3072, 512, 64, "gate_up_silu_tiles_lds"),
    (4128, 512, 64, "gate_up_silu_tiles_lds"),
    (2816, 1152, 64, "gate_up_silu_tiles_lds"),
    (2817, 1152, 64, "gemm_w4"),
    (2304, 2048, 64, "gate_up_silu_tiles_lds"),
    (2305, 2048, 64, "gemm_w4"),
    (2304, 2176, 64, "gemm_w4"),
    (16384, 512, 32, "gemm_w4"),
    (16385, 512, 32, "gate_up_silu_tiles_lds"),
    (24577, 512, 32, "gemm_w4"),
    (16385, 384, 32, "gemm_w4"),
    (18433, 2048, 32, "gemm_w4"),
    (13824, 128, 32, "gate_up_silu_tiles_lds"),
    (13825, 128, 32, "gemm_w4<4, 1, 4, 2, true>"),
    (10240, 128, 64, "gate_up_silu_tiles_lds"),
    (10241, 128, 64, "gemm_w4<4, 1, 4, 2, true>"),
])
def test_gate_up_routes(lib, i, h, b, kernel):
    assert _abi.describe_gate_up(lib, i, h, b)["kernel"].startswith("void dk::" + kernel)


def test_up_to_16_batch_rows_linear_is_gemv(lib):
    rng = np.random.default_rng(3)
    for _ in range(200):
        m, k, b = int(rng.integers(1, 30000)), 128 * int(rng.integers(1, 230)), int(rng.integers(1, 17))
        assert _abi.describe_linear(lib, m, k, b) == _abi.describe(lib, m, k, b, reuse_weights=1)


def _weight(m: int, k: int, seed: int):
    """Arbitrary words (every nibble, -8 among them) and scales, some zero."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    packed = torch.randint(-2**31, 2**31, (m, k // 8), device="cuda", generator=g,
                           dtype=torch.int64).to(torch.int32)
    scales = (torch.rand(m, k // 128, device="cuda", generator=g) * 0.01).half()
    scales[::7] = 0
    return packed, scales


def _x(b: int, k: int, seed: int):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(b, k, device="cuda", generator=g).half()


def _dense(packed, scales):
    m, words = packed.shape
    q = torch.stack([(packed << (28 - 4 * n)) >> 28 for n in range(8)], dim=2).double()
    return (q.view(m, -1, 128) * scales.double()[:, :, None]).view(m, words * 8)


def _check(y: torch.Tensor, ref: torch.Tensor, label: str):
    ref = ref.cpu().numpy()
    err = np.abs(y.double().cpu().numpy() - ref)
    assert (err <= 0.5 * oracle.fp16_ulp(ref) + 1e-3).all(), f"{label}: {err.max()}"


LINEAR = [
    ((4095, 384, 33), "<1, 8, 1, 1,"), ((8191, 4224, 31), "<1, 8, 1, 1,"), ((513, 128, 250), "<1, 8, 1, 1,"),
    ((5000, 4224, 24), "<1, 8, 1, 1,"), ((4095, 2176, 33), "<1, 8, 1, 1,"),
    ((2049, 640, 128), "<1, 8, 2, 1,"), ((4090, 4224, 65), "<1, 8, 2, 1,"),
    ((8193, 1280, 17), "<1, 8, 1, 2,"), ((5000, 1152, 80), "<1, 8, 1, 2,"), ((8193, 640, 49), "<1, 8, 2, 2,"),
    ((5000, 4224, 129), "<1, 8, 2, 2,"),
    ((16385, 640, 64), "<2, 4, 2, 2,"), ((21505, 640, 17), "<2, 4, 2, 2,"),
    ((4100, 4224, 300), "<2, 4, 2, 2,"),
    ((2040, 11136, 640), "<1, 8, 4, 2,"), ((11008, 4224, 129), "<2, 4, 4, 2,"),
    ((5000, 4224, 520), "<2, 4, 4, 2,"),
    ((8321, 384, 65), "<1, 4, 4, 2,"), ((2049, 640, 1030), "<1, 4, 4, 2,"),
    ((16392, 128, 129), "<4, 1, 4, 2,"), ((2053, 128, 1000), "<4, 1, 4, 2,"),
]


@pytest.mark.gpu
@pytest.mark.parametrize("shape,kernel", LINEAR)
def test_linear_many_batch_rows(lib, shape, kernel):
    from decode_kernel import _cuda, w4a16_linear

    m, k, b = shape
    assert "gemm_w4" + kernel in _abi.describe_linear(lib, m, k, b)["kernel"]
    print(f"[gemm] M={m} K={k} B={b} {kernel}", flush=True)
    packed, scales = _weight(m, k, seed=m + b)
    x = _x(b, k, seed=b)
    y = w4a16_linear(x, packed, scales)
    assert _cuda.last_kernel_stamp() == 15
    _check(y, x.double() @ _dense(packed, scales).T, f"{m}x{k} B={b}")
    assert torch.equal(w4a16_linear(x, packed, scales), y)
    # The matrix cores' fp32 sums are not rounded alike for both signs in the
    # last bit (2-7 of 12.6 million outputs, on the 16-row tiles as well), so a
    # sum next to the middle of two fp16 values may fall either way.
    yn = w4a16_linear(-x, packed, scales)
    off = (yn != -y).nonzero(as_tuple=True)
    assert off[0].numel() <= 2 + 1e-5 * y.numel()
    step = torch.from_numpy(oracle.fp16_ulp(y[off].double().cpu().numpy())).to(y.device)
    assert ((yn[off].double() + y[off].double()).abs() <= step).all()
    # Batch rows do not mix, whatever one of them holds.
    bad = x.clone()
    bad[b // 2] = float("nan")
    bad[b // 2, ::3] = float("inf")
    yb = w4a16_linear(bad, packed, scales)
    keep = torch.arange(b, device="cuda") != b // 2
    assert torch.equal(yb[keep], y[keep])
    # One-hot activations select single scaled weights bit for bit.
    e = torch.zeros_like(x)
    cols = [(37 * i + 5) % k for i in range(b)]
    e[torch.arange(b), torch.tensor(cols)] = 1.0
    assert torch.equal(w4a16_linear(e, packed, scales), _dense(packed, scales)[:, cols].T.half())


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(8200, 1280, 17), (4096, 1536, 100), (8200, 1280, 70)])
def test_linear_least_alignment(lib, shape):
    """Scales and y on 2 bytes: 2-byte stores, the same bits, nothing past y."""
    m, k, b = shape
    packed, scales = _weight(m, k, seed=m)
    x = _x(b, k, seed=b)
    stream = torch.cuda.current_stream().cuda_stream

    def call(sp, yp):
        _abi.check(lib, lib.dk_w4a16_linear(packed.data_ptr(), sp, x.data_ptr(), yp, m, k, b, None,
                                            0, stream))

    y = torch.empty(b * m, dtype=torch.float16, device="cuda")
    call(scales.data_ptr(), y.data_ptr())
    s2 = torch.empty(scales.numel() + 1, dtype=torch.float16, device="cuda")
    s2[1:] = scales.reshape(-1)
    y2 = torch.full((b * m + 2,), 7.0, dtype=torch.float16, device="cuda")
    call(s2[1:].data_ptr(), y2[1:].data_ptr())
    assert y2[1:].data_ptr() % 4 == 2
    assert torch.equal(y2[1:-1], y) and y2[0] == 7 and y2[-1] == 7
    _check(y.view(b, m), x.double() @ _dense(packed, scales).T, f"{m}x{k} B={b}")


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(4161, 384, 17), (5000, 4224, 24), (8200, 1280, 70),
                                   (4096, 4096, 100)])
def test_linear_agrees_with_gemv(lib, shape):
    """dk_w4a16_gemv keeps the 16-row tiles: the same bits where dk_w4a16_linear
    does too, else both within their bound (fp32 sums in another order)."""
    m, k, b = shape
    packed, scales = _weight(m, k, seed=m + b)
    x = _x(b, k, seed=b)
    cfg = _abi.default_config(lib, reuse_weights=1)
    y = torch.empty(2, b, m, dtype=torch.float16, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    args = (packed.data_ptr(), scales.data_ptr(), x.data_ptr())
    _abi.check(lib, lib.dk_w4a16_gemv(*args, y[0].data_ptr(), m, k, b, ctypes.byref(cfg), None, 0,
                                      stream))
    _abi.check(lib, lib.dk_w4a16_linear(*args, y[1].data_ptr(), m, k, b, None, 0, stream))
    if _abi.describe_linear(lib, m, k, b) == _abi.describe(lib, m, k, b, reuse_weights=1):
        assert torch.equal(y[0], y[1])
    ref = x.double() @ _dense(packed, scales).T
    for out, entry in zip(y, ("gemv", "linear")):
        _check(out, ref, f"{entry} {m}x{k} B={b}")


GATE_UP = [
    ((5633, 1152, 17), "<1, 8, 1, 2,"), ((1000, 384, 250), "<1, 8, 1, 2,"), ((4100, 1152, 33), "<1, 8, 2, 2,"),
    ((2049, 1152, 128), "<1, 8, 2, 2,"), ((8193, 1152, 17), "<2, 4, 2, 2,"), ((8193, 384, 33), "<2, 4, 2, 2,"),
    ((8193, 4224, 65), "<2, 4, 4, 2,"), ((4100, 256, 97), "<1, 4, 4, 2,"), ((3000, 384, 250), "<1, 4, 4, 2,"),
    ((13825, 128, 17), "<4, 1, 4, 2,"), ((1000, 128, 2100), "<4, 1, 4, 2,"), ((2049, 128, 449), "<4, 1, 4, 2,"),
    ((5888, 13184, 70), "<1, 8, 4, 2,"),
]


@pytest.mark.gpu
@pytest.mark.parametrize("shape,kernel", GATE_UP)
def test_gate_up_many_batch_rows(lib, shape, kernel):
    from decode_kernel import _cuda, gate_up_silu

    i, h, b = shape
    assert "gemm_w4" + kernel in _abi.describe_gate_up(lib, i, h, b)["kernel"]
    print(f"[gemm] I={i} H={h} B={b} {kernel}", flush=True)
    gate, up = _weight(i, h, seed=i), _weight(i, h, seed=i + 1)
    x = _x(b, h, seed=b) * 0.5
    out = gate_up_silu(x, *gate, *up)
    assert _cuda.last_kernel_stamp() == 20
    g, u = (x.double() @ _dense(*w).T for w in (gate, up))
    # The fp32 sums of g and u meet in a product: 1e-3 of each, times the other.
    ref = (torch.nn.functional.silu(g) * u).cpu().numpy()
    slack = 1e-3 * (1 + g.abs() + u.abs()).cpu().numpy() * 0.1
    err = np.abs(out.double().cpu().numpy() - ref)
    assert (err <= 0.5 * oracle.fp16_ulp(ref) + 1e-3 + slack).all(), err.max()
    assert torch.equal(gate_up_silu(x, *gate, *up), out)
    assert torch.isfinite(out).all()


@pytest.mark.gpu
def test_graph_replays_match_eager(lib):
    """Captured with the eager work of other inputs between the replays."""
    from decode_kernel import gate_up_silu, w4a16_linear

    (p1, s1), (p2, s2), (p3, s3) = (_weight(4352, 2048, 1), _weight(4352, 2048, 2), _weight(2048, 4352, 3))
    x, other = _x(260, 2048, 4), _x(260, 2048, 5)
    eager = w4a16_linear(gate_up_silu(x, p1, s1, p2, s2), p3, s3)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = w4a16_linear(gate_up_silu(x, p1, s1, p2, s2), p3, s3)
    for _ in range(4):
        y.zero_()
        graph.replay()
        between = w4a16_linear(gate_up_silu(other, p1, s1, p2, s2), p3, s3)
        torch.cuda.synchronize()
        assert torch.equal(y, eager) and not torch.equal(between, eager)
