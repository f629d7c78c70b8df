"""Products with f16 and bf16 weights, which go in as they are: few f32 rows in 32-bit products, more as addends of the weight's own type, bf16 rows
directly, at the edges of the tiles, of K in parts and of the row counts where the kernel changes.

Bound: root mean square of the error over the results' 3e-7 for f32 sums (1e-7 is measured) and, for f16 weights, rows of two f16 addends: 2^-22 of
every element; bf16 weights take all 24 bits.  The largest tiles have no rounding addition: see _cut_off."""
import ctypes

import numpy as np
import pytest

import oracle as o
from axonml_amd import quant as q
from axonml_amd._lib import MEM_DEVICE
from axonml_amd.quant import QuantType

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _run(ctx, kind, n, k, x, bias=None, bf16=False, shift=0):
    """x on the device, `shift` elements behind a 16-byte boundary; -> (result, the same in 64 bits)."""
    g = torch.Generator(device="cuda").manual_seed(n + k + len(x))
    w = (torch.randn(n, k, generator=g, device="cuda") * 0.02).to(torch.float16 if kind == "F16" else torch.bfloat16)
    torch.cuda.synchronize()
    h = ctypes.c_void_p()
    ctx.check(ctx.lib.axq_weight_upload(ctx.handle, int(QuantType[kind]), n, k, w.data_ptr(), w.numel() * 2, MEM_DEVICE, ctypes.byref(h)))
    t = x.bfloat16() if bf16 else x
    room = torch.empty(t.numel() + 64, dtype=t.dtype, device="cuda")
    room[shift:shift + t.numel()] = t.reshape(-1)
    at = room.data_ptr() + shift * t.element_size()
    y = torch.full((len(x), n), float("nan"), device="cuda")
    torch.cuda.synchronize()
    if bf16:
        ctx.check(ctx.lib.axq_gemm_bf16(ctx.handle, h, at, len(x), y.data_ptr(), MEM_DEVICE))
    else:
        ctx.check(ctx.lib.axq_gemv_f32(ctx.handle, h, at, len(x), bias.data_ptr() if bias is not None else None, y.data_ptr(), MEM_DEVICE))
    ctx.synchronize()
    ctx.lib.axq_weight_free(ctx.handle, h)
    want = t.double() @ w.double().T
    return y.double(), want if bias is None else want + bias.double()


def _check(got, want, bound):
    off = float((got - want).square().mean().sqrt() / want.square().mean().sqrt())
    assert off <= bound, f"{off:.2e}, bound {bound:.2e}"
    assert float((got - want).abs().max() / want.square().mean().sqrt()) <= 20 * bound


def _x(rows, k):
    return torch.randn(rows, k, generator=torch.Generator(device="cuda").manual_seed(rows * k), device="cuda")


@pytest.mark.parametrize("kind", ["F16", "BF16"])
@pytest.mark.parametrize("rows", [2, 15, 16, 17, 31, 32, 33, 64, 130, 300])
@pytest.mark.parametrize("n,k", [(1, 64), (17, 4160), (300, 2048), (4100, 8192), (8200, 192)])
def test_f32_rows(ctx, kind, rows, n, k):
    x, bias = _x(rows, k), torch.randn(n, device="cuda") * 0.1
    _check(*_run(ctx, kind, n, k, x, bias), 3e-7 + 2.0 ** -22)
    if n == 300:
        _check(*_run(ctx, kind, n, k, x, bias, shift=1), 3e-7 + 2.0 ** -22)  # rows that lie at no 16-byte boundary


@pytest.mark.parametrize("kind", ["F16", "BF16"])
@pytest.mark.parametrize("rows", [1, 42, 64, 65, 128, 129, 700])
@pytest.mark.parametrize("n,k", [(1, 64), (65, 4160), (515, 2048), (4100, 1600), (9001, 128)])
def test_bf16_rows(ctx, kind, rows, n, k):
    x = _x(rows, k)
    _check(*_run(ctx, kind, n, k, x, bf16=True), 3e-7)
    if n == 515:
        _check(*_run(ctx, kind, n, k, x, bf16=True, shift=4), 3e-7)


def _cut_off(k):
    """The matrix pipe adds K / 16 products to a total that it cuts off, by up to a unit in the last place of what the total has grown to: evenly
    spread, independent, and of a total that grows like a square root.  (Measured: 4.1e-7 at K = 4160, 2.6e-7 at 1600; this is 7.8e-7 and 4.9e-7.)"""
    return 2.0 ** -23 * (k / 16 / 2) ** 0.5 / 3 ** 0.5


@pytest.mark.parametrize("kind", ["F16", "BF16"])
@pytest.mark.parametrize("n,k,rows,bf16", [
    (4101, 1600, 2047, True), (4101, 4160, 2047, True), (8193, 1536, 1025, True),
    (4101, 512, 2047, False), (4100, 832, 2047, False), (8193, 1600, 1025, False),
])
def test_tiles_of_256_by_256(ctx, kind, n, k, rows, bf16):
    """More 128 x 128 outputs than two to a compute unit; f32 rows as two or three addends, one behind the other, against the same columns."""
    addends = 1 if bf16 else 2 if kind == "F16" else 3
    bias = None if bf16 else torch.randn(n, device="cuda") * 0.1
    _check(*_run(ctx, kind, n, k, _x(rows, k), bias, bf16), _cut_off(addends * k) + (0 if bf16 else 2.0 ** -22) + 1e-7)


@pytest.mark.parametrize("rows", [3, 40])
def test_weights_beyond_f16s_range(ctx, rows):
    """bf16 weights of 1e-30 and of 1e30 go in without a change of type."""
    k = 256
    x = _x(rows, k)
    g, w = _run(ctx, "BF16", 64, k, x * 1e30)
    _check(g, w, 3e-7)
    g, w = _run(ctx, "BF16", 64, k, x * 1e-30)
    _check(g, w, 3e-7)


@pytest.mark.parametrize("kind", ["F16", "BF16"])
@pytest.mark.parametrize("rows", [5, 40])
def test_rows_with_infinities_and_nan(ctx, kind, rows):
    x = _x(rows, 512)
    x[1, 7], x[2, 300], x[3, 5] = float("inf"), float("nan"), -float("inf")
    got, want = _run(ctx, kind, 96, 512, x)
    clean = [r for r in range(rows) if r not in (1, 2, 3)]
    _check(got[clean], want[clean], 3e-7 + 2.0 ** -22)
    assert not torch.isfinite(got[1:4]).any()


def test_without_room(monkeypatch):
    ctx = q.Context(0)
    x = _x(6, 4096)
    monkeypatch.setenv("AXQ_GEMM_SCRATCH_MAX", "0")
    _check(*_run(ctx, "BF16", 100, 4096, x), 3e-7)  # K whole
    _check(*_run(ctx, "BF16", 100, 4096, _x(100, 4096), bf16=True), 3e-7)
    monkeypatch.delenv("AXQ_GEMM_SCRATCH_MAX")
    _check(*_run(ctx, "BF16", 100, 4096, x), 3e-7)
    ctx.close()
