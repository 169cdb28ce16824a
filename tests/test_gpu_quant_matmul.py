"""One quantised matrix, and grouped quantised rows, on the matrix cores: the
edges of row chunks, slices and column tiles, and every quantised kernel that
the row count selects, against a float64 product of the stored codes."""

import pytest
import torch

import quantaweave_amd as qa
from quantaweave_amd import _hip, _lib

pytestmark = pytest.mark.gpu

ULP = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}  # of a value in [1, 2)


def check(got, x, deq):
    """|error| of each output: half an ulp of the output, half an ulp of every
    weight (rounded to the activation type) times |x|, and the fp32 sum's
    roundings."""
    xd = x.double()
    ref = xd @ deq.double().t()
    mass = xd.abs() @ deq.double().abs().t()
    half_ulp = ULP[x.dtype] / 2
    bound = half_ulp * ref.abs() * 1.01 + mass * (half_ulp + x.shape[1] * 2.0 ** -23) + 1e-6
    bad = ((got.double() - ref).abs() > bound).sum().item()
    assert bad == 0, f"{bad} of {ref.numel()} outputs outside the rounding bound"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("bits,group,cols,out", [
    (8, None, 64, 7), (8, None, 320, 300), (8, 64, 192, 256), (8, None, 2112, 513),
    (4, None, 64, 33), (4, None, 128, 256), (4, None, 192, 300), (4, 64, 384, 260), (4, 128, 2048, 1024),
    (4, None, 4224, 64), (8, None, 1000, 31), (4, 16, 128, 40),
])
def test_quantized_matrix_over_row_counts(bits, group, cols, out, dtype):
    torch.manual_seed(cols + out + bits)
    lin = torch.nn.Linear(cols, out, bias=False).cuda()
    q = qa.QuantizedLinear.from_linear(lin, bits, group)
    deq = q.dequantize()
    for rows in (1, 4, 5, 20, 21, 32, 33, 48, 49, 64, 65, 96, 97, 130, 200):
        print(f"case int{bits} group {group} {cols}x{out} rows {rows} {dtype}", flush=True)
        x = torch.randn(rows, cols, device="cuda").to(dtype)
        with torch.no_grad():
            check(q(x), x, deq)


@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("counts", [[200, 0, 33], [97, 1, 0, 16, 15, 96, 64, 65, 31, 0, 130]])
def test_grouped_quantised_rows(counts, bits):
    """Fewer experts than XCDs (tiles dealt by column) and more (by expert),
    with empty experts and chunks found on the device (no row bound given)."""
    torch.manual_seed(len(counts))
    E, N, K = len(counts), 320, 192
    qs = [qa.QuantizedLinear.from_linear(torch.nn.Linear(K, N, bias=False).cuda(), bits) for _ in counts]
    w, s = torch.stack([q.qweight for q in qs]), torch.stack([q.scales for q in qs])
    x = torch.randn(sum(counts), K, device="cuda").bfloat16()
    offsets = torch.tensor([0, *torch.tensor(counts).cumsum(0).tolist()], dtype=torch.int32, device="cuda")
    out = torch.full((sum(counts), N), float("nan"), dtype=torch.bfloat16, device="cuda")
    print(f"case grouped int{bits} {counts}", flush=True)
    _lib.call("qw_grouped_matmul", _hip.ptr(x), _lib.QW_BF16, _hip.ptr(w), qs[0].w_format, _hip.ptr(s),
              qs[0].group_size, E, N, K, _hip.ptr(offsets), x.shape[0], 0, _hip.ptr(out), _hip.stream(x.device))
    first = 0
    for n, q in zip(counts, qs):
        check(out[first:first + n], x[first:first + n], q.dequantize())
        first += n


def test_quantized_matmul_refuses_bad_arguments():
    lib = _lib.load()
    bad = [(_lib.QW_BF16, 7, 32, 8, 64), (_lib.QW_BF16, _lib.QW_BF16, 32, 8, 64), (9, _lib.QW_I8, 32, 8, 64),
           (_lib.QW_BF16, _lib.QW_U4, 31, 8, 64), (_lib.QW_BF16, _lib.QW_I8, 0, 8, 64),
           (_lib.QW_BF16, _lib.QW_I8, 32, 0, 64)]
    for act, fmt, group, out, cols in bad:
        assert lib.qw_quantized_matmul(None, act, None, fmt, None, group, out, cols, 4, None, None) == \
            _lib.QW_ERR_INVALID
    assert lib.qw_quantized_matmul(None, _lib.QW_BF16, None, _lib.QW_I8, None, 32, 8, 64, 4, None, None) == \
        _lib.QW_ERR_INVALID and b"pointers" in lib.qw_last_error()
    assert lib.qw_quantized_matmul(None, _lib.QW_BF16, None, _lib.QW_I8, None, 32, 8, 64, 0, None, None) == 0
