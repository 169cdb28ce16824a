"""Float experts of a few rows each: the rows per expert at which the kernels
change, and rows too long for the shorter streaming variants, against a float64
evaluation with the reference's 16-bit rounding points."""

import pytest
import torch
import torch.nn.functional as F

from quantaweave_amd import _lib
from tests import hipcall

pytestmark = pytest.mark.gpu

FMT = {torch.bfloat16: _lib.QW_BF16, torch.float16: _lib.QW_F16}


def reference(x, counts, gate, up, down):
    dtype, rows, first = x.dtype, [], 0
    for e, n in enumerate(counts):
        xe = x[first:first + n].double()
        g = (xe @ gate[e].double().t()).to(dtype)
        u = (xe @ up[e].double().t()).to(dtype)
        h = F.silu(g.double()).to(dtype).double() * u.double()
        rows.append(h.to(dtype).double() @ down[e].double().t())
        first += n
    return torch.cat(rows)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D,F_,counts", [
    (4096, 192, [1, 0, 5, 2]), (192, 4096, [3, 4, 0, 9]), (2112, 128, [1]), (2048, 128, [2, 3, 0]),
    (128, 128, [3] * 9), (128, 192, [2] * 9 + [1]), (256, 64, [15, 3, 40, 0, 1, 7, 16, 2, 0, 11]),
])
def test_few_rows_per_expert(D, F_, counts, dtype):
    torch.manual_seed(D + F_)
    E = len(counts)
    make = lambda *s: (torch.randn(*s, device="cuda") * 0.05).to(dtype)  # noqa: E731
    gate, up, down = make(E, F_, D), make(E, F_, D), make(E, D, F_)
    x = torch.randn(sum(counts), D, device="cuda").to(dtype)
    offsets = torch.tensor([0, *torch.tensor(counts).cumsum(0).tolist()], dtype=torch.int32, device="cuda")
    ref = reference(x, counts, gate, up, down)
    # 16-bit outputs of sums whose operands went through three 16-bit roundings:
    # four half ulps of the largest output
    tol = 4 * (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11)
    for path in ("auto", "stream", "mfma"):
        print(f"case {D}x{F_} {counts} {dtype} {path}", flush=True)
        y = hipcall.experts(x, offsets, FMT[dtype], gate, up, down, path=path)
        err = ((y.double() - ref).abs().max() / ref.abs().max()).item()
        assert err <= tol, (path, err)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D,F_,counts,path", [
    # widths that are no multiples of 64: no matrix-core kernel takes them
    (200, 520, [3, 2, 0, 7, 4, 1], "stream"), (200, 520, [8] * 12, "stream"), (200, 520, [15, 14, 15], "stream"),
    (520, 192, [9, 0, 5], "stream"), (192, 72, [3], "stream"), (200, 520, [16, 17], "generic"),
    # few experts stream longer than many
    (1024, 1024, [8], "stream"), (512, 1024, [3] * 8, "stream"), (512, 1024, [8] * 8, "mfma"),
    (256, 512, [2, 4, 3], "stream"), (256, 512, [12] * 8, "mfma"), (64, 128, [3] * 4, "mfma"),
])
def test_kernel_family_of_few_rows(D, F_, counts, path, dtype):
    """auto takes the family that is the faster one at the size (same bits as that
    family), and its result is right."""
    torch.manual_seed(D + F_ + len(counts))
    E = len(counts)
    make = lambda *s: (torch.randn(*s, device="cuda") * 0.05).to(dtype)  # noqa: E731
    gate, up, down = make(E, F_, D), make(E, F_, D), make(E, D, F_)
    x = torch.randn(sum(counts), D, device="cuda").to(dtype)
    offsets = torch.tensor([0, *torch.tensor(counts).cumsum(0).tolist()], dtype=torch.int32, device="cuda")
    print(f"case {D}x{F_} {counts} {dtype} {path}", flush=True)
    y = hipcall.experts(x, offsets, FMT[dtype], gate, up, down)
    assert torch.equal(y, hipcall.experts(x, offsets, FMT[dtype], gate, up, down, path=path))
    ref = reference(x, counts, gate, up, down)
    tol = 4 * (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11)  # as above
    assert ((y.double() - ref).abs().max() / ref.abs().max()).item() <= tol


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,path", [(1, "stream"), (5, "stream"), (15, "stream"), (40, "generic")])
def test_rows_that_start_off_16_bytes(rows, path, dtype):
    """Activations at an odd element of their buffer: the kernels that copy 16-byte
    pieces straight to LDS do not take them."""
    torch.manual_seed(rows)
    E, D, F_ = 9, 128, 192
    make = lambda *s: (torch.randn(*s, device="cuda") * 0.05).to(dtype)  # noqa: E731
    gate, up, down = make(E, F_, D), make(E, F_, D), make(E, D, F_)
    x = torch.randn(rows * E * D + 1, device="cuda").to(dtype)[1:].view(rows * E, D)
    assert x.data_ptr() % 16
    offsets = torch.arange(0, rows * E + 1, rows, dtype=torch.int32, device="cuda")
    print(f"case off 16 bytes, {rows} rows {dtype}", flush=True)
    y = hipcall.experts(x, offsets, FMT[dtype], gate, up, down)
    assert torch.equal(y, hipcall.experts(x.clone(), offsets, FMT[dtype], gate, up, down, path=path))
    with pytest.raises(RuntimeError, match="do not take"):
        hipcall.experts(x, offsets, FMT[dtype], gate, up, down, path="mfma")
