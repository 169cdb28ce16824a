"""The 16-bit backward products on operands as they lie (256-column tiles): one
product and a pair, at edges of the tiles, slices and row counts, against the
64-bit product of the same 16-bit values."""

import pytest
import torch

from quantaweave_amd import _hip, _lib, moe

pytestmark = pytest.mark.gpu

# rows per expert: none, one, around a 64-row slice, around both tile heights
UNEVEN = [0, 1, 63, 64, 65, 129, 0, 257]
SIZES = [(128, 192), (64, 264), (96, 200), (320, 576), (1408, 512)]
# the last three: enough tiles for the 256-row ones
CASES = [(c, *nk) for c in (UNEVEN, [700], [5] * 40) for nk in SIZES] + [
    (UNEVEN * 10, 128, 1024), (UNEVEN * 10, 64, 1000), (UNEVEN * 4 + [1], 576, 2816)]


def check(got, want, bound, dtype):
    """Rounding of the stored type, and one 2^-24 per addition of fp32 sums."""
    unit = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -23}[dtype]
    tiny = 2.0 ** -24 if dtype == torch.float16 else 0.0  # subnormal fp16 results
    assert ((got.double() - want).abs() <= want.abs() * unit + bound + tiny).all()


def products(gys, x, ws, starts, counts):
    """grad_x (sum over the products) and each grad_w in 64 bits, with the bound on the fp32 sums."""
    R, K, N = x.size(0), x.size(1), gys[0].size(1)
    f64 = dict(dtype=torch.float64, device="cuda")
    dx, dx_abs = torch.zeros(R, K, **f64), torch.zeros(R, K, **f64)
    dws, dw_abs = [], []
    for gy, w in zip(gys, ws):
        dw, da = torch.zeros(len(counts), N, K, **f64), torch.zeros(len(counts), N, K, **f64)
        for e, c in enumerate(counts):
            at = slice(starts[e], starts[e] + c)
            g, xe, we = gy[at].double(), x[at].double(), w[e].double()
            dx[at] += g @ we
            dx_abs[at] += g.abs() @ we.abs()
            dw[e], da[e] = g.t().contiguous() @ xe, g.abs().t().contiguous() @ xe.abs()
        dws.append(dw)
        dw_abs.append(da * (max(counts) + 64) * 2.0 ** -24)
    return dx, dx_abs * (len(gys) * N) * 2.0 ** -24, dws, dw_abs


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("counts,N,K", CASES, ids=lambda v: str(len(v)) if isinstance(v, list) else str(v))
def test_backward_on_operands_as_they_lie(dtype, counts, N, K):
    torch.manual_seed(N + K + len(counts))
    E, R, code = len(counts), sum(counts), _hip.HALF[dtype][0]
    starts = [0, *torch.tensor(counts).cumsum(0).tolist()]
    offsets = torch.tensor(starts, dtype=torch.int32, device="cuda")
    x = torch.randn(R, K, device="cuda").to(dtype)
    gys = [torch.randn(R, N, device="cuda").to(dtype) for _ in range(2)]
    ws = [(torch.randn(E, N, K, device="cuda") * 0.05).to(dtype) for _ in range(2)]
    nb = _lib.load().qw_grouped_matmul_backward_workspace_bytes(E, N, K, R, code)
    space = _hip.workspace(nb, x.device)
    one, two = products(gys[:1], x, ws[:1], starts, counts), products(gys, x, ws, starts, counts)
    formats = [(code, ws)]
    if N % 64 == 0 and K % 64 == 0:
        formats.append((_hip.HALF[dtype][1], [moe.tile_bf16(w) for w in ws]))
    for out in (dtype, torch.float32):
        for fmt, weights in formats:
            print(f"case {N}x{K} {dtype} rows {R} out {out} format {fmt}", flush=True)
            out_code = _hip.act_code(torch.empty(0, dtype=out), "out")
            gx = torch.full((R, K), 3.0, dtype=dtype, device="cuda")
            gw = torch.full((3, E, N, K), 3.0, dtype=out, device="cuda")
            tail = (E, N, K, _hip.ptr(offsets), R, 0, _hip.ptr(gx))
            end = (out_code, _hip.ptr(space), nb, _hip.stream(x.device))
            _lib.call("qw_grouped_matmul_backward_fmt", _hip.ptr(gys[0]), _hip.ptr(x), _hip.ptr(weights[0]), code, fmt,
                      *tail, 0, _hip.ptr(gw[0]), *end)
            check(gx, one[0], one[1], dtype)
            check(gw[0], one[2][0], one[3][0], out)
            gx.fill_(3.0)
            _lib.call("qw_grouped_matmul_backward_pair", _hip.ptr(gys[0]), _hip.ptr(gys[1]), _hip.ptr(x),
                      _hip.ptr(weights[0]), _hip.ptr(weights[1]), code, fmt, *tail, _hip.ptr(gw[1]), _hip.ptr(gw[2]),
                      *end)
            # as two products the first is rounded before the second is added
            check(gx, two[0], two[1] + 2.0 ** -8 * one[0].abs(), dtype)
            for i in range(2):
                check(gw[1 + i], two[2][i], two[3][i], out)
            assert torch.equal(gw[0], gw[1])
            for e, c in enumerate(counts):
                assert c or not gw[:, e].any()  # exactly zero without rows


def test_rows_past_an_expert_stay_out():
    """Infinities and NaN in the rows after an expert's last do not reach its gradient."""
    x, gy = torch.randn(128, 256, device="cuda").bfloat16(), torch.randn(128, 128, device="cuda").bfloat16()
    x[70:], gy[70:] = float("inf"), float("nan")
    w = torch.zeros(2, 128, 256, device="cuda").bfloat16()
    offsets = torch.tensor([0, 70, 128], dtype=torch.int32, device="cuda")
    gw = torch.empty(2, 128, 256, device="cuda")
    code = _hip.HALF[torch.bfloat16][0]
    _lib.call("qw_grouped_matmul_backward", _hip.ptr(gy), _hip.ptr(x), _hip.ptr(w), code, 2, 128, 256,
              _hip.ptr(offsets), 128, 0, None, 0, _hip.ptr(gw), _lib.QW_F32, None, 0, _hip.stream(x.device))
    g = gy[:70].double().t().contiguous()
    check(gw[0], g @ x[:70].double(), (g.abs() @ x[:70].double().abs()) * 134 * 2.0 ** -24, torch.float32)


@pytest.mark.parametrize("counts,N,K", [(UNEVEN, 64, 64), (UNEVEN, 68, 132), (UNEVEN, 4, 8), ([700], 100, 64),
                                        ([31, 32, 33], 128, 68)])
def test_fp32_backward_on_operands_as_they_lie(counts, N, K):
    """Slices of 32 and tiles of 64 with remainders in every direction, rows past an expert not finite."""
    torch.manual_seed(N + K)
    counts, E = [*counts, 9], len(counts) + 1
    starts, R = [0, *torch.tensor(counts).cumsum(0).tolist()], sum(counts)
    offsets = torch.tensor(starts, dtype=torch.int32, device="cuda")
    x, gy = torch.randn(R, K, device="cuda"), torch.randn(R, N, device="cuda")
    x[-9:], gy[-9:] = float("inf"), float("nan")
    w = torch.randn(E, N, K, device="cuda") * 0.05
    gx, gw = torch.ones(R, K, device="cuda"), torch.full((E, N, K), 3.0, device="cuda")
    print(f"case fp32 {N}x{K} rows {R}", flush=True)
    for accumulate in (0, 1):
        _lib.call("qw_grouped_matmul_backward", _hip.ptr(gy), _hip.ptr(x), _hip.ptr(w), _lib.QW_F32, E, N, K,
                  _hip.ptr(offsets), R, 0, _hip.ptr(gx), accumulate, _hip.ptr(gw), _lib.QW_F32, None, 0,
                  _hip.stream(x.device))
        live = R - 9
        dx, bound, dws, bounds = products([gy[:live]], x[:live], [w], starts, counts[:-1])
        check(gx[:live], dx * (1 + accumulate), bound * (1 + accumulate), torch.float32)
        check(gw[:-1], dws[0], bounds[0], torch.float32)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("E,N,K,rows", [(8, 128, 256, 1600), (3, 64, 192, 300), (2, 192, 264, 500)])
def test_input_gradient_without_workspace(dtype, E, N, K, rows):
    """At sizes where the 128 x 128 tiles are the preferred kernel, which need a
    workspace: without one grad_x still runs on the 256-column tiles (the bits of a
    pair whose second product is zero), plain weights and tiles alike."""
    torch.manual_seed(N + K)
    code, tile_code = _hip.HALF[dtype]
    counts = [rows // E] * (E - 1) + [rows - rows // E * (E - 1)]
    starts = [0, *torch.tensor(counts).cumsum(0).tolist()]
    offsets = torch.tensor(starts, dtype=torch.int32, device="cuda")
    gy = torch.randn(rows, N, device="cuda").to(dtype)
    w = (torch.randn(E, N, K, device="cuda") * 0.05).to(dtype)
    x = torch.empty(rows, K, dtype=dtype, device="cuda")  # read by the weight gradients only
    want, bound, _, _ = products([gy], x.zero_(), [w], starts, counts)
    zero = torch.zeros_like(gy)
    formats = [(code, w)]
    if N % 64 == 0 and K % 64 == 0:
        formats.append((tile_code, moe.tile_bf16(w)))
    for fmt, weights in formats:
        print(f"case {N}x{K} {dtype} rows {rows} format {fmt}", flush=True)
        gx, pair = (torch.full((rows, K), 3.0, dtype=dtype, device="cuda") for _ in range(2))
        tail = (E, N, K, _hip.ptr(offsets), rows, 0)
        _lib.call("qw_grouped_matmul_backward_fmt", _hip.ptr(gy), None, _hip.ptr(weights), code, fmt, *tail,
                  _hip.ptr(gx), 0, None, code, None, 0, _hip.stream(gy.device))
        _lib.call("qw_grouped_matmul_backward_pair", _hip.ptr(gy), _hip.ptr(zero), None, _hip.ptr(weights),
                  _hip.ptr(weights), code, fmt, *tail, _hip.ptr(pair), None, None, code, None, 0,
                  _hip.stream(gy.device))
        check(gx, want, bound, dtype)
        assert torch.equal(gx, pair)
