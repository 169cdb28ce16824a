"""Expert weights stacked, cast and tiled in one pass, the backward product on
tiles, and rows gathered with a cast: each equal, bit for bit, to the separate
torch operations (or the plain layout) it stands for."""

import pytest
import torch

import quantaweave_amd as qa
from quantaweave_amd import _hip, _lib, moe

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.bfloat16, torch.float16]


@pytest.mark.parametrize("src", DTYPES)
@pytest.mark.parametrize("dst", DTYPES)
@pytest.mark.parametrize("E,rows,cols", [(1, 64, 64), (3, 128, 192), (70, 64, 64), (2, 100, 520), (2, 5, 8), (3, 7, 12)])
def test_packed_weights_equal_stack_and_cast(src, dst, E, rows, cols):
    torch.manual_seed(E + rows + cols)
    ws = [(torch.randn(rows, cols, device="cuda") * 0.05).to(src) for _ in range(E)]
    want = torch.stack(ws).to(dst)
    assert torch.equal(moe.pack_weights(ws, dst, False), want)
    if dst in _hip.HALF and rows % 64 == 0 and cols % 64 == 0:
        assert torch.equal(moe.pack_weights(ws, dst, True), moe.tile_bf16(want))


def test_packing_takes_views_and_strides():
    base = torch.randn(2 * 64 * 64 + 1, device="cuda")
    odd = [base[1 + i * 4096:1 + (i + 1) * 4096].view(64, 64) for i in range(2)]      # 4-byte aligned
    turned = [torch.randn(64, 128, device="cuda").t() for _ in range(2)]               # not contiguous
    for ws in (odd, turned):
        assert torch.equal(moe.pack_weights(ws, torch.float32, False), torch.stack(ws))
        assert torch.equal(moe.pack_weights(ws, torch.bfloat16, True), moe.tile_bf16(torch.stack(ws).bfloat16()))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("N,K,counts", [(64, 64, [3, 0, 70]), (128, 320, [1, 129, 0, 64]), (192, 128, [200])])
def test_grad_x_from_tiles_equals_plain(dtype, N, K, counts):
    torch.manual_seed(N + K)
    E, R = len(counts), sum(counts)
    w = (torch.randn(E, N, K, device="cuda") * 0.05).to(dtype)
    gy, x = torch.randn(R, N, device="cuda").to(dtype), torch.randn(R, K, device="cuda").to(dtype)
    offsets = torch.tensor([0, *torch.tensor(counts).cumsum(0).tolist()], dtype=torch.int32, device="cuda")
    nb = _lib.load().qw_grouped_matmul_backward_workspace_bytes(E, N, K, R, _hip.act_code(w, "w"))
    ws = _hip.workspace(nb, w.device)
    got = []
    for fmt, weights in ((_hip.HALF[dtype][0], w), (_hip.HALF[dtype][1], moe.tile_bf16(w))):
        for accumulate in (0, 1):
            gx = torch.ones(R, K, dtype=dtype, device="cuda")
            print(f"case {N}x{K} {counts} {dtype} format {fmt} accumulate {accumulate}", flush=True)
            _lib.call("qw_grouped_matmul_backward_fmt", _hip.ptr(gy), _hip.ptr(x), _hip.ptr(weights),
                      _hip.HALF[dtype][0], fmt, E, N, K, _hip.ptr(offsets), R, 0, _hip.ptr(gx), accumulate, None,
                      _hip.HALF[dtype][0], _hip.ptr(ws), nb, _hip.stream(w.device))
            got.append(gx)
    assert torch.equal(got[0], got[2]) and torch.equal(got[1], got[3])


@pytest.mark.parametrize("src", DTYPES)
@pytest.mark.parametrize("dst", DTYPES)
@pytest.mark.parametrize("D", [8, 33, 2056])
def test_gathered_rows_with_a_cast(src, dst, D):
    x = torch.randn(9, D, device="cuda").to(src)
    slots = torch.tensor([8, 0, 3, 3, 7, 5], dtype=torch.int32, device="cuda")
    totals = torch.tensor([5, 0], dtype=torch.int32, device="cuda")
    out = torch.full((6, D), 2.0, dtype=dst, device="cuda")
    _lib.call("qw_moe_permute_cast", _hip.ptr(x), _hip.act_code(x, "x"), D, _hip.ptr(slots), _hip.ptr(totals), 6,
              _hip.ptr(out), _hip.act_code(out, "out"), _hip.stream(x.device))
    assert torch.equal(out[:5], x.to(dst)[slots[:5].long()])
    assert (out[5] == 2.0).all()  # past the kept rows: untouched


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_pack_does_not_hold_the_experts_weights(dtype):
    """A layer and a decode step keep their stacks, not the storage the stacks were
    made from: moving the module frees it."""
    config = qa.QuantaWeaveConfig(vocab_size=2, hidden_size=256, layers=1, ffn_size=512, num_experts=16, top_k=2,
                                  attention_heads=1, max_sequence_length=64)
    layer = qa.TopKMoE(config).to("cuda", dtype)
    with torch.no_grad():
        layer(torch.randn(1, 8, 256, device="cuda", dtype=dtype))
    step = qa.MoEDecodeStep(layer, precision="bf16")
    weights = sum(p.numel() * p.element_size() for p in layer.experts.parameters())
    x = torch.randn(1, 256, device="cuda")
    want = step.step(x).clone()
    before = torch.cuda.memory_allocated()
    layer.cpu()
    assert before - torch.cuda.memory_allocated() >= weights
    assert torch.equal(step.step(x), want)


def layer_of(ffn, seed=0):
    config = qa.QuantaWeaveConfig(vocab_size=2, hidden_size=64, layers=1, ffn_size=ffn, num_experts=4, top_k=2,
                                  attention_heads=1, max_sequence_length=64)
    torch.manual_seed(seed)
    return qa.TopKMoE(config).cuda()


@torch.no_grad()
def test_calls_follow_the_weights_width():
    """Experts whose matrices were replaced by narrower ones (pruned hidden units,
    nn.Linear's attributes as they were) are evaluated at the width of the matrices,
    also after a call at the old width."""
    layer, narrow = layer_of(128), layer_of(64, seed=1)
    x = torch.randn(1, 32, 64, device="cuda")
    layer(x)
    layer.router.weight.copy_(narrow.router.weight)
    for mine, other in zip(layer.experts, narrow.experts):
        for name in ("gate", "up", "down"):
            getattr(mine, name).weight = torch.nn.Parameter(getattr(other, name).weight.clone())
    assert torch.equal(layer(x)[0], narrow(x)[0])
    counts = [10, 0, 21, 1]
    assert torch.equal(qa.moe_kernels.grouped_swiglu(x[0], layer.experts, counts),
                       qa.moe_kernels.grouped_swiglu(x[0], narrow.experts, counts))


@torch.no_grad()
def test_a_layer_pickled_by_an_earlier_release_runs():
    """Whole-module pickles carry the module's cache of workspace sizes; entries of
    the earlier form (four sizes per shape) are left alone."""
    layer = layer_of(64)
    x = torch.randn(1, 32, 64, device="cuda")
    want = layer(x)[0]
    layer.__dict__["_qw_sizes"] = {(32, 64, 4, 2, _lib.QW_F32): (64, 256, 256, 256)}
    assert torch.equal(layer(x)[0], want)
