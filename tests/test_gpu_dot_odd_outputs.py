"""Outputs whose rows begin anywhere, tiles past whose last query or key the output ends: every int8-image kernel writes what it writes
into aligned rows, and nothing beside them."""
import ctypes

import pytest
import torch

from test_gpu_parity import ops  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu
BITS = {torch.float32: torch.int32, torch.float16: torch.int16, torch.bfloat16: torch.int16}


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("tile", [128, 1284, 12864, 64, 6432, 256])
@pytest.mark.parametrize("Q,R,stride,offset", [(129, 257, 257, 0), (65, 95, 99, 1), (33, 64, 65, 3), (255, 130, 136, 8), (600, 4161, 4161, 0), (513, 385, 416, 2),
                                               (128, 128, 128, 0)])
def test_rows_that_begin_anywhere(ops, dtype, tile, Q, R, stride, offset):
    from bsipytorch_amd import _lib

    L, d = _lib.lib, 512
    gen = torch.Generator(device="cuda").manual_seed(Q * R)
    x = torch.randn(Q, d, generator=gen, device="cuda").to(dtype)
    bias = torch.randn(R, generator=gen, device="cuda")
    keys = ops.build_bsi_keys_cuda(torch.randn(R, d, generator=gen, device="cuda") * 0.02, 2, 0.5)[0]
    code = {torch.float32: _lib.DTYPE_F32, torch.float16: _lib.DTYPE_F16, torch.bfloat16: _lib.DTYPE_BF16}[dtype]
    ws = torch.empty(int(L.bsi_hip_linear_workspace_bytes(Q, d, 7)), dtype=torch.uint8, device="cuda")

    def run(row, first):  # rows of `row` outputs, the first of them `first` outputs into the buffer
        buf = torch.full((first + Q * row + 64,), float("nan"), dtype=dtype, device="cuda")
        rc = L.bsi_hip_linear_out(x.data_ptr(), code, Q, d, 2, 7, 1, ws.data_ptr(), ws.numel(), keys.ints8.data_ptr(), _lib.LAYOUT_INT8,
                                  keys.slice_weights.data_ptr(), 6, R, 1e-4, row, bias.data_ptr(), buf.data_ptr() + first * buf.element_size(),
                                  code, _lib.CORE_AUTO, None, 0, torch.cuda.current_stream().cuda_stream)
        assert rc == 0
        return buf

    try:
        assert L.bsi_hip_set_option(1, tile) == 0
        want = run((R + 255) // 256 * 256, 0)[: Q * ((R + 255) // 256 * 256)].view(Q, -1)[:, :R]
        buf = run(stride, offset)
    finally:
        L.bsi_hip_set_option(1, 0)
    rows = buf[offset:offset + Q * stride].view(Q, stride)
    assert torch.equal(rows[:, :R].contiguous().view(BITS[dtype]), want.contiguous().view(BITS[dtype]))
    assert not torch.isnan(want).any()
    assert torch.isnan(buf[:offset]).all() and torch.isnan(rows[:, R:]).all() and torch.isnan(buf[offset + Q * stride:]).all()


@pytest.mark.parametrize("Q,d,R,streamed", [(1281, 2048, 16384, 1), (2561, 2000, 8192, 1), (5130, 2048, 4100, 0), (5130, 2048, 4128, 1), (1279, 2048, 16384, 0),
                                            (5130, 1792, 4128, 0)])
def test_large_float32_outputs_streamed(ops, Q, d, R, streamed):
    """80 MiB of outputs and more than 1792 elements a row, rows of whole lines: the stores' kind changes, not what they write."""
    from bsipytorch_amd import _lib
    from bsipytorch_amd.linear import BSIQuantizedLinear

    tile, plan = ctypes.c_int(), ctypes.c_int()
    for dtype, want in ((_lib.DTYPE_F32, streamed), (_lib.DTYPE_BF16, 0)):
        assert _lib.lib.bsi_hip_linear_plan(Q, d, R, R, dtype, ctypes.byref(tile), ctypes.byref(plan)) == 0
        assert plan.value == want
    gen = torch.Generator(device="cuda").manual_seed(R)
    x = torch.randn(Q, d, generator=gen, device="cuda")
    dense = torch.nn.Linear(d, R, device="cuda")
    layer = BSIQuantizedLinear(dense, 2, 0.5)
    got = []
    try:
        for kind in (0, 1, 2):
            assert _lib.lib.bsi_hip_set_option(4, kind) == 0
            with torch.no_grad():
                got.append(layer(x.clone()))
    finally:
        _lib.lib.bsi_hip_set_option(4, 0)
    assert torch.equal(got[0], got[1]) and torch.equal(got[0], got[2])
