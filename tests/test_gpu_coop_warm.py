"""The keys that a layer touches for the next one: a launch with the build inside and workgroups there for the build alone touches as much
as the dot's launch of two does."""
import pytest
import torch

from test_gpu_parity import ops  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Q,d,R", [(33, 768, 768), (64, 1536, 1000), (200, 704, 300)])  # chunk scales; bands of tiles; row scales
def test_all_lines_are_touched(ops, Q, d, R):
    """512 MiB, which no cache holds, make up the launch's time; the same workgroups touch them in both forms, so the times differ only if a
    part is left out (the workgroups without a tile are four of five here)."""
    from bsipytorch_amd import _lib

    L = _lib.lib
    gen = torch.Generator(device="cuda").manual_seed(Q)
    keys = ops.build_bsi_keys_cuda(torch.randn(R, d, generator=gen, device="cuda") * 0.02, 2, 0.5)[0]
    assert L.bsi_hip_linear_coop_serves(Q, d, R, 2, 7, _lib.LAYOUT_INT8, 6) == 1
    x = torch.randn(Q, d, generator=gen, device="cuda")
    area = torch.zeros(int(L.bsi_hip_linear_coop_bytes()), dtype=torch.uint8, device="cuda")
    ws = torch.empty(int(L.bsi_hip_linear_workspace_bytes(Q, d, 7)), dtype=torch.uint8, device="cuda")
    warm = torch.zeros(512 << 20, dtype=torch.uint8, device="cuda")
    out = torch.empty(Q, R, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    number = [0]

    def one():
        number[0] += 1
        return L.bsi_hip_linear_coop_out(x.data_ptr(), _lib.DTYPE_F32, Q, d, 2, 7, number[0], area.data_ptr(), keys.ints8.data_ptr(), _lib.LAYOUT_INT8,
                                         keys.slice_weights.data_ptr(), 6, R, 1e-4, R, None, out.data_ptr(), _lib.DTYPE_F32, warm.data_ptr(), warm.numel(), stream)

    def two():
        return L.bsi_hip_linear_out(x.data_ptr(), _lib.DTYPE_F32, Q, d, 2, 7, 1, ws.data_ptr(), ws.numel(), keys.ints8.data_ptr(), _lib.LAYOUT_INT8,
                                    keys.slice_weights.data_ptr(), 6, R, 1e-4, R, None, out.data_ptr(), _lib.DTYPE_F32, _lib.CORE_AUTO, warm.data_ptr(),
                                    warm.numel(), stream)

    times = {one: [], two: []}
    for _ in range(4):
        for call in (one, two):
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            begin.record()
            assert call() == 0
            end.record()
            end.synchronize()
            times[call].append(begin.elapsed_time(end))
    assert min(times[one]) > 0.6 * min(times[two]), times
