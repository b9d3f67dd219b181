"""Small layers in one launch where shares of the build belong to no workgroup: the workgroups of an XCD build different ones when their
wait runs out, so that there are fewer waits than such shares."""
import pytest
import torch

from test_gpu_parity import ops  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu

PATIENCE, SHARES = 6, 7  # BSI_OPT_COOP_PATIENCE, BSI_OPT_COOP_SHARES


@pytest.mark.parametrize("Q,d,R,owned,most", [(33, 768, 768, 13, 32), (100, 512, 512, 25, 32), (16, 1024, 512, 16, 32),  # chunk scales, both kernels
                                              (5, 300, 64, 1, 5), (64, 320, 320, 8, 32)])  # row scales: a copy has one workgroup, and eight
def test_waits_that_run_out(ops, Q, d, R, owned, most):
    from bsipytorch_amd import _lib

    L = _lib.lib
    gen = torch.Generator(device="cuda").manual_seed(Q)
    keys = ops.build_bsi_keys_cuda(torch.randn(R, d, generator=gen, device="cuda") * 0.02, 2, 0.5)[0]
    operand, layout = (keys.words, keys.layout) if Q <= 32 else (keys.ints8, _lib.LAYOUT_INT8)
    assert L.bsi_hip_linear_coop_serves(Q, d, R, 2, 7, layout, 6) == 1
    x = torch.randn(Q, d, generator=gen, device="cuda")
    x[Q // 2] *= 3.0e6  # a row that is quantised in 64 bits
    area = torch.zeros(int(L.bsi_hip_linear_coop_bytes()), dtype=torch.uint8, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream

    def run(number):
        out = torch.full((Q, R), float("nan"), device="cuda")
        begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        begin.record()
        rc = L.bsi_hip_linear_coop_out(x.data_ptr(), _lib.DTYPE_F32, Q, d, 2, 7, number, area.data_ptr(), operand.data_ptr(), layout,
                                       keys.slice_weights.data_ptr(), 6, R, 1e-4, R, None, out.data_ptr(), _lib.DTYPE_F32, None, 0, stream)
        end.record()
        assert rc == 0
        end.synchronize()
        return out, begin.elapsed_time(end)

    want = run(1)[0]
    assert not torch.isnan(want).any()
    try:
        assert L.bsi_hip_set_option(SHARES, 32) == 0
        assert L.bsi_hip_set_option(PATIENCE, 100000) == 0  # 1 ms
        got = [run(2 + i) for i in range(3)]
        assert L.bsi_hip_set_option(PATIENCE, 0) == 0
        got += [run(10 + i) for i in range(3)]
    finally:
        L.bsi_hip_set_option(SHARES, 0)
        L.bsi_hip_set_option(PATIENCE, 500)
    assert all(torch.equal(want, out) for out, _ in got)
    times = [ms for _, ms in got]
    # a wait for each of them where a copy has one workgroup, and where all workgroups build the same one
    waits = most - owned if owned == 1 else (most - owned) // 2
    assert 0.95 < min(times[:3]) < waits + 0.5, times
    assert min(times[3:]) < 0.4, times
