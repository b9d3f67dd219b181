"""Small layers in one launch where shares of the build belong to no workgroup: a workgroup waits a patience for the first, half of it for
the next, down to 2.5 us, and builds them itself."""
import pytest
import torch

from test_gpu_parity import ops  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu

PATIENCE, SHARES = 6, 7  # BSI_OPT_COOP_PATIENCE, BSI_OPT_COOP_SHARES


@pytest.mark.parametrize("Q,d,R", [(33, 768, 768), (100, 512, 512), (16, 1024, 512),  # chunk scales, both kernels: 13, 25 and 16 of 32 shares owned
                                   (5, 300, 64), (64, 320, 320)])  # row scales, both kernels: 1 of 5, 8 of 32
def test_waits_that_run_out(ops, Q, d, R):
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
        L.bsi_hip_set_option(PATIENCE, 2000)
    assert all(torch.equal(want, out) for out, _ in got)
    times = [ms for _, ms in got]
    # 1 + 1/2 + 1/4 ... ms, at most 2, and 2.5 us and the build of a share for each of up to 31; at 1 ms each, the four of the fewest
    # here would take 4
    assert 0.95 < min(times[:3]) < 3.0, times
    assert min(times[3:]) < 0.4, times
