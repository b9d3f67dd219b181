"""Small layers in one launch, the query build inside: the bits of the build and dot in launches of their own, for chunk and
row scales, every type and kernel, also where workgroups build the shares they wait for themselves."""
import pytest
import torch

from test_gpu_parity import ops  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu

PATIENCE = 6  # BSI_OPT_COOP_PATIENCE


@pytest.mark.parametrize("Q,d,R", [(5, 256, 64), (5, 1, 700), (16, 4096, 4096), (32, 1600, 4800), (17, 2047, 16400), (32, 2048, 16384), (7, 300, 1000),
                                   (9, 4000, 2000), (33, 256, 4096), (64, 512, 3328), (121, 512, 14848)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("patience", [2000, 0])
def test_same_bits_as_two_launches(ops, monkeypatch, Q, d, R, dtype, patience):
    from bsipytorch_amd import _native
    from bsipytorch_amd.linear import BSIQuantizedLinear

    gen = torch.Generator(device="cuda").manual_seed(Q + d + R)
    layer = BSIQuantizedLinear(torch.nn.Linear(d, R).cuda(), 2, 0.5)
    keys = layer._bsi_keys_cuda
    layout = keys.layout if Q <= 32 else 2  # BSI_LAYOUT_INT8
    assert ops.lib.bsi_hip_linear_coop_serves(Q, d, R, 2, 7, layout, keys.Sb) == 1
    ops.lib.bsi_hip_set_option(PATIENCE, patience)
    try:
        with torch.no_grad():
            for i in range(4):
                x = torch.randn(Q, d, generator=gen, device="cuda")
                x[:, :: 50] *= 20.0
                if i == 3:
                    x[Q // 2] *= 3.0e6 if dtype != torch.float16 else 100.0  # beyond the float32 quantiser
                x = x.to(dtype)
                layer(x)
                got = _native.linear(layer.__dict__, x)
                assert got is not None
                with monkeypatch.context() as m:
                    m.setenv("BSI_QUERY_CACHE", "0")  # the Python path: build, then dot
                    assert torch.equal(got, layer(x))
    finally:
        ops.lib.bsi_hip_set_option(PATIENCE, 2000)
        ops.linear_cuda_forget()


def test_streams_side_by_side(ops):
    from bsipytorch_amd.linear import BSIQuantizedLinear

    layers = [BSIQuantizedLinear(torch.nn.Linear(1024, 2048).cuda(), 2, 0.5) for _ in range(3)]
    xs = [torch.randn(16, 1024, device="cuda") for _ in range(3)]
    streams = [torch.cuda.Stream() for _ in range(3)]
    with torch.no_grad():
        want = [layer(x).clone() for layer, x in zip(layers, xs)]
        torch.cuda.synchronize()
        for _ in range(50):
            got = []
            for layer, x, stream in zip(layers, xs, streams):
                with torch.cuda.stream(stream):
                    got.append(layer(x.clone()))
            torch.cuda.synchronize()
            assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_areas_are_bounded_and_given_back(ops):
    """33 streams for 32 areas: the one without runs its layers in two launches, until areas have been idle for 4096 launches."""
    from bsipytorch_amd.linear import BSIQuantizedLinear

    area = ops.lib.bsi_hip_linear_coop_bytes()
    layer = BSIQuantizedLinear(torch.nn.Linear(1024, 2048).cuda(), 2, 0.5)
    x = torch.randn(16, 1024, device="cuda")
    streams = [torch.cuda.default_stream()] + [torch.cuda.Stream() for _ in range(32)]
    assert len({s.cuda_stream for s in streams}) == 33

    def on(stream):
        with torch.cuda.stream(stream):
            got = layer(x)
        stream.synchronize()
        return got

    with torch.no_grad():
        ops.linear_cuda_forget()
        want = layer(x)
        for _ in range(2):
            assert all(torch.equal(on(s), want) for s in streams)
        held = torch.cuda.memory_allocated()
        assert held >= 32 * area
        on(streams[-1])
        assert torch.cuda.memory_allocated() < held + area
        with torch.cuda.stream(streams[5]):
            for _ in range(4200):
                layer(x)
        assert torch.cuda.memory_allocated() > held - area  # nothing is taken back before another stream asks
        assert torch.equal(on(streams[-1]), want)
        assert torch.cuda.memory_allocated() < held - 29 * area
        assert all(torch.equal(on(s), want) for s in streams)
    ops.linear_cuda_forget()
    assert torch.cuda.memory_allocated() < held - 30 * area
