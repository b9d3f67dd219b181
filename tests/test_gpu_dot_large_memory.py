"""The workspace of layers: no images for a large layer's kernel where none has run, and layers whose workspace lacks them."""
import pytest
import torch

from test_gpu_parity import hip, ops  # noqa: F401  (fixtures)

pytestmark = pytest.mark.gpu


def layer_of(d, R):
    from bsipytorch_amd.linear import BSIQuantizedLinear

    return BSIQuantizedLinear(torch.nn.Linear(d, R, device="cuda"), 2, 0.5)


@pytest.fixture
def fresh(ops):
    ops._linear_ws.clear()
    ops._reserved_linear_shapes.clear()
    yield ops._linear_ws
    ops._linear_ws.clear()
    ops._reserved_linear_shapes.clear()


def test_bytes_of_a_layer_that_never_uses_the_images(hip, ops, fresh):
    layer, x = layer_of(2048, 8192), torch.randn(512, 2048, device="cuda")
    with torch.no_grad():
        layer(x), layer(x.clone())
    plain = 512 * (7 * 32 * 8 + 8 * (256 + 8))
    assert plain <= fresh[0]["bytes"] < plain + 4096


def test_a_large_layer_behind_a_small_one(hip, ops, fresh):
    """On one input: the workspace grows, and both have the bits of a layer by itself."""
    small, large, x = layer_of(4096, 256), layer_of(4096, 16384), torch.randn(1024, 4096, device="cuda")
    with torch.no_grad():
        got = [small(x), large(x), small(x), large(x)]
        hip.check(hip.lib.bsi_hip_set_option(hip.OPT_I8_TILE, 128), "tile")
        try:
            want = [small(x.clone()), large(x.clone())] * 2
        finally:
            hip.check(hip.lib.bsi_hip_set_option(hip.OPT_I8_TILE, 0), "tile")
    assert fresh[0]["bytes"] == hip.lib.bsi_hip_linear_workspace_bytes(1024, 4096, 7)
    assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_a_large_layer_recorded_without_a_call_of_its_own(hip, ops, fresh):
    """A capture finds the workspace of the layers that have run; it did so before the images were there."""
    small, large, x = layer_of(4096, 256), layer_of(4096, 16384), torch.randn(1024, 4096, device="cuda")
    ops.device_bias(large.bias, x.device)
    with torch.no_grad():
        small(x)
        before = fresh[0]["bytes"]
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = large(x)
        assert fresh[0]["bytes"] == before
        for seed in (1, 2, 3):
            x.copy_(torch.randn(1024, 4096, generator=torch.Generator().manual_seed(seed)))
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, large(x.clone()))
