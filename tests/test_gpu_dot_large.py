"""Large layers as integer sums in units of a row's smallest scale: the bits of the fp32 chain over the chunks, on ragged edges,
row lengths around the masks' words, row scales, every type; rows whose scales lie far apart, whose magnitudes could make the
chain round, or whose blocks are mostly in the second image, which go through the chain; zeros."""
import pytest
import torch

from test_gpu_parity import hip, ops  # noqa: F401  (fixtures)

pytestmark = pytest.mark.gpu

SHAPES = [(512, 256, 256), (513, 4096, 300), (700, 1024, 257), (1029, 4352, 130), (600, 8192, 500), (520, 16384, 260), (777, 1600, 640),
          (512, 100, 513), (640, 64, 16)]


def layers(hip, ops, Q, d, R, x, bias=True):
    """The layer's output with tiles of 256 x 256 and of 128 x 128."""
    from bsipytorch_amd.linear import BSIQuantizedLinear

    layer = BSIQuantizedLinear(torch.nn.Linear(d, R, bias=bias).cuda(), 2, 0.5)
    outs = []
    for tile in (256, 128):
        hip.check(hip.lib.bsi_hip_set_option(hip.OPT_I8_TILE, tile), "tile")
        try:
            with torch.no_grad():
                outs.append(layer(x.clone()))
                outs.append(layer(x.clone()))
        finally:
            hip.check(hip.lib.bsi_hip_set_option(hip.OPT_I8_TILE, 0), "tile")
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[2], outs[3])
    return outs[0], outs[2]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Q,d,R", SHAPES)
def test_same_bits_as_the_chain(hip, ops, Q, d, R, dtype):
    gen = torch.Generator(device="cuda").manual_seed(Q + d + R)
    x = torch.randn(Q, d, generator=gen, device="cuda")
    x[:, torch.rand(d, generator=gen, device="cuda") < 0.004] *= 25.0
    x[3] = 0
    x[5, d // 2:] = 0
    got, want = layers(hip, ops, Q, d, R, x.to(dtype), bias=Q % 2 == 0)
    assert torch.equal(got, want)


@pytest.mark.parametrize("what", ["wide", "far", "huge", "tails", "one row", "nan"])
def test_what_the_chain_has_to_take(hip, ops, what):
    Q, d, R = 600, 2048, 300
    gen = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn(Q, d, generator=gen, device="cuda")
    if what == "wide":  # the first chunk's values a thousand times the others'
        x[:, :256] *= 1000.0
    elif what == "far":
        x[:, :256] *= 1.0e5
    elif what == "huge":  # same signs: the sums of magnitudes exceed 2^24 units
        x = x.abs() * 30 + 1
        x[:, -256:] *= 0.002
    elif what == "tails":
        x = x * torch.exp(2.5 * torch.randn(Q, d, generator=gen, device="cuda"))
    elif what == "one row":
        x[300, 17] = 3.0e8
    else:
        x[300, 17] = float("nan")
        x[4, 5] = float("inf")
    got, want = layers(hip, ops, Q, d, R, x)
    assert torch.equal(got, want)


def test_bits_of_the_popcount_core(hip, ops):
    from bsipytorch_amd.linear import BSIQuantizedLinear

    Q, d, R = 515, 1280, 270
    gen = torch.Generator(device="cuda").manual_seed(9)
    layer = BSIQuantizedLinear(torch.nn.Linear(d, R, bias=False).cuda(), 2, 0.5)
    x = torch.randn(Q, d, generator=gen, device="cuda")
    x[:, ::300] *= 20.0
    hip.check(hip.lib.bsi_hip_set_option(hip.OPT_I8_TILE, 256), "tile")
    try:
        with torch.no_grad():
            got = layer(x)
    finally:
        hip.check(hip.lib.bsi_hip_set_option(hip.OPT_I8_TILE, 0), "tile")
    queries = ops.build_bsi_queries_cuda_batch_packed(x, 2, 0.5)
    assert torch.equal(got, ops.debug_chunk_ints(queries, layer._bsi_keys_cuda, "valu")[1])
