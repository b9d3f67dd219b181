"""The native host path serves the default calls with the Python path's bits, follows what happens to the layer, and leaves
everything else to the Python path."""
import threading

import pytest
import torch

from test_gpu_parity import ops  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("shape", [(512,), (1, 512), (4, 512), (2, 9, 512), (33, 512), (3, 100, 512)])
def test_served_calls_match_the_python_path(ops, monkeypatch, shape, dtype):
    from bsipytorch_amd import _native
    from bsipytorch_amd.linear import BSIQuantizedLinear

    torch.manual_seed(3)
    layer = BSIQuantizedLinear(torch.nn.Linear(512, 200).cuda(), 2, 0.5)
    x = torch.randn(*shape, device="cuda").to(dtype)
    strided = torch.randn(*shape, 2, device="cuda").to(dtype)[..., 0]
    with torch.no_grad():
        layer(x)  # the first call of a shape makes the workspace
        assert layer.dot_calls == 1
        got = _native.linear(layer.__dict__, x)
        assert got is not None and got.shape == shape[:-1] + (200,) and got.dtype == dtype and layer.dot_calls == 2
        got_strided = _native.linear(layer.__dict__, strided)
        x2 = x.clone()
        got2 = layer(x2)
        x2.mul_(2)
        got3 = layer(x2)  # an in-place change is seen
        monkeypatch.setenv("BSI_LINEAR_ONE_CALL", "0")
        monkeypatch.setenv("BSI_FUSED_LINEAR", "0")
        assert _native.linear(layer.__dict__, x) is None  # a switch is set
        assert torch.equal(got, layer(x)) and torch.equal(got2, got) and torch.equal(got_strided, layer(strided))
        assert torch.equal(got3, layer(x2))
    assert not layer(x.requires_grad_()).requires_grad


def test_calls_it_leaves_alone(ops):
    from bsipytorch_amd import _native
    from bsipytorch_amd.linear import BSIQuantizedLinear

    layer = BSIQuantizedLinear(torch.nn.Linear(256, 64).cuda(), 2, 0.5)
    x = torch.randn(8, 256, device="cuda")
    layer(x)
    assert _native.linear(layer.__dict__, x) is not None
    for other in (x.cpu(), x[:0], x.double(), x[:, :128].contiguous()):
        assert _native.linear(layer.__dict__, other) is None
    layer.bias = layer.bias.cpu()
    assert _native.linear(layer.__dict__, x) is None
    ops._reset_flag_cache()
    assert _native.linear(layer.__dict__, x) is None  # the flags have not been read yet
    with pytest.raises(RuntimeError, match="Word count mismatch"):
        ops.batch_dot_product_multiquery_cuda_batch_caps(ops.build_bsi_queries_cuda_batch_packed(x[:, :128].contiguous(), 2),
                                                         layer._bsi_keys_cuda)


@pytest.mark.parametrize("rows", [1, 16, 64])
@pytest.mark.parametrize("how", ["parameter", "parametrization", "attribute"])
def test_a_bias_that_is_no_buffer_is_added(ops, rows, how):
    from bsipytorch_amd.linear import BSIQuantizedLinear
    from torch.nn.utils import parametrize

    torch.manual_seed(6)
    layer = BSIQuantizedLinear(torch.nn.Linear(512, 96).cuda(), 2, 0.5)
    x = torch.randn(rows, 512, device="cuda")
    other = torch.randn(96, device="cuda")
    with torch.no_grad():
        for _ in range(2):  # the first call of a shape is the Python path's
            before = layer(x)
        if how == "parameter":
            layer.bias = torch.nn.Parameter(other)
        elif how == "parametrization":
            class Other(torch.nn.Module):
                def forward(self, bias):
                    return other

            parametrize.register_parametrization(layer, "bias", Other(), unsafe=True)
        else:
            layer.__dict__["bias"] = other
        plain = BSIQuantizedLinear(torch.nn.Linear(512, 96, bias=False).cuda(), 2, 0.5)
        plain._bsi_keys_cuda = layer._bsi_keys_cuda
        for _ in range(2):
            got = layer(x)
            assert torch.equal(got, plain(x) + other) and not torch.equal(got, before)


@pytest.mark.parametrize("rows", [256, 512])
def test_a_tensor_given_other_storage_is_built_anew(ops, rows):
    from bsipytorch_amd.linear import BSIQuantizedLinear

    torch.manual_seed(7)
    d, out = 2048, 8192
    assert not ops.lib.bsi_hip_linear_coop_serves(rows, d, out, 2, 7, 2, 6)  # build and dot in launches of their own
    layer = BSIQuantizedLinear(torch.nn.Linear(d, out).cuda(), 2, 0.5)
    x = torch.randn(rows, d, device="cuda")
    other = torch.randn(rows, d, device="cuda")
    with torch.no_grad():
        want = layer(other).clone()
        for _ in range(2):  # the first call of a shape is the Python path's
            layer(x)
        x.data = torch.empty(0, device="cuda")  # frees the storage; the version stays as it is
        fresh = torch.empty(rows, d, device="cuda").copy_(other)  # where the freed one was, if nothing holds that
        x.data = fresh
        assert torch.equal(layer(x), want)


def test_threads_on_one_stream(ops):
    from bsipytorch_amd.linear import BSIQuantizedLinear

    torch.manual_seed(4)
    layers = [BSIQuantizedLinear(torch.nn.Linear(512, 256).cuda(), 2, 0.5) for _ in range(4)]
    xs = [torch.randn(64, 512, device="cuda") for _ in range(4)]
    with torch.no_grad():
        want = [layer(x).clone() for layer, x in zip(layers, xs)]
    wrong = []

    def work(i):
        with torch.no_grad():
            for _ in range(200):
                if not torch.equal(layers[i](xs[i]), want[i]):
                    wrong.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not wrong


def test_operands_replaced_by_another_thread(ops):
    from bsipytorch_amd.linear import BSIQuantizedLinear

    torch.manual_seed(8)
    layer = BSIQuantizedLinear(torch.nn.Linear(512, 256).cuda(), 2, 0.5)
    kept = layer._bsi_keys_cuda
    xs = [torch.randn(rows, 512, device="cuda") for rows in (1, 16, 512)]
    batch, streams = ops.build_bsi_queries_cuda_batch_packed(xs[1], 2), ops.build_bsi_queries_cuda_batch_hybrid(xs[1], 2)

    def results():
        dots = [ops.batch_dot_product_multiquery_cuda_batch_caps(q, layer._bsi_keys_cuda)[0] for q in (batch, streams)]
        return [layer(x) for x in xs] + dots

    done = threading.Event()

    def replace():
        owners = [kept, batch, streams]
        tensors = [{n: t for n, t in vars(o).items() if torch.is_tensor(t)} for o in owners]
        while not done.is_set():
            for owner, named in zip(owners, tensors):
                vars(owner).update({n: t.clone() for n, t in named.items()})

    with torch.no_grad():
        want = results()
        thread = threading.Thread(target=replace)
        thread.start()
        try:
            for _ in range(300):
                assert all(torch.equal(a, b) for a, b in zip(results(), want))
        finally:
            done.set()
            thread.join()


@pytest.mark.parametrize("rows,d,dtype", [(1, 64, torch.float32), (33, 300, torch.bfloat16), (64, 8192, torch.float16)])
def test_key_build_matches_the_python_path(ops, rows, d, dtype):
    from bsipytorch_amd import _native

    torch.manual_seed(5)
    K = (torch.randn(rows, d, device="cuda") * 0.1).to(dtype)
    column_major = torch.empty(d, rows, dtype=dtype, device="cuda").t().copy_(K)
    got, want = ops.build_bsi_keys_cuda(torch.nn.Parameter(K), 2, 0.5), ops.build_bsi_keys_cuda(K.double(), 2, 0.5)
    assert _native.build_keys(K.double(), 2, 6) is None and _native.build_keys(K, 3, 6) is None
    assert column_major.is_contiguous() or _native.build_keys(column_major, 2, 6) is None
    assert got[1:] == want[1:]
    a, b = vars(got[0]), vars(want[0])
    assert set(a) == set(b) == set(vars(ops.PrebuiltBSIKeysCUDA()))
    for name in a:
        assert torch.equal(a[name], b[name]) if torch.is_tensor(a[name]) else a[name] == b[name], name
