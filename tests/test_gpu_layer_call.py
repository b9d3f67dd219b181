"""A BSI layer's __call__ goes straight to its native forward only where nn.Module.__call__ would do nothing else."""
import pytest
import torch

from test_gpu_parity import ops  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 5, 40])
def test_whatever_hangs_on_a_call_is_honoured(ops, rows):
    from bsipytorch_amd.linear import BSIQuantizedLinear
    from torch.nn.modules import module as nn_module

    layer = BSIQuantizedLinear(torch.nn.Linear(512, 96).cuda(), 2, 0.5)
    x = torch.randn(rows, 512, device="cuda")
    with torch.no_grad():
        want = layer.forward(x)
        assert torch.equal(layer(x), want) and torch.equal(layer(x=x), want)
        seen = []
        for register in (layer.register_forward_hook, nn_module.register_module_forward_hook):
            handle = register(lambda m, i, o: seen.append(m) or o + 1)
            assert torch.equal(layer(x), want + 1)
            handle.remove()
        for register in (layer.register_forward_pre_hook, nn_module.register_module_forward_pre_hook):
            handle = register(lambda m, i: seen.append(m) or (i[0] * 0,))
            assert torch.equal(layer(x), layer.forward(x * 0))
            handle.remove()
        assert len(seen) == 4 and all(m is layer for m in seen)
        layer.forward = lambda t: t  # an instance's own forward
        assert layer(x) is x
        del layer.forward

        class Doubled(BSIQuantizedLinear):
            def forward(self, t):
                return super().forward(t) * 2

        assert torch.equal(Doubled(torch.nn.Linear(512, 96).cuda(), 2, 0.5)(x) * 0, want * 0)
        original, calls = torch.nn.Module.__call__, []
        torch.nn.Module.__call__ = lambda m, *a, **k: calls.append(m) or original(m, *a, **k)
        try:
            assert torch.equal(layer(x), want) and calls == [layer]
        finally:
            torch.nn.Module.__call__ = original
        assert torch.equal(layer(x), want) and len(calls) == 1
    with pytest.raises(TypeError):
        layer(x, x)


def test_a_profiler_sees_the_modules(ops, tmp_path):
    import sys

    from bsipytorch_amd.linear import BSIQuantizedLinear

    layer = BSIQuantizedLinear(torch.nn.Linear(512, 96).cuda(), 2, 0.5)
    x = torch.randn(16, 512, device="cuda")
    with torch.no_grad():
        want = layer(x)
        frames = []
        sys.setprofile(lambda frame, event, arg: frames.append(frame.f_code) if event == "call" else None)
        try:
            got = layer(x)
        finally:
            sys.setprofile(None)
        assert torch.equal(got, want) and BSIQuantizedLinear.forward.__code__ in frames
        with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU], with_stack=True) as profile:
            layer(x)
    profile.export_chrome_trace(str(tmp_path / "trace.json"))
    assert "nn.Module: BSIQuantizedLinear" in (tmp_path / "trace.json").read_text()

def test_compiled_models_break_at_the_layer_without_a_warning(ops):
    """torch.compile of a model with such a layer: the layer runs as it does eagerly, between the graphs."""
    import os
    import subprocess
    import sys

    code = """
import torch
from bsipytorch_amd.linear import BSIQuantizedLinear
class Model(torch.nn.Module):
    def __init__(self):
        super().__init__()
        self.a, self.b = (BSIQuantizedLinear(torch.nn.Linear(512, n).cuda(), 2, 0.5) for n in (512, 96))
    def forward(self, x):
        return self.b(torch.relu(self.a(x * 2))) * 3
model = Model()
for rows in (1, 16, 64):
    x = torch.randn(rows, 512, device="cuda")
    with torch.no_grad():
        want = model(x)
        torch._dynamo.reset()
        compiled = torch.compile(model, backend="eager")
        assert all(torch.equal(compiled(x), want) for _ in range(3))
print("same")
"""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    run = subprocess.run([sys.executable, "-c", code], cwd=root, capture_output=True, text=True, timeout=100)
    assert run.returncode == 0 and "same" in run.stdout, run.stderr
    assert "Dynamo does not know how to trace" not in run.stderr, run.stderr
