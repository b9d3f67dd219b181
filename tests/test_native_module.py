"""The native host path is optional: a process that cannot load it says so and has the whole package without it."""
import glob
import os
import subprocess
import sys
import sysconfig

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _run(code):
    return subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=300)


def test_the_module_carries_this_pythons_tag():
    built = [os.path.basename(p) for p in glob.glob(os.path.join(ROOT, "bsipytorch_amd", "_native*.so"))]
    assert "_native" + sysconfig.get_config_var("EXT_SUFFIX") in built and "_native.so" not in built


def test_import_without_the_module():
    r = _run("import sys, warnings\n"
             "sys.modules['bsipytorch_amd._native'] = None\n"
             "with warnings.catch_warnings(record=True) as seen:\n"
             "    warnings.simplefilter('always')\n"
             "    import bsi_ops, bsipytorch_amd.linear as linear, torch\n"
             "assert len([w for w in seen if 'native host path' in str(w.message)]) == 1\n"
             "assert linear.BSIQuantizedLinear.__call__ is torch.nn.Module.__call__\n"
             "bsi_ops._reset_flag_cache()\n"
             "x = torch.zeros(2, 3)\n"
             "a = bsi_ops._native.build_key(x, 2, 6)\n"
             "assert a == bsi_ops._native.build_key(x, 2, 6) != bsi_ops._native.build_key(x.add_(1), 2, 6)\n"
             "print('whole')")
    assert r.returncode == 0 and "whole" in r.stdout, r.stderr


def test_functions_of_an_unbound_module():
    """Imported by itself the module knows no library and no layer class: every call is left alone, none ends the process."""
    r = _run("import torch\n"
             "from bsipytorch_amd import _native\n"
             "x = torch.zeros(2, 64)\n"
             "assert _native.linear({}, x) is None and _native.dot(x, x) is None and _native.dot_streams(x, x) is None\n"
             "assert _native.build(x, 2, True, True) is None and _native.build_keys(x, 2, 6) is None and _native.hybrid(x, 2, 0.5) is None\n"
             "assert _native.ewah_streams(x.long(), 0.5) is None and _native.scalar_query(x[0], x, x, 2, 0.5, 1.0) is None\n"
             "try:\n"
             "    _native.layer_call(torch.nn.ReLU(), x)\n"
             "except RuntimeError as e:\n"
             "    print(e)\n"
             "_native.forget()")
    assert r.returncode == 0 and "bind_layer" in r.stdout, (r.returncode, r.stderr)


def test_another_torch_is_refused():
    r = _run("import torch\n"
             "torch.__version__ = '2.1.0'\n"
             "try:\n"
             "    from bsipytorch_amd import _native\n"
             "except ImportError as e:\n"
             "    print(e)")
    assert r.returncode == 0 and "this is 2.1.0" in r.stdout, r.stderr


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["float32", "float16"])
def test_results_without_the_module(monkeypatch, dtype):
    import torch

    from bsipytorch_amd import _host, bsi_ops, bsi_scalar, linear

    gen = torch.Generator(device="cuda").manual_seed(9)
    kind = getattr(torch, dtype)
    weights = torch.randn(384, 512, generator=gen, device="cuda") * 0.1
    dense = torch.nn.Linear(512, 384).cuda()
    xs = [torch.randn(rows, 512, generator=gen, device="cuda").to(kind) for rows in (1, 16, 40, 512)]

    def results():
        keys = bsi_ops.build_bsi_keys_cuda(weights.to(kind), 2, 0.5)[0]
        layer = linear.BSIQuantizedLinear(dense, 2, 0.5)
        out = [keys.words, keys.ints8, keys.slice_weights]
        with torch.no_grad():
            for x in xs:
                out += [torch.nn.Module.__call__(layer, x) for _ in range(2)]
                out.append(bsi_ops.batch_dot_product_multiquery_cuda_batch_caps(
                    bsi_ops.build_bsi_queries_cuda_batch_packed(x, 2, 0.5), keys)[0])
                streams = bsi_ops.build_bsi_queries_cuda_batch_hybrid(x, 2, 0.5)
                out += [streams.comp_words, streams.comp_off, streams.comp_len, streams.flags,
                        bsi_ops.batch_dot_product_multiquery_cuda_batch_caps(streams, keys)[0]]
        decimal = bsi_ops.build_bsi_keys(weights, 2, 0.5)[0]
        return out + [bsi_ops.batch_dot_product_prebuilt(xs[0][0].float(), decimal)[0]]

    want = results()
    for module in (bsi_ops, bsi_scalar, linear):
        monkeypatch.setattr(module, "_native", _host.PythonPath)
    got = results()
    bsi_ops.linear_cuda_forget()
    assert len(got) == len(want) and all(torch.equal(a, b) for a, b in zip(got, want))
