"""CPU: the package's host-only surface neither loads torch nor needs it."""
import os
import subprocess
import sys
import types

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _python(code):
    out = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True,
                         timeout=120)
    assert out.returncode == 0, out.stderr
    return out.stdout.strip()


def test_import_does_not_load_torch():
    assert _python("import sys, ferrum_amd; print('torch' in sys.modules)") == "False"


def test_without_torch_import_works_and_device_calls_raise_import_error():
    for error in ("ImportError('not installed')", "OSError('a library is missing')"):
        assert _python(f"""
import sys
class Finder:
    def find_spec(self, name, path=None, target=None):
        if name == "torch":
            raise {error}
sys.meta_path.insert(0, Finder())
import ferrum_amd as fa
calls = [lambda: fa.gemv_q8_0(None, 1, 32, None, None),
         lambda: fa.gemm_q8_0_multi([None], [1], 32, None, 1, [None]),
         lambda: fa.gemm_q8_0_batched([None], [1], 32, None, 1, [None]),
         lambda: fa.PagedKvPool.copy_blocks(None, None),
         lambda: fa.PagedKvPool.append(None, 0, None, None, None)]
for call in calls:
    try:
        call()
    except {error.split('(')[0]} as e:
        assert str(e) == {error}.args[0]
    else:
        raise AssertionError("no error")
print("ok")
""") == "ok"


def test_stream_handle_without_torch_private_functions(monkeypatch):
    """A torch without the C-layer functions: the public call gives the handle."""
    from ferrum_amd import kvcache
    stream = types.SimpleNamespace(cuda_stream=1234)
    cuda = types.SimpleNamespace(is_initialized=lambda: True, current_stream=lambda: stream)
    fake = types.SimpleNamespace(_C=types.SimpleNamespace(), cuda=cuda, Tensor=object)
    monkeypatch.setitem(sys.modules, "torch", fake)
    monkeypatch.setattr(kvcache, "_torch_loaded", None)
    monkeypatch.setattr(kvcache, "_raw_stream", None)
    monkeypatch.setattr(kvcache, "_Tensor", None)
    assert kvcache._stream_ptr(None) == 1234
    fake._C._cuda_getCurrentRawStream = lambda device: 100 + device
    fake._C._cuda_getDevice = lambda: 3
    monkeypatch.setattr(kvcache, "_torch_loaded", None)
    assert kvcache._stream_ptr(None) == 103
    cuda.is_initialized = lambda: False
    assert kvcache._stream_ptr(None) == 1234
    assert kvcache._stream_ptr(7) == 7
