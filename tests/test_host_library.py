"""Which host extension goes with which library, and what is said first where one is missing (CPU)."""
import importlib.util
import os
import subprocess
import sys

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, 'flash-linear-attention_amd')
BUILT = os.path.join(PKG, 'fla_hip', '_C')

needs_build = pytest.mark.skipif(not os.path.exists(os.path.join(BUILT, 'gdn_host.so')), reason='not built in this checkout')


def run(code, library):
    env = dict(os.environ, PYTHONPATH=PKG, FLA_HIP_LIBRARY=str(library))
    r = subprocess.run([sys.executable, '-c', code], env=env, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    return r.stdout.split()


def test_arguments_are_checked_before_the_library_is_asked_for(tmp_path):
    out = run(r'''
import torch
from fla_hip import _lib
from fla_hip.ops.gated_delta_rule import chunk_gated_delta_rule, fused_recurrent_gated_delta_rule
z = torch.zeros
for call in (lambda: fused_recurrent_gated_delta_rule(z(1, 1, 2, 64), z(1, 1, 3, 64), z(1, 1, 2, 64)),
             lambda: fused_recurrent_gated_delta_rule(z(2, 1, 2, 64), z(2, 1, 2, 64), z(2, 1, 2, 64), cu_seqlens=torch.tensor([0, 1, 2])),
             lambda: chunk_gated_delta_rule(z(1, 1, 2, 64), z(1, 1, 3, 64), z(1, 1, 2, 64), z(1, 1, 2), z(1, 1, 2)),
             _lib.load):
    try:
        call()
    except Exception as exc:
        print(type(exc).__name__)
''', tmp_path / 'libgdn_hip.so')
    assert out == ['ValueError', 'ValueError', 'ValueError', 'GDNLibraryError']


@needs_build
@pytest.mark.parametrize('beside', [False, True])
def test_the_host_extension_follows_the_library(tmp_path, beside):
    for name in ('libgdn_hip.so', *(['gdn_host.so'] if beside else [])):
        os.symlink(os.path.join(BUILT, name), tmp_path / name)
    out = run('from fla_hip import _lib; print(_lib.host().__file__)', tmp_path / 'libgdn_hip.so')
    assert out == [str((tmp_path if beside else type(tmp_path)(BUILT)) / 'gdn_host.so')]


@needs_build
def test_a_library_elsewhere_without_any_host_extension_runs_behind_the_python_path(tmp_path):
    os.symlink(os.path.join(BUILT, 'libgdn_hip.so'), tmp_path / 'libgdn_hip.so')
    out = run('''
from fla_hip import _lib
_lib._HERE = '/nowhere'
print(_lib.host().__name__, _lib.host().chunk_fwd(1, 2, 3), _lib.load().gdn_hip_abi_version() == _lib.ABI_VERSION)
''', tmp_path / 'libgdn_hip.so')
    assert out == ['_PythonHost', 'None', 'True']


@needs_build
def test_the_package_s_own_library_needs_its_extension(monkeypatch):
    from fla_hip import _lib
    monkeypatch.setattr(_lib, '_host', None)
    monkeypatch.setattr(_lib, '_host_path', lambda: '/nowhere/gdn_host.so')
    with pytest.raises(_lib.GDNLibraryError, match='missing'):
        _lib.host()


@needs_build
def test_an_extension_of_another_torch_is_refused(monkeypatch):
    from fla_hip import _lib
    monkeypatch.setattr(_lib, '_host', None)
    monkeypatch.setattr(torch, '__version__', '1.0')
    with pytest.raises(_lib.GDNLibraryError, match='built with torch'):
        _lib.host()


@needs_build
def test_another_torch_rebuilds_the_extension(monkeypatch):
    spec = importlib.util.spec_from_file_location('gdn_build', os.path.join(PKG, 'build.py'))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    built = []
    monkeypatch.setattr(build, '_compile', lambda *a: None)
    monkeypatch.setattr(build, '_newer', lambda *a: False)
    monkeypatch.setattr(build, '_compile_host', lambda: built.append(1))
    if not os.path.exists(build.HOST_TORCH):
        pytest.skip('built elsewhere')
    build.build(verbose=False)
    assert built == []
    monkeypatch.setattr(build, '_torch_version', lambda: '1.0')
    build.build(verbose=False)
    assert built == [1]


@needs_build
@pytest.mark.skipif(os.path.exists('/dev/kfd') or torch.cuda.is_available(), reason='a launch that fails by itself: only where there is no GPU')
@pytest.mark.parametrize('N,hidden,kernel', [(1, 2048, 'gdn_step_linear_few_kernel'), (16, 256, 'gdn_step_linear_few_kernel'), (17, 256, 'gdn_step_linear_kernel'),
                                             (129, 256, 'gdn_step_linear_kernel')])
def test_a_failed_launch_of_the_step_projections_names_its_kernel(N, hidden, kernel):
    import ctypes

    from fla_hip import _lib

    class Segment(ctypes.Structure):
        _fields_ = [('weight', ctypes.c_void_p), ('cols', ctypes.c_int64), ('out', ctypes.c_void_p), ('conv_weight', ctypes.c_void_p),
                    ('conv_bias', ctypes.c_void_p), ('conv_state', ctypes.c_void_p), ('A_log', ctypes.c_void_p), ('dt_bias', ctypes.c_void_p),
                    ('kind', ctypes.c_int), ('conv_size', ctypes.c_int), ('gate_dtype', ctypes.c_int), ('reserved', ctypes.c_int)]

    x, w, out = (torch.zeros(n, hidden, dtype=torch.bfloat16) for n in (N, 32, N))
    assert x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0
    seg = Segment(weight=w.data_ptr(), cols=32, out=out.data_ptr())              # (kind 0: the map alone)
    status = _lib.load().gdn_step_linear(x.data_ptr(), N, hidden, ctypes.addressof(seg), 1, _lib.DTYPE_BF16, None)
    assert status == _lib.GDN_ERR_LAUNCH
    assert _lib.last_error().startswith(kernel + ':'), _lib.last_error()
