"""The native binding leaves the GIL while a library call runs (a launch blocks while the
stream's queue is full), on a second copy of the module whose entry points block until
another Python thread lets them go."""
import ctypes
import importlib.util
import os
import shutil
import subprocess
import threading

import pytest
import torch

from deep_gemm import _ffi

# An entry point returns 7 once another thread has set `go`, and 0 after 5 s without it.
STUB = r'''
#include <atomic>
#include <chrono>
#include <cstdint>
#include <thread>
extern "C" {
std::atomic<int> entered{0}, go{0};
int blocked() {
    entered = 1;
    for (auto t = std::chrono::steady_clock::now(); std::chrono::steady_clock::now() - t < std::chrono::seconds(5);) {
        if (go) return 7;
        std::this_thread::sleep_for(std::chrono::milliseconds(1));
    }
    return 0;
}
int64_t workspace_size(int64_t m, int64_t, int64_t) { return m == 64 ? 256 : 0; }
}
'''


@pytest.fixture(scope='module')
def stub(tmp_path_factory):
    d = tmp_path_factory.mktemp('stub')
    (d / 'stub.cpp').write_text(STUB)
    subprocess.run(['g++', '-O1', '-std=c++17', '-shared', '-fPIC', str(d / 'stub.cpp'), '-o', str(d / 'stub.so')], check=True)
    lib = ctypes.CDLL(str(d / 'stub.so'))
    copy = shutil.copy(_ffi.bind.__file__, d / os.path.basename(_ffi.bind.__file__))
    spec = importlib.util.spec_from_file_location('_dgbind', copy)
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    assert mod is not _ffi.bind
    addr = [ctypes.cast(lib.blocked, ctypes.c_void_p).value] * 11
    addr[2] = ctypes.cast(lib.workspace_size, ctypes.c_void_p).value
    mod.init(*addr)
    return lib, mod


@pytest.mark.parametrize('name,nargs,tensors', [
    ('gemm_nt', 10, 5), ('gemm_nt_ws', 10, 5), ('contiguous', 13, 6), ('masked', 11, 6), ('cast', 6, 3),
    ('dispatch', 14, (0, 1, 2, 7, 8, 9, 10, 12)), ('swiglu', 8, (0, 4, 5)), ('contiguous_swiglu', 12, (0, 1, 2, 3, 4, 7, 8)),
    ('masked_swiglu', 11, (0, 1, 2, 3, 4, 8, 9)), ('combine', 5, (0, 1, 3))])
def test_other_threads_run_during_a_call(stub, name, nargs, tensors):
    lib, mod = stub
    entered, go = (ctypes.c_int.in_dll(lib, v) for v in ('entered', 'go'))
    entered.value = go.value = 0
    t = torch.zeros((64 if name == 'gemm_nt_ws' else 128, 8), dtype=torch.bfloat16)
    at = range(tensors) if isinstance(tensors, int) else tensors
    optional = {'gemm_nt': (5,), 'gemm_nt_ws': (5,), 'dispatch': (3, 11), 'swiglu': (1, 2), 'contiguous_swiglu': (5,),
                'masked_swiglu': (6,), 'combine': (2,)}.get(name, ())
    args = [t if i in at else None if i in optional else 0 for i in range(nargs)]
    got = []
    th = threading.Thread(target=lambda: got.append(getattr(mod, name.replace('_ws', ''))(*args)))
    th.start()
    for _ in range(8000):
        if entered.value or got:
            break
        threading.Event().wait(0.001)
    go.value = 1
    th.join(20)
    assert got == [7], got
