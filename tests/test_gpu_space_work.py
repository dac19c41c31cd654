"""Work arrays of Space2's operations: none for the row operators on interleaved arrays, no more than the
transforms use, and smaller chunks of the batch where the card cannot hold those of the whole one."""
import os
import subprocess
import sys

import pytest

from conftest import ROOT

pytestmark = pytest.mark.gpu

# Both tests run in processes of their own: torch, which measures and allocates here, has to be imported
# before the library.
HELD = """
import sys
sys.path.insert(0, %r)
import torch
from rustpde_amd import Space2, _lib
L, batch, MIB = _lib.load(), 16, 1 << 20
# arrays: how many work arrays of the whole batch the operations need
for ops, k0, n0, k1, n1, arrays in (("rows", 4, 512, 1, 513, 0), ("transform", 4, 512, 1, 513, 2),
                                    ("transform", 1, 500, 2, 471, 1), ("transform", 0, 512, 1, 513, 2)):
    sp = Space2((k0, n0), (k1, n1))
    two = 2 if sp.is_complex else 1
    v, spec, ortho = (torch.randn((batch,) + s + (t,), device="cuda", dtype=torch.float64)
                      for s, t in ((sp.shape_physical, 1), (sp.shape_spectral, two), (sp.shape_ortho, two)))
    outs = [torch.empty_like(t) for t in (v, spec, ortho)]

    def calls(b):
        if ops == "rows":
            for d0, d1 in ((1, 0), (0, 1), (0, 2)):
                _lib.check(L.fs_gradient(sp._h, spec.data_ptr(), outs[2].data_ptr(), d0, d1, 2.0, 1.0, b))
            _lib.check(L.fs_to_ortho(sp._h, spec.data_ptr(), outs[2].data_ptr(), b))
            _lib.check(L.fs_from_ortho(sp._h, ortho.data_ptr(), outs[1].data_ptr(), b))
        else:
            _lib.check(L.fs_forward(sp._h, v.data_ptr(), outs[1].data_ptr(), b))
            _lib.check(L.fs_backward(sp._h, spec.data_ptr(), outs[0].data_ptr(), b))

    calls(1)  # operators and tables, work arrays of one field
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    calls(batch)
    used = before - torch.cuda.mem_get_info()[0]
    one = 8 * batch * (n0 + 2) * n1
    print(ops, k0, n0, k1, n1, used / MIB, one / MIB, flush=True)
    assert used <= arrays * one + 6 * MIB
print("all held", flush=True)
"""


def test_work_arrays_held():
    print("case work arrays held", flush=True)
    r = subprocess.run([sys.executable, "-u", "-c", HELD % ROOT], timeout=100, capture_output=True, text=True)
    assert r.returncode == 0 and "all held" in r.stdout, r.stdout + r.stderr


# The runtime refuses single allocations above a thousandth of the card (set before the process starts; the
# limit is checked first); the caller's arrays lie in pinned host memory, which kernels read and write like
# device arrays.
CHILD = """
import ctypes, sys
sys.path.insert(0, %r)
import torch
from rustpde_amd import Space2, _lib
L, p = _lib.load(), ctypes.c_void_p()
batch = 200
for k0, n0, k1, n1 in ((4, 512, 1, 513), (1, 500, 2, 471)):
    sp = Space2((k0, n0), (k1, n1))
    size = (n0 + 2) * n1
    assert L.rbc_dev_malloc(ctypes.byref(p), 8 * batch * size) != 0, "no limit on allocations"
    v = torch.randn((batch,) + sp.shape_physical, dtype=torch.float64).pin_memory()
    two = 2 if sp.is_complex else 1
    got = torch.empty((batch,) + sp.shape_spectral + (two,), dtype=torch.float64, pin_memory=True)
    one = torch.empty_like(got[0]).pin_memory()
    _lib.check(L.fs_forward(sp._h, v.data_ptr(), got.data_ptr(), batch))
    for b in (0, 1, 99, 100, batch - 1):
        _lib.check(L.fs_forward(sp._h, v[b].data_ptr(), one.data_ptr(), 1))
        assert torch.equal(got[b], one), (k0, b)
    _lib.check(L.fs_backward(sp._h, got.data_ptr(), v.data_ptr(), batch))
    back = torch.empty_like(v[0]).pin_memory()
    for b in (0, batch - 1):
        _lib.check(L.fs_backward(sp._h, got[b].data_ptr(), back.data_ptr(), 1))
        assert torch.equal(v[b], back), (k0, b)
print("whole batches done", flush=True)
"""


def test_smaller_chunks_where_memory_is_short():
    print("case work arrays larger than an allocation may be", flush=True)
    env = dict(os.environ, GPU_MAX_HEAP_SIZE="1", GPU_SINGLE_ALLOC_PERCENT="10")
    r = subprocess.run([sys.executable, "-u", "-c", CHILD % ROOT], env=env, timeout=100, capture_output=True, text=True)
    assert r.returncode == 0 and "whole batches done" in r.stdout, r.stdout + r.stderr
