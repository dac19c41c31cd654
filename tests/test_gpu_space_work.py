"""Work arrays of Space2's operations: none for the row operators on interleaved arrays, no more than the
transforms use, and smaller chunks of the batch where the card cannot hold those of the whole one."""
import os
import subprocess
import sys

import pytest

from conftest import ROOT

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def _field(shape, batch, cplx):
    import torch
    g = torch.Generator(device="cuda").manual_seed(3)
    return torch.randn((batch,) + tuple(shape) + ((2,) if cplx else ()), generator=g, device="cuda", dtype=torch.float64)


@pytest.mark.parametrize("case", [("rows", 4, 512, 1, 513, 0), ("transform", 4, 512, 1, 513, 2),
                                  ("transform", 1, 500, 2, 471, 1), ("transform", 0, 512, 1, 513, 2)])
def test_work_arrays_held(case):
    """arrays: how many of the whole batch the operations of a case need"""
    import torch
    from rustpde_amd import Space2, _lib
    ops, k0, n0, k1, n1, arrays = case
    print("case work arrays", case, flush=True)
    L, sp, batch = _lib.load(), Space2((k0, n0), (k1, n1)), 16
    c = sp.is_complex
    v, spec, ortho = (_field(s, batch, x) for s, x in ((sp.shape_physical, False), (sp.shape_spectral, c),
                                                       (sp.shape_ortho, c)))
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
    one = 8 * batch * max(n0 + 2, n0) * n1
    assert used <= arrays * one + 6 * MIB, (used / MIB, one / MIB)


# In a process of its own, whose runtime refuses single allocations above a tenth of a hundredth of the card
# (set before it starts; the limit is checked first), with the caller's arrays in pinned host memory, which
# kernels read and write like device arrays.
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
