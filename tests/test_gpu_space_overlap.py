"""Operations of Space2 that change nothing (to_ortho and from_ortho of plain Chebyshev and Fourier axes) on
arrays that overlap in part: each field moves as if its input had been read whole before its output was
written, fields in turn."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("op", ["fs_from_ortho", "fs_to_ortho"])
@pytest.mark.parametrize("case", [(4, 64, 0, 65, 16), (4, 64, 0, 65, 8), (4, 12, 0, 40, 160), (0, 33, 0, 40, 8),
                                  (0, 33, 0, 40, 4000)])
def test_identity_on_overlapping_arrays(case, op):
    from rustpde_amd import Space2, _lib
    from rustpde_amd.funspace import _Dev
    k0, n0, k1, n1, shift = case  # the output starts `shift` bytes beyond the input, or before it
    print("case overlap", case, op, flush=True)
    L, sp = _lib.load(), Space2((k0, n0), (k1, n1))
    a = np.random.default_rng(2).standard_normal(sp.shape_ortho + ((2,) if sp.is_complex else ()))
    buf = _Dev(a.nbytes + shift)
    for src, dst in ((0, shift), (shift, 0)):
        _lib.check(L.rbc_memcpy_h2d(ctypes.c_void_p(buf.p.value + src), a.ctypes.data, a.nbytes))
        _lib.check(getattr(L, op)(sp._h, ctypes.c_void_p(buf.p.value + src), ctypes.c_void_p(buf.p.value + dst), 1))
        got = np.zeros_like(a)
        _lib.check(L.rbc_memcpy_d2h(got.ctypes.data, ctypes.c_void_p(buf.p.value + dst), a.nbytes))
        assert np.array_equal(got, a), (src, dst)
