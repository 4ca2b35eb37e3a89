"""The pair-by-pair form of partitioned operators (five passes once per source
and target partition on one slot per right-hand side), which runs where the
planes of all partitions are not at hand: planes pinned by a recorded batch of
one right-hand side, then two right-hand sides, against the oracle's partition
matvec, plain and with alpha / beta, on planes with and without the two-pass
kernels; and the allocation-free entry where all partitions exceed its
scratch."""
import ctypes
from fractions import Fraction

import numpy as np
import pytest

H = Fraction(1, 32)

# (source partition cells, target partition cells, source divisors, target divisors);
# branch lengths 8 to 24 on axes 1 and 2 run the two-pass kernels
CASES = {
    "src_211_planes": ((8, 6, 10), (8, 10, 6), (2, 1, 1), (1, 1, 1)),
    "src_222": ((4, 6, 10), (6, 4, 8), (2, 2, 2), (1, 1, 1)),
    "trg_112_planes": ((10, 8, 6), (6, 16, 26), (1, 1, 1), (1, 1, 2)),
    "trg_123": ((8, 4, 6), (4, 8, 26), (1, 1, 1), (1, 2, 3)),
    "both_21_12_planes": ((12, 30, 8), (12, 18, 8), (2, 1, 1), (1, 2, 1)),
    "both_31_13_long": ((2, 4, 150), (2, 2, 106), (3, 1, 1), (1, 3, 1)),
}


def _operator(gila, S, T, sdiv, tdiv, dtype):
    lat = [H * max(a, b) for a, b in zip(sdiv, tdiv)]
    sS, sT = tuple(m / v for m, v in zip(lat, sdiv)), tuple(m / v for m, v in zip(lat, tdiv))
    Sf, Tf = tuple(c * v for c, v in zip(S, sdiv)), tuple(c * v for c, v in zip(T, tdiv))
    vt, vs = gila.GlaVol(Tf, sT), gila.GlaVol(Sf, sS, (0, 0, 400 * H))
    shp = tuple((s + t) // 2 for s, t in zip(S, T)) + (6, int(np.prod(sdiv)), int(np.prod(tdiv)))
    rng = np.random.default_rng(9)
    fur = [(rng.standard_normal(shp) + 1j * rng.standard_normal(shp)).astype(dtype) for _ in range(8)]
    mem = gila.GlaOprMem(gila.GlaKerOpt(True), vt, vs, egoFur=fur, setTyp=dtype)
    assert tuple(mem._dims.src_div) == sdiv and tuple(mem._dims.trg_div) == tdiv
    return mem, np.concatenate([f.reshape(-1, order="F") for f in fur]).astype(np.complex128), Sf, Tf


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


@pytest.mark.gpu
@pytest.mark.parametrize("case", list(CASES))
@pytest.mark.parametrize("dtype,tol", [(np.complex128, 1e-12), (np.complex64, 1e-5)])
def test_pair_by_pair_under_a_batch(gila, orc, gpu, case, dtype, tol):
    import torch
    from gila_amd import _capi
    print(f"case pair by pair {case} {np.dtype(dtype).name}", flush=True)
    S, T, sdiv, tdiv = CASES[case]
    mem, fur, Sf, Tf = _operator(gila, S, T, sdiv, tdiv, dtype)
    L, n = gila.lib(), 2
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    nx, ny = 3 * int(np.prod(Sf)), 3 * int(np.prod(Tf))
    x = [orc.complex_gaussian(Sf + (3,), seed=80 + r).astype(dtype) for r in range(n)]
    y0 = [orc.complex_gaussian(Tf + (3,), seed=90 + r).astype(dtype) for r in range(n)]
    xd = torch.from_numpy(np.concatenate([v.reshape(-1, order="F") for v in x])).cuda()
    zd = torch.from_numpy(np.concatenate([v.reshape(-1, order="F") for v in y0])).cuda()
    yd, one, both = torch.empty_like(zd), torch.empty_like(zd[:ny]), torch.empty_like(zd)
    al, be = 0.5 - 1.5j, -0.75 + 0.25j
    b = ctypes.c_void_p()
    _capi.check(L.gla_batch_create((ctypes.c_void_p * 1)(mem._h), (ctypes.c_void_p * 1)(xd.data_ptr()),
                                   (ctypes.c_void_p * 1)(one.data_ptr()), (ctypes.c_int64 * 1)(1), 1, 1,
                                   ctypes.byref(b)))
    try:
        _capi.check(L.gla_opr_apply(mem._h, _ptr(xd), nx * n, _ptr(yd), ny * n, n, st))
        _capi.check(L.gla_opr_apply_axpby(mem._h, _ptr(xd), nx * n, _ptr(zd), ny * n, n, al.real, al.imag, be.real,
                                          be.imag, st))
        torch.cuda.synchronize()
    finally:
        L.gla_batch_destroy(b)
    _capi.check(L.gla_opr_apply(mem._h, _ptr(xd), nx * n, _ptr(both), ny * n, n, st))
    torch.cuda.synchronize()
    if int(np.prod(sdiv)) > 1:      # sums over sources round apart: the two forms did run
        assert not torch.equal(yd, both)
    for r in range(n):
        ref = orc.partition_matvec(S, T, sdiv, tdiv, fur, x[r].astype(np.complex128))
        y, z, w = (t[r * ny:(r + 1) * ny].cpu().numpy().reshape(Tf + (3,), order="F") for t in (yd, zd, both))
        assert orc.rel_l2(y, ref) <= tol
        assert orc.rel_l2(z, al * ref + be * y0[r]) <= tol
        assert orc.rel_l2(w, ref) <= tol


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,tol", [(np.complex128, 1e-12), (np.complex64, 1e-5)])
def test_scratch_holds_the_pair_form_only(gila, orc, gpu, dtype, tol):
    # 8 source partitions of 24^3: all of them take more than the scratch
    import torch
    from gila_amd import _capi
    S = T = (24, 24, 24)
    mem, _, Sf, Tf = _operator(gila, S, T, (2, 2, 2), (1, 1, 1), dtype)
    L = gila.lib()
    n = _capi.GLA_NOALLOC_SCRATCH_BYTES // L.gla_opr_workspace_bytes(mem._h, 1) + 1
    print(f"case scratch pair form {np.dtype(dtype).name} nrhs={n}", flush=True)
    nx, ny = 3 * int(np.prod(Sf)), 3 * int(np.prod(Tf))
    xd = torch.from_numpy(orc.complex_gaussian((n * nx,), seed=95).astype(dtype)).cuda()
    yd = torch.empty(n * ny, dtype=xd.dtype, device="cuda")
    zd = torch.empty_like(yd)
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    _capi.check(L.gla_opr_apply_noalloc(mem._h, _ptr(xd), nx * n, _ptr(yd), ny * n, n, st))
    _capi.check(L.gla_opr_apply(mem._h, _ptr(xd), nx * n, _ptr(zd), ny * n, n, st))
    torch.cuda.synchronize()
    assert not torch.equal(yd, zd)
    assert orc.rel_l2(yd.cpu().numpy(), zd.cpu().numpy()) <= tol
