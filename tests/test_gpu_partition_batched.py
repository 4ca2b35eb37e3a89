"""Partitioned operators with all partitions of a pass in one launch, against
the oracle's partition matvec on the same random Fourier data: several source
partitions (a count that does not fill the thread groups of a workgroup
evenly, more partitions than groups), several target partitions (results in
slots of their own), both at once, unequal axis-3 cell counts in either
direction, odd transform lengths, several right-hand sides and the alpha /
beta form."""
from fractions import Fraction

import ctypes
import numpy as np
import pytest

H = Fraction(1, 32)

# (source partition cells, target partition cells, source divisors, target divisors)
CASES = {
    "src_222": ((4, 6, 10), (6, 4, 8), (2, 2, 2), (1, 1, 1)),
    "src_311_spill": ((2, 4, 30), (4, 2, 6), (3, 1, 1), (1, 1, 1)),
    "src_115": ((6, 2, 6), (2, 6, 24), (1, 1, 5), (1, 1, 1)),
    "trg_123": ((8, 4, 6), (4, 8, 26), (1, 1, 1), (1, 2, 3)),
    "both_21_12": ((4, 4, 58), (4, 6, 58), (2, 1, 1), (1, 2, 1)),
    "both_long": ((2, 2, 150), (2, 2, 106), (1, 2, 1), (2, 1, 1)),
}


def _operator(gila, case, dtype):
    S, T, sdiv, tdiv = CASES[case]
    lat = [H * max(a, b) for a, b in zip(sdiv, tdiv)]
    sS = tuple(m / v for m, v in zip(lat, sdiv))
    sT = tuple(m / v for m, v in zip(lat, tdiv))
    Sf = tuple(c * v for c, v in zip(S, sdiv))
    Tf = tuple(c * v for c, v in zip(T, tdiv))
    vt, vs = gila.GlaVol(Tf, sT), gila.GlaVol(Sf, sS, (0, 0, 400 * H))
    B = tuple((s + t) // 2 for s, t in zip(S, T))
    Ps, Pt = int(np.prod(sdiv)), int(np.prod(tdiv))
    rng = np.random.default_rng(7)
    fur = [(rng.standard_normal(B + (6, Ps, Pt)) + 1j * rng.standard_normal(B + (6, Ps, Pt))).astype(dtype)
           for _ in range(8)]
    mem = gila.GlaOprMem(gila.GlaKerOpt(True), vt, vs, egoFur=fur, setTyp=dtype)
    assert tuple(mem._dims.src_div) == sdiv and tuple(mem._dims.trg_div) == tdiv
    flat = np.concatenate([f.reshape(-1, order="F") for f in fur]).astype(np.complex128)
    return mem, flat, S, T, sdiv, tdiv, Sf, Tf


@pytest.mark.gpu
@pytest.mark.parametrize("case", list(CASES))
@pytest.mark.parametrize("dtype,tol", [(np.complex128, 1e-12), (np.complex64, 1e-5)])
def test_partitions_in_one_launch(gila, orc, gpu, case, dtype, tol):
    import torch
    from gila_amd import _capi
    print(f"case partitions in one launch {case} {np.dtype(dtype).name}", flush=True)
    mem, fur, S, T, sdiv, tdiv, Sf, Tf = _operator(gila, case, dtype)
    L, nrhs = gila.lib(), 2
    st = torch.cuda.current_stream()
    nx, ny = 3 * int(np.prod(Sf)), 3 * int(np.prod(Tf))
    x = [orc.complex_gaussian(Sf + (3,), seed=40 + r).astype(dtype) for r in range(nrhs)]
    y0 = [orc.complex_gaussian(Tf + (3,), seed=50 + r).astype(dtype) for r in range(nrhs)]
    xd = torch.from_numpy(np.concatenate([v.reshape(-1, order="F") for v in x])).cuda()
    y0d = torch.from_numpy(np.concatenate([v.reshape(-1, order="F") for v in y0])).cuda()
    yd, zd = torch.empty_like(y0d), y0d.clone()
    al, be = 0.5 - 1.5j, -0.75 + 0.25j
    _capi.check(L.gla_opr_apply(mem._h, ctypes.c_void_p(xd.data_ptr()), nx * nrhs, ctypes.c_void_p(yd.data_ptr()),
                                ny * nrhs, nrhs, ctypes.c_void_p(st.cuda_stream)))
    _capi.check(L.gla_opr_apply_axpby(mem._h, ctypes.c_void_p(xd.data_ptr()), nx * nrhs,
                                      ctypes.c_void_p(zd.data_ptr()), ny * nrhs, nrhs, al.real, al.imag, be.real,
                                      be.imag, ctypes.c_void_p(st.cuda_stream)))
    one = torch.empty(ny, dtype=yd.dtype, device="cuda")
    _capi.check(L.gla_opr_apply_noalloc(mem._h, ctypes.c_void_p(xd.data_ptr()), nx, ctypes.c_void_p(one.data_ptr()),
                                        ny, 1, ctypes.c_void_p(st.cuda_stream)))
    torch.cuda.synchronize()
    assert torch.equal(one, yd[:ny])
    for r in range(nrhs):
        ref = orc.partition_matvec(S, T, sdiv, tdiv, fur, x[r].astype(np.complex128))
        y = yd[r * ny:(r + 1) * ny].cpu().numpy().reshape(Tf + (3,), order="F")
        z = zd[r * ny:(r + 1) * ny].cpu().numpy().reshape(Tf + (3,), order="F")
        assert orc.rel_l2(y, ref) <= tol
        assert orc.rel_l2(z, al * ref + be * y0[r]) <= tol
