"""Pass 3 away from the self operator: unequal axis-3 cell counts in either
direction (spill-over and padded results), columns that do not fill a tile,
no mirror storage, several right-hand sides and a partitioned source, at the
lengths whose kernels differ from the general form."""
from fractions import Fraction

import numpy as np
import pytest

TOL = {np.complex128: 1e-12, np.complex64: 1e-5}
H = Fraction(1, 32)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [64, 80, 96, 128, 160, 192])
@pytest.mark.parametrize("typ", [np.complex128, np.complex64])
def test_uneven_axis_3(gila, orc, gpu, n, typ):
    import torch
    from gila_amd import _capi
    for S, T in (((3, 4, n + 14), (7, 2, n - 14)), ((7, 2, 9), (3, 4, 2 * n - 9)), ((20, 1, n), (12, 5, n))):
        print(f"case pass 3 S={S} T={T} {np.dtype(typ).name}", flush=True)
        sym = (0, 0, 0)
        B, U = orc.dims(S, T, sym)
        rng = np.random.default_rng(n)
        m = 48 * int(np.prod(U))
        fur = (rng.standard_normal(m) + 1j * rng.standard_normal(m)).astype(typ)
        src = gila.GlaVol(S, (H,) * 3)
        trg = gila.GlaVol(T, (H,) * 3, (200 * H, 300 * H, 999 * H))
        mem = gila.GlaOprMem(gila.GlaKerOpt(True), trg, src, egoFur=orc.fur_branches(fur, U), setTyp=typ)
        assert tuple(mem._dims.sym) == sym and int(mem._dims.dev_brn[2]) == n
        nrhs = 2
        x = [orc.complex_gaussian(tuple(S) + (3,), seed=n + r).astype(typ) for r in range(nrhs)]
        xd = torch.from_numpy(np.concatenate([v.reshape(-1, order="F") for v in x])).cuda()
        yd = torch.full((nrhs * 3 * int(np.prod(T)),), 7.0, dtype=xd.dtype, device="cuda")
        _capi.check(gila.lib().gla_opr_apply(mem._h, xd.data_ptr(), xd.numel(), yd.data_ptr(), yd.numel(), nrhs,
                                             torch.cuda.current_stream().cuda_stream))
        y = yd.cpu().numpy().reshape(tuple(T) + (3, nrhs), order="F")
        for r in range(nrhs):
            ref = orc.matvec(S, T, sym, fur.astype(np.complex128), x[r].astype(np.complex128))
            assert orc.rel_l2(y[..., r], ref) <= TOL[typ], (S, T, r)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [96, 160, 192])
def test_partitioned_source(gila, orc, gpu, n):
    print(f"case pass 3 partitioned n={n}", flush=True)
    S, T, sdiv, tdiv = (2, 3, n), (4, 3, n), (2, 1, 1), (1, 1, 1)
    Sf = (4, 3, n)
    B = tuple((s + t) // 2 for s, t in zip(S, T))
    rng = np.random.default_rng(n)
    fur = [(rng.standard_normal(B + (6, 2, 1)) + 1j * rng.standard_normal(B + (6, 2, 1))).astype(np.complex64)
           for _ in range(8)]
    mem = gila.GlaOprMem(gila.GlaKerOpt(True), gila.GlaVol(T, (2 * H, H, H)),
                         gila.GlaVol(Sf, (H, H, H), (0, 0, 999 * H)), egoFur=fur, setTyp=np.complex64)
    assert tuple(mem._dims.src_div) == sdiv
    x = orc.complex_gaussian(Sf + (3,), seed=n).astype(np.complex64)
    flat = np.concatenate([f.reshape(-1, order="F") for f in fur]).astype(np.complex128)
    ref = orc.partition_matvec(S, T, sdiv, tdiv, flat, x.astype(np.complex128))
    assert orc.rel_l2(gila.egoOpr_(mem, x), ref) <= 1e-5
