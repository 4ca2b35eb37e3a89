"""The plane kernels (passes 1 + 2 and 4 + 5 of branch lengths up to 64 in one
launch each) against the oracle: every pair of lengths they are built for,
volumes that pad, spill over and crop on axes 1 and 2 (a plane too large for
LDS among them, which takes the five-launch form), several right-hand sides
and the alpha / beta form."""
import ctypes

import numpy as np
import pytest

TOL = {np.complex128: 1e-12, np.complex64: 1e-5}
LENGTHS = [8, 12, 16, 20, 24, 32, 40, 48, 64]


def _mem(gila, orc, S, T, typ):
    """A random operator T <- S with no symmetric axis."""
    sym = (0, 0, 0)
    B, U = orc.dims(S, T, sym)
    rng = np.random.default_rng(11)
    n = 48 * int(np.prod(U))
    fur = (rng.standard_normal(n) + 1j * rng.standard_normal(n)).astype(typ)
    src = gila.GlaVol(S, ((1, 32),) * 3)
    trg = gila.GlaVol(T, ((1, 32),) * 3, ((400, 64), (500, 64), (600, 64)))
    mem = gila.GlaOprMem(gila.GlaKerOpt(True), trg, src, egoFur=orc.fur_branches(fur, U), setTyp=typ)
    assert tuple(mem._dims.sym) == sym and tuple(mem._dims.dev_brn) == tuple(B)
    return mem, fur.astype(np.complex128)


def _check(gila, orc, S, T, typ, nrhs=1, axpby=None):
    import torch
    from gila_amd import _capi
    mem, fur = _mem(gila, orc, S, T, typ)
    x = [orc.complex_gaussian(tuple(S) + (3,), seed=3 + r).astype(typ) for r in range(nrhs)]
    y0 = [orc.complex_gaussian(tuple(T) + (3,), seed=30 + r).astype(typ) for r in range(nrhs)]
    xd = torch.from_numpy(np.concatenate([v.reshape(-1, order="F") for v in x])).cuda()
    yd = torch.from_numpy(np.concatenate([v.reshape(-1, order="F") for v in y0])).cuda()
    st = torch.cuda.current_stream().cuda_stream
    args = (mem._h, xd.data_ptr(), xd.numel(), yd.data_ptr(), yd.numel(), nrhs)
    if axpby is None:
        _capi.check(gila.lib().gla_opr_apply(*args, st))
    else:
        al, be = axpby
        _capi.check(gila.lib().gla_opr_apply_axpby(*args, al.real, al.imag, be.real, be.imag, st))
    y = yd.cpu().numpy().reshape(tuple(T) + (3, nrhs), order="F")
    for r in range(nrhs):
        ref = orc.matvec(S, T, (0, 0, 0), fur, x[r].astype(np.complex128))
        if axpby is not None:
            ref = axpby[0] * ref + axpby[1] * y0[r]
        assert orc.rel_l2(y[..., r], ref) <= TOL[typ], (S, T, r)


@pytest.mark.gpu
@pytest.mark.parametrize("n1", LENGTHS)
@pytest.mark.parametrize("typ", [np.complex128, np.complex64])
def test_every_pair_of_lengths(gila, orc, gpu, n1, typ):
    print(f"case planes n1={n1} {np.dtype(typ).name}", flush=True)
    for n2 in LENGTHS:
        _check(gila, orc, (n1, n2, 2), (n1, n2, 2), typ)


@pytest.mark.gpu
@pytest.mark.parametrize("S,T", [((2, 30, 3), (30, 2, 5)), ((30, 2, 3), (2, 30, 5)), ((46, 17, 1), (18, 47, 3)),
                                 ((3, 127, 2), (29, 1, 2)), ((127, 1, 2), (1, 127, 2))])
@pytest.mark.parametrize("typ", [np.complex128, np.complex64])
def test_pad_spill_and_crop(gila, orc, gpu, S, T, typ):
    print(f"case planes S={S} T={T} {np.dtype(typ).name}", flush=True)
    _check(gila, orc, S, T, typ)
    _check(gila, orc, S, T, typ, nrhs=3, axpby=(0.5 - 1.25j, -0.75 + 2.0j))
