"""Fourier data handed in at branch lengths without a compiled transform is
used as it is given: the longer spectrum it is re-expressed at is its own
mirror image only if the data's self-image entries (frequency 0 and L / 2) of
the components odd in the axis vanish, so mirror storage of G^ may not be
assumed.  Random branches against the oracle, on self operators with every
axis re-embedded and on the symmetric axis of an external pair."""
import numpy as np
import pytest

TOL = {np.complex128: 1e-12, np.complex64: 1e-5}
H = ((1, 32),) * 3

# source cells, target cells, target origin, symmetric axes of the layout
CASES = {
    "self_7_9_11": ((7, 9, 11), (7, 9, 11), (0, 0, 0), (1, 1, 1)),
    "self_14_7_33": ((14, 7, 33), (14, 7, 33), (0, 0, 0), (1, 1, 1)),
    "external_axis_2": ((10, 7, 4), (16, 7, 8), ((1, 2), 0, (3, 4)), (0, 1, 0)),
}


def _operator(gila, orc, case, typ):
    """An operator from random branches."""
    S, T, org, sym = CASES[case]
    B, U = orc.dims(S, T, sym)
    n = U[0] * U[1] * U[2]
    rng = np.random.default_rng(17)
    fur = rng.standard_normal((8, 6, n)) + 1j * rng.standard_normal((8, 6, n))
    fur = fur.astype(typ).reshape(-1)
    src = gila.GlaVol(S, H)
    trg = src if S == T else gila.GlaVol(T, H, org)
    mem = gila.GlaOprMem(gila.GlaKerOpt(True), trg, src, egoFur=orc.fur_branches(fur, U), setTyp=typ)
    assert tuple(mem._dims.brn) == tuple(B) and tuple(mem._dims.dev_brn) != tuple(B)
    return mem, fur.astype(np.complex128), S, T, sym


@pytest.mark.gpu
@pytest.mark.parametrize("case", list(CASES))
@pytest.mark.parametrize("typ", [np.complex128, np.complex64])
def test_any_branches_at_uncompiled_lengths(gila, orc, gpu, case, typ):
    print(f"case any branches {case} {np.dtype(typ).name}", flush=True)
    mem, fur, S, T, sym = _operator(gila, orc, case, typ)
    x = orc.complex_gaussian(S + (3,), seed=71).astype(typ)
    assert orc.rel_l2(gila.egoOpr_(mem, x), orc.matvec(S, T, sym, fur, x.astype(np.complex128))) <= TOL[typ]
