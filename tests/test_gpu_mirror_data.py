"""Fourier data handed in at branch lengths without a compiled transform is
used as it is given: the longer spectrum it is re-expressed at is its own
mirror image only if the data's self-image entries (frequency 0 and L / 2) of
the components odd in the axis vanish, so mirror storage of G^ may not be
assumed.  Random branches against the oracle, on self operators with every
axis re-embedded or some of them, and on the symmetric axis of an external pair."""
import numpy as np
import pytest

TOL = {np.complex128: 1e-12, np.complex64: 1e-5}
H = ((1, 32),) * 3

# source cells, target cells, target origin, symmetric axes of the layout
CASES = {
    "self_7_9_11": ((7, 9, 11), (7, 9, 11), (0, 0, 0), (1, 1, 1)),
    "self_14_7_33": ((14, 7, 33), (14, 7, 33), (0, 0, 0), (1, 1, 1)),
    "self_14_8_33": ((14, 8, 33), (14, 8, 33), (0, 0, 0), (1, 1, 1)),
    "external_axis_2": ((10, 7, 4), (16, 7, 8), ((1, 2), 0, (3, 4)), (0, 1, 0)),
}


def _operator(gila, orc, case, typ, scale=(1,) * 6):
    """An operator from random branches, component c of them times scale[c]."""
    S, T, org, sym = CASES[case]
    B, U = orc.dims(S, T, sym)
    n = U[0] * U[1] * U[2]
    rng = np.random.default_rng(17)
    fur = rng.standard_normal((8, 6, n)) + 1j * rng.standard_normal((8, 6, n))
    fur = (fur * np.asarray(scale)[None, :, None]).astype(typ).reshape(-1)
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


def _product(opr_mem, x):
    """The product in numpy from the branches an operator hands out."""
    d = opr_mem._dims
    S, T, L = tuple(d.src_cel), tuple(d.trg_cel), tuple(2 * int(b) for b in d.dev_brn)
    full = np.zeros(L + (6,), np.complex128)
    for b, f in enumerate(opr_mem.egoFur):
        at = [np.arange(f.shape[a]) * 2 + ((b >> (2 - a)) & 1) for a in range(3)]
        full[np.ix_(*at, range(6))] = f
    X = np.fft.fftn(x.astype(np.complex128), L, axes=(0, 1, 2))
    pick = ((0, 3, 4), (3, 1, 5), (4, 5, 2))
    y = np.stack([sum(full[..., pick[c][k]] * X[..., k] for k in range(3)) for c in range(3)], axis=-1)
    return np.fft.ifftn(y, axes=(0, 1, 2))[:T[0], :T[1], :T[2]]


@pytest.mark.gpu
@pytest.mark.parametrize("typ,small", [(np.complex128, 1e-13), (np.complex64, 1e-7)])
def test_small_components_are_kept(gila, orc, gpu, typ, small, tmp_path):
    # the xy component random and far below the others' largest entry: a y
    # source's x field is made of it alone, so what the check lets through
    # shows in full; handed in, and read back from a file
    print(f"case small component {np.dtype(typ).name}", flush=True)
    mem, fur, S, T, sym = _operator(gila, orc, "self_7_9_11", typ, (1, 1, 1, small, 0, 0))
    x = np.zeros(S + (3,), dtype=typ)
    x[..., 1] = orc.complex_gaussian(S + (3,), seed=72)[..., 1]
    ref = orc.matvec(S, T, sym, fur, x.astype(np.complex128))
    assert orc.rel_l2(gila.egoOpr_(mem, x)[..., 0], ref[..., 0]) <= TOL[typ]
    path = tmp_path / "x.gfur"
    mem.save(path)
    back = gila.GlaOprMem.load(path)
    assert all(int(u) == int(b) for u, b in zip(back._dims.fur_ext, back._dims.dev_brn))
    assert orc.rel_l2(gila.egoOpr_(back, x)[..., 0], _product(back, x)[..., 0]) <= TOL[typ]
