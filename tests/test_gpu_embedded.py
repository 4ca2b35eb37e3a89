"""Axes embedded in a longer transform whose device G^ uses mirror storage:
operators from geometry on cell counts without a fast transform, against the
same product in numpy from the full branches the library hands out -- also
when a Green-data file holds branches without the mirror symmetry, which must
then be used as they are."""
import numpy as np
import pytest

H = (1, 32)


def _numpy_matvec(mem, x):
    d = mem._dims
    S, T, L = tuple(d.src_cel), tuple(d.trg_cel), tuple(2 * int(b) for b in d.dev_brn)
    full = np.zeros(L + (6,), np.complex128)
    for b, f in enumerate(mem.egoFur):
        p = (b >> 2, (b >> 1) & 1, b & 1)
        U = f.shape[:3]
        idx = [np.arange(U[a]) * 2 + p[a] for a in range(3)]
        full[np.ix_(*idx, range(6))] = f
        for a in range(3):                      # stored mirror halves (symmetric axes of the layout)
            assert U[a] == L[a] // 2, "every axis of these operators stores its full branches"
    X = np.fft.fftn(x.astype(np.complex128), L, axes=(0, 1, 2))
    pick = ((0, 3, 4), (3, 1, 5), (4, 5, 2))
    y = np.stack([sum(full[..., pick[c][k]] * X[..., k] for k in range(3)) for c in range(3)], axis=-1)
    return np.fft.ifftn(y, axes=(0, 1, 2))[:T[0], :T[1], :T[2]]


CASES = {
    "self_7_7_9": ((7, 7, 9), None),            # odd and even extended lengths 8, 8, 10
    "self_11_27_14": ((11, 27, 14), None),
    "self_41_7_35": ((41, 7, 35), None),
    "external_axis1": ((14, 6, 9), (14, 8, 13)),   # the same cells on axis 1 only
}


@pytest.mark.gpu
@pytest.mark.parametrize("case", list(CASES))
@pytest.mark.parametrize("typ,tol", [(np.complex128, 1e-12), (np.complex64, 1e-5)])
@pytest.mark.parametrize("broken", [False, True])
def test_embedded_axes(gila, orc, gpu, case, typ, tol, broken, tmp_path):
    print(f"case embedded {case} {np.dtype(typ).name} broken={broken}", flush=True)
    T, S = CASES[case]
    vt = gila.GlaVol(T, (H,) * 3)
    vs = vt if S is None else gila.GlaVol(S, (H,) * 3)
    mem = gila.GlaOprMem(gila.GlaKerOpt(True), vt, vs, setTyp=typ)
    if broken:
        path = tmp_path / "x.gfur"
        mem.save(path)
        raw = bytearray(path.read_bytes())
        n = (len(raw) - 512) // np.dtype(typ).itemsize
        rng = np.random.default_rng(3)
        raw[512:] = (rng.standard_normal(n) + 1j * rng.standard_normal(n)).astype(typ).tobytes()
        h = 1469598103934665603
        for byte in bytes(raw[512:]):
            h = ((h ^ byte) * 1099511628211) & 0xFFFFFFFFFFFFFFFF
        raw[384:392] = h.to_bytes(8, "little")
        path.write_bytes(bytes(raw))
        mem = gila.GlaOprMem.load(path)
    S = T if S is None else S
    if any(int(d) == int(b) for d, b in zip(mem._dims.dev_brn, mem._dims.brn)) and S == T:
        pytest.skip("an axis of this operator is not embedded")
    x = orc.complex_gaussian(S + (3,), seed=5).astype(typ)
    assert orc.rel_l2(gila.egoOpr_(mem, x), _numpy_matvec(mem, x)) <= tol
