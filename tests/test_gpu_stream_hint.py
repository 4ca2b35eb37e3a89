"""Batches whose work planes pass the size from which passes 1, 2, 4 and 5
mark their accesses as not needed again, against the same right-hand sides one
at a time below it: plane kernels and separate passes, ragged and uneven cell
counts, the plain and the alpha / beta epilogue."""
from fractions import Fraction

import numpy as np
import pytest

H = Fraction(1, 32)
LINE = 192 << 20   # bytes of work planes


@pytest.mark.gpu
@pytest.mark.parametrize("typ", [np.complex64, np.complex128])
@pytest.mark.parametrize("S,T,planes", [((30, 41, 13), (34, 39, 19), True), ((45, 101, 31), (35, 91, 17), False),
                                        ((7, 64, 15), (9, 96, 33), False)])
def test_batch_matches_single(gila, orc, gpu, typ, S, T, planes):
    import torch
    from gila_amd import _capi
    B = tuple((s + t) // 2 for s, t in zip(S, T))
    cb = np.dtype(typ).itemsize
    z = max(S[2], T[2])
    w1, w2 = (6 * B[0] * max(S[1], T[1]) * z, 12 * B[0] * B[1] * z)
    per = (w2 if planes else w1 + w2) * cb
    nrhs = -(-LINE // per)
    print(f"case stream hint S={S} T={T} {np.dtype(typ).name} nrhs={nrhs}", flush=True)
    assert per < LINE <= nrhs * per
    rng = np.random.default_rng(3)
    m = 48 * int(np.prod(B))
    fur = (rng.standard_normal(m) + 1j * rng.standard_normal(m)).astype(typ)
    mem = gila.GlaOprMem(gila.GlaKerOpt(True), gila.GlaVol(T, (H,) * 3, (200 * H, 300 * H, 999 * H)),
                         gila.GlaVol(S, (H,) * 3), egoFur=orc.fur_branches(fur, B), setTyp=typ)
    assert tuple(mem._dims.dev_brn) == B and tuple(mem._dims.sym) == (0, 0, 0)
    td = torch.complex64 if typ is np.complex64 else torch.complex128
    gen = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn((nrhs, 3 * int(np.prod(S))), dtype=td, device="cuda", generator=gen)
    y0 = torch.randn((nrhs, 3 * int(np.prod(T))), dtype=td, device="cuda", generator=gen)
    s = torch.cuda.current_stream().cuda_stream
    lib = gila.lib()

    def run(xs, ys, n, scaled):
        a = (mem._h, xs.data_ptr(), xs.numel(), ys.data_ptr(), ys.numel(), n)
        _capi.check(lib.gla_opr_apply_axpby(*a, 0.5, -1.0, 2.0, 0.25, s) if scaled else lib.gla_opr_apply(*a, s))

    for scaled in (False, True):
        many, one = y0.clone(), y0.clone()
        run(x, many, nrhs, scaled)
        for r in range(nrhs):
            run(x[r], one[r], 1, scaled)
        # the same sums at most reordered: 24 transform stages of eps each
        err = ((many - one).abs().norm(dim=1) / one.abs().norm(dim=1)).max().item()
        assert err <= 24 * np.finfo(typ).eps, (scaled, err)
