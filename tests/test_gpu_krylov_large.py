"""Bases larger than the last-level cache, whose vectors the Krylov kernels
read with a hint: bit for bit the results of one right-hand side at a time,
which is below that size.  Odd and even lengths (element and 16-byte loads),
more than one sweep of vectors, column counts."""
import pytest

KEEP = 192 << 20   # bytes


@pytest.mark.gpu
@pytest.mark.parametrize("dt,k,nv,n", [("complex64", 3, 18, 1000002), ("complex64", 3, 18, 1000001),
                                       ("complex128", 3, 17, 600000), ("complex64", 2, 16, 1500000)])
def test_large_basis_matches_single(gila, gpu, dt, k, nv, n):
    import torch
    print(f"case krylov large {dt} k={k} nv={nv} n={n}", flush=True)
    td = getattr(torch, dt)
    per = nv * n * torch.empty(0, dtype=td).element_size()
    assert per <= KEEP < k * per
    gen = torch.Generator(device="cuda").manual_seed(23)
    V = torch.randn((k, nv, n), dtype=td, device="cuda", generator=gen)
    w = torch.randn((k, n), dtype=td, device="cuda", generator=gen)
    ncol = torch.tensor([nv - r for r in range(k)], dtype=torch.int64, device="cuda")
    kry, st = gila.solve.KrylovOps(), torch.cuda.current_stream().cuda_stream

    def step(V, w, ncol):
        k, w = w.shape[0], w.clone()
        h = torch.zeros((k, nv), dtype=torch.complex128, device="cuda")
        n0, n1 = (torch.zeros(k, dtype=torch.float64, device="cuda") for _ in range(2))
        kry.dots(V, k, nv, w, h, st, w2=n0, ncol=ncol)
        kry.axpy(V, k, nv, h, w, -0.5, st, w2=n1, ncol=ncol)
        return h, n0, w, n1

    many = step(V, w, ncol)
    for r in range(k):
        for a, b in zip(many, step(V[r:r + 1], w[r:r + 1], ncol[r:r + 1])):
            assert torch.equal(a[r:r + 1], b), r
