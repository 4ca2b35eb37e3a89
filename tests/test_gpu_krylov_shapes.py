"""The Krylov products and updates at the shapes where their kernels change
form: one to more than one sweep of basis vectors, lengths around a workgroup's
step and chunk, odd lengths and strides (element loads) and even ones (16-byte
loads), a view at an odd element offset, no vectors at all."""
import numpy as np
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("dt", ["complex64", "complex128"])
@pytest.mark.parametrize("k,nv,n,off", [(1, 1, 1, 0), (2, 0, 7, 0), (3, 15, 512, 0), (2, 16, 513, 0), (1, 17, 1025, 1),
                                        (2, 33, 2048, 0), (1, 31, 2049, 0), (2, 5, 4098, 1), (1, 3, 2100001, 0)])
def test_products_and_updates(gila, gpu, dt, k, nv, n, off):
    import torch
    print(f"case krylov shapes {dt} k={k} nv={nv} n={n} off={off}", flush=True)
    td = getattr(torch, dt)
    gen = torch.Generator().manual_seed(17)
    flat = torch.randn(k * (nv + 1) * n + off, dtype=td, generator=gen).cuda()
    V = flat[off:].reshape(k, nv + 1, n)[:, :max(nv, 1)] if nv else flat[off:].reshape(k, 1, n)
    w = torch.randn((k, n), dtype=td, generator=gen).cuda()
    ncol = torch.tensor([max(0, nv - r) for r in range(k)], dtype=torch.int64).cuda()
    h = torch.full((k, max(nv, 1)), 9.0, dtype=torch.complex128, device="cuda")[:, :nv].contiguous()
    w2 = torch.full((k,), 9.0, dtype=torch.float64, device="cuda")
    kry, st = gila.solve.KrylovOps(), torch.cuda.current_stream().cuda_stream
    kry.dots(V, k, nv, w, h, st, w2=w2, ncol=ncol)
    V64, w64 = V[:, :nv].cpu().to(torch.complex128), w.cpu().to(torch.complex128)
    use = (torch.arange(nv)[None, :] < ncol.cpu()[:, None]).to(torch.complex128)
    ref = torch.stack([(V64[:, i].conj() * w64).sum(1) for i in range(nv)], 1) * use if nv else torch.zeros((k, 0))
    scale = float(n) ** 0.5
    # FP64 sums of n terms of size one: 1e-14 sqrt(n) bounds their rounding here
    assert (h.cpu() - ref).abs().max().item() <= 1e-13 * scale * 10 if nv else True
    n0 = (w64.abs() ** 2).sum(1)
    assert ((w2.cpu() - n0).abs() / n0).max().item() <= 1e-13
    kry.axpy(V, k, nv, h, w, -0.5, st, w2=w2, ncol=ncol)
    new = w64 - 0.5 * sum((ref[:, i:i + 1] * V64[:, i] for i in range(nv)), torch.zeros_like(w64))
    eps = 1e-6 if dt == "complex64" else 1e-13
    assert (w.cpu().to(torch.complex128) - new).norm().item() <= eps * max(new.norm().item(), w64.norm().item())
    n1 = (w.cpu().to(torch.complex128).abs() ** 2).sum(1)
    assert ((w2.cpu() - n1).abs() / n1).max().item() <= 1e-12
