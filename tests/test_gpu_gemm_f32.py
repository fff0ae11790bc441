"""moc_gemm_f32 (the small float32 products of the float32 layers) against float64 at the edges of its
32 x 64 tiles and 32-long reduction chunks, in the three forms of a linear layer and its gradients."""

import pytest
import torch

from helpers import gen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ta,tb", [(0, 1), (0, 0), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K", [(1, 4, 8), (31, 60, 24), (33, 68, 40), (32, 64, 256), (200, 256, 264), (640, 512, 256),
                                   (5, 1000, 512), (100, 64, 5), (70, 8, 131)])
def test_gemm_f32(gpu_device, ta, tb, M, N, K):
    from memory_amd import _lib as lib
    if K % 8 and (not ta or tb):
        assert not lib.query("moc_gemm_f32_takes", ta, tb, M, N, K)
        return
    dev = gpu_device
    g = gen(M + N + K)
    a = torch.randn(*((K, M) if ta else (M, K)), generator=g)
    b = torch.randn(*((N, K) if tb else (K, N)), generator=g)
    want = (a.double().t() if ta else a.double()) @ (b.double().t() if tb else b.double())
    ad, bd = a.to(dev), b.to(dev)
    c = torch.full((M + 1, N + 4), 7.0, device=dev)
    lib.call("moc_gemm_f32", ta, tb, M, N, K, ad.data_ptr(), a.shape[1], bd.data_ptr(), b.shape[1], c.data_ptr(), N + 4,
             torch.cuda.current_stream().cuda_stream)
    got = c[:M, :N].double().cpu()
    # K products and sums of unit normals, each rounded once: sqrt(K) 2^-24 per element at most a few times over
    assert ((got - want).norm() / want.norm()).item() < 4 * K ** 0.5 * 2.0 ** -24 + 2.0 ** -23
    assert bool((c[M:] == 7).all()) and bool((c[:, N:] == 7).all()), "writes past the output"


def test_matmul2d_routes(gpu_device):
    """matmul2d gives the library's result for what the small kernel does not take (unaligned or strided
    operands, other types, large sizes)."""
    from memory_amd import ops
    dev = gpu_device
    g = gen(9)
    x, w = torch.randn(50, 40, generator=g).to(dev), torch.randn(36, 40, generator=g).to(dev)
    flat = torch.randn(50 * 40 + 1, generator=g).to(dev)
    for a, b in ((x, w), (x.t().contiguous().t(), w), (flat[1:].view(50, 40), w), (x.bfloat16(), w.bfloat16()),
                 (x.double(), w.double())):
        ref = a.double() @ b.double().t()
        tol = 2e-2 if a.dtype == torch.bfloat16 else 1e-5
        assert ((ops.matmul2d(a, b, tb=True).double() - ref).norm() / ref.norm()).item() < tol
    with pytest.raises(RuntimeError):
        ops.matmul2d(x, w)


def test_recorded_backward_and_autocast(gpu_device):
    """A backward that is itself differentiated, and autocast, keep the library's products."""
    from memory_amd import ops
    dev = gpu_device
    g = gen(4)
    x, w, u = (torch.randn(*s, generator=g).to(dev) for s in ((80, 64), (64, 64), (80, 64)))
    second = []
    for f in (ops.linear, torch.nn.functional.linear):
        a, b = x.clone().requires_grad_(), w.clone().requires_grad_()
        ga, gb = torch.autograd.grad(f(a, b), (a, b), u, create_graph=True)
        (ga.square().sum() + gb.square().sum()).backward()
        second.append((a.grad, b.grad))
    for got, want in zip(*second):
        assert ((got - want).norm() / want.norm()).item() < 1e-5
    with torch.autocast("cuda", torch.bfloat16):
        assert ops.matmul2d(x, w, tb=True).dtype == torch.bfloat16
