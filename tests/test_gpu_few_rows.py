"""Row counts and widths around the few-row paths of the projections: moc_rows_linear and its residual
form (64 x 32 tiles up to 512 of them, the persistent tiles above, rows off 16-byte alignment) and the K/V
projection and its input gradient on 128 x 256 tiles for few chapters, against float64."""

import pytest
import torch

from helpers import assert_parity, gen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,K", [(768, 768), (256, 256), (512, 1024), (256, 640), (1024, 1536)])
@pytest.mark.parametrize("R", [1, 63, 65, 509, 1400])
@pytest.mark.parametrize("res", [False, True])
def test_rows_linear(gpu_device, N, K, R, res):
    from memory_amd import _lib as lib
    dev = gpu_device
    g = gen(N + K + R)
    x = torch.randn(R, K, generator=g).bfloat16()
    w = (torch.randn(N, K, generator=g) * 0.05).bfloat16()
    r = torch.randn(R, N, generator=g).bfloat16()
    want = x.double() @ w.double().t() + (r.double() if res else 0)
    xd, wd, rd = x.to(dev), w.to(dev), r.to(dev)
    for off in (0, 2):                       # off = 2: rows that start 4 bytes past a 16-byte boundary
        flat = torch.empty(x.numel() + 8, device=dev, dtype=torch.bfloat16)
        xo = flat[off:off + x.numel()].view(R, K)
        xo.copy_(xd)
        y = torch.empty(R, N, device=dev, dtype=torch.bfloat16)
        s = torch.cuda.current_stream().cuda_stream
        if res:
            lib.call("moc_rows_linear_residual", xo.data_ptr(), K, R, wd.data_ptr(), N, K, rd.data_ptr(), N, y.data_ptr(),
                     N, s)
        else:
            lib.call("moc_rows_linear", xo.data_ptr(), K, R, wd.data_ptr(), N, K, y.data_ptr(), N, s)
        assert_parity(y, want, torch.bfloat16, f"R={R} N={N} K={K} off={off}")


@pytest.mark.parametrize("nsel,C,N,K", [(1, 7, 1536, 768), (65, 80, 1536, 768), (9, 12, 512, 1024), (84, 90, 768, 256),
                                         (87, 90, 768, 256)])
@pytest.mark.parametrize("gather", [True, False])
def test_few_chapter_projection(gpu_device, nsel, C, N, K, gather):
    from memory_amd import ops
    dev = gpu_device
    g = gen(nsel + N)
    bank = torch.randn(C * 64, K, generator=g).bfloat16()
    w = (torch.randn(N, K, generator=g) * 0.05).bfloat16()
    ids = torch.randperm(C, generator=g)[:nsel].to(torch.int32)
    plan = ops.chapter_plan(ids.to(dev), C)
    rows = (ids.long().sort().values.unsqueeze(-1) * 64 + torch.arange(64)).reshape(-1)
    x = bank if gather else bank[rows]
    y = ops.chapter_project(x.to(dev), plan, w.to(dev), gather=gather)
    assert_parity(y[: nsel * 64], bank[rows].double() @ w.double().t(), torch.bfloat16, "projection")


@pytest.mark.parametrize("nsel,C,N,K", [(1, 7, 768, 512), (85, 90, 768, 256), (170, 180, 768, 256), (171, 180, 768, 256),
                                         (84, 90, 1536, 512), (86, 90, 1536, 512), (9, 12, 512, 256)])
@pytest.mark.parametrize("bank_rows", [True, False])
def test_few_chapter_input_gradient(gpu_device, nsel, C, N, K, bank_rows):
    """moc_chapter_dx on both sides of its line between 128 x 256 and 256 x 384 tiles ((chapters + 1) / 2 *
    N / 256 against 256 workgroups): 170 chapters are the last of the narrow side at N = 768, 84 at 1,536."""
    from memory_amd import ops
    dev = gpu_device
    g = gen(nsel + N)
    ids = torch.randperm(C, generator=g)[:nsel].to(torch.int32)
    plan = ops.chapter_plan(ids.to(dev), C)
    dkv = torch.randn(nsel * 64, K, generator=g).bfloat16()          # one edge per chapter, in edge order
    wt = (torch.randn(N, K, generator=g) * 0.05).bfloat16()          # [Wk; Wv]^T
    want = dkv.double() @ wt.double().t()                            # edge order
    out = torch.full(((C if bank_rows else nsel) * 64, N), float("nan"), device=dev, dtype=torch.bfloat16)
    ops.chapter_dx(dkv.to(dev), dkv.to(dev), plan.uniq, plan.n_uniq, plan.max_u, plan.csr_off, plan.csr_edge, wt.to(dev),
                   out, bank_rows=bank_rows)
    place = ids.long() if bank_rows else ids.long().argsort().argsort()
    rows = (place.unsqueeze(-1) * 64 + torch.arange(64)).reshape(-1)
    assert_parity(out.cpu()[rows], want, torch.bfloat16, "dx")
    if bank_rows:
        rest = torch.ones(C, dtype=torch.bool)
        rest[ids.long()] = False
        assert bool(torch.isnan(out.cpu().view(C, -1)[rest]).all())
