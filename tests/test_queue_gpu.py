"""The tile queue of a jagged contraction: more tiles than workgroups, groups of very different lengths (empty ones
among them), with the counters in the workspace and, without one, dealt round by round."""
import pytest
import torch

import grouped_mm_bf16_amd.kernels as K_
from oracle import grouped_mm_oracle as oracle

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _sizes(groups, total, seed):
    gen = torch.Generator().manual_seed(seed)
    w = torch.exp(2.0 * torch.randn(groups, generator=gen)) * (torch.rand(groups, generator=gen) > 0.2)
    sizes = (w / w.sum() * total).long()
    sizes[int(w.argmax())] += total - int(sizes.sum())
    return sizes


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("a_col,b_col", [(True, False), (False, True), (True, True)])
@pytest.mark.parametrize("groups,M,N", [(70, 312, 528), (300, 256, 64), (9, 1280, 2048), (256, 8, 8), (257, 8, 8),
                                           (512, 72, 8), (513, 8, 8), (3, 40, 72)])
def test_every_tile_once_and_counters_back_at_zero(groups, M, N, a_col, b_col, out_dtype):
    K = 3000
    gen = torch.Generator().manual_seed(groups)
    a = torch.randn(M, K, generator=gen).to(torch.bfloat16)
    b = torch.randn(K, N, generator=gen).to(torch.bfloat16)
    offs = _sizes(groups, K, groups).cumsum(0).to(torch.int32)
    ad = a.t().contiguous().to(DEV).t() if a_col else a.to(DEV)
    bd = b.t().contiguous().to(DEV).t() if b_col else b.to(DEV)
    od = offs.to(DEV)
    with K_.forced_path("mfma"), K_.forced_mfma_config(1):
        outs = []
        for queue in (True, True, False, True):
            out = torch.full((groups, M, N), float("nan"), device=DEV, dtype=out_dtype)
            with K_.tail_split(queue):
                K_.grouped_mm_2d2d(ad, bd, od, out)
            outs.append(out)
        torch.cuda.synchronize()
    bits = torch.int32 if out_dtype == torch.float32 else torch.int16
    for out in outs[1:]:      # a tile's sum does not depend on who runs it, nor when
        assert torch.equal(out.view(bits), outs[0].view(bits))
    ws, nbytes = K_.workspace(od.device, torch.cuda.current_stream().cuda_stream)
    assert nbytes and not K_._workspaces[(od.device.index, torch.cuda.current_stream().cuda_stream)][:4096].any()
    want = oracle.grouped_mm(a, b, offs, out_dtype=out_dtype)
    oracle.assert_close_grouped(outs[0].cpu(), want, a, b, offs, what=f"{groups} groups")
