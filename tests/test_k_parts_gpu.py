"""Jagged contractions whose groups are cut along K: parts, clusters of parts and their counters, against fp64 and against
the same launch without a workspace (nothing is cut)."""
import pytest
import torch

import grouped_mm_bf16_amd.kernels as K_

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _launches(a, b, offs, shape, out_dtype):
    outs = []
    for cut in (True, True, False, True):
        out = torch.full(shape, float("nan"), device=DEV, dtype=out_dtype)
        with K_.tail_split(cut), K_.forced_path("generic"):
            K_.grouped_mm_2d2d(a, b, offs, out)
        outs.append(out)
    torch.cuda.synchronize()
    stream = torch.cuda.current_stream().cuda_stream
    assert K_.workspace(a.device, stream)[1] and not K_._workspaces[(a.device.index, stream)][:4096].any()
    bits = torch.int32 if out_dtype == torch.float32 else torch.int16
    for again in (outs[1], outs[3]):       # the sum does not depend on which part comes last
        assert torch.equal(outs[0].view(bits), again.view(bits))
    return outs


# group lengths at the edges of a part (256 elements or an even share), of a cluster (8 parts: 2048) and of the most parts
# a group has (64: 16384); elements past the last offset belong to nobody and are NaN
@pytest.mark.parametrize("a_col,b_col", [(True, False), (False, True), (False, False), (True, True)])
@pytest.mark.parametrize("dtype,out_dtype", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32),
                                             (torch.float32, torch.float32)])
@pytest.mark.parametrize("sizes,M,N,extra", [([256, 257, 0, 1, 511, 513, 2048, 2049], 32, 64, 5),
                                             ([0, 16384, 16385, 30], 17, 130, 8), ([4097], 200, 136, 0),
                                             ([40] * 69 + [2200, 0], 136, 72, 3)])
def test_parts_add_up(sizes, M, N, extra, dtype, out_dtype, a_col, b_col):
    gen = torch.Generator().manual_seed(len(sizes) + M)
    tot, G = sum(sizes), len(sizes)
    a = torch.randn(M, tot + extra, generator=gen).to(dtype)
    b = torch.randn(tot + extra, N, generator=gen).to(dtype)
    a[:, tot:], b[tot:] = float("nan"), float("nan")
    offs = torch.tensor(sizes).cumsum(0).to(torch.int32)
    ad = a.to(DEV).t().contiguous().t() if a_col else a.to(DEV)
    bd = b.to(DEV).t().contiguous().t() if b_col else b.to(DEV)
    outs = _launches(ad, bd, offs.to(DEV), (G, M, N), out_dtype)
    # |fl(sum) - sum| <= (n + 1) u sum |a||b| in any order of n fp32 additions (u = 2^-24), here against fp64;
    # plus the rounding of a 16-bit result (2^-8 of the value)
    ends = [0] + offs.tolist()
    for g in range(G):
        x, y = a[:, ends[g]:ends[g + 1]].double(), b[ends[g]:ends[g + 1]].double()
        want, size = x @ y, x.abs() @ y.abs()
        bound = (sizes[g] + 1) * 2.0 ** -24 * size + (0 if out_dtype == torch.float32 else 2.0 ** -8) * want.abs()
        for out in (outs[0], outs[2]):
            assert ((out[g].double().cpu() - want).abs() <= bound).all(), f"group {g} of {sizes[g]}"


@pytest.mark.parametrize("G", [60, 100])       # the table of the groups in registers, and in LDS
def test_offsets_that_overlap_are_not_cut(G):
    """Offsets that go back: more parts than the workspace has counters for, so the launch runs uncut."""
    K, M, N = 32768, 32, 64
    gen = torch.Generator().manual_seed(3)
    a = torch.randn(M, K, generator=gen).bfloat16().to(DEV)
    b = torch.randn(K, N, generator=gen).bfloat16().to(DEV)
    offs = torch.tensor([K, 0] * (G // 2), dtype=torch.int32, device=DEV)
    assert G // 2 * 64 > 1020                  # parts of the groups that hold all of K, counters
    outs = _launches(a, b, offs, (G, M, N), torch.bfloat16)
    assert torch.equal(outs[0].view(torch.int16), outs[2].view(torch.int16))
    x, y = a.cpu().double(), b.cpu().double()
    want, size = x @ y, x.abs() @ y.abs()
    bound = (K + 1) * 2.0 ** -24 * size + 2.0 ** -8 * want.abs()     # as above
    got = outs[0].double().cpu()
    assert ((got[0::2] - want).abs() <= bound).all()
    assert (outs[0][1::2] == 0).all()          # [K, 0): empty
