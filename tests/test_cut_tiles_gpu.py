"""Products of few tiles with a long contraction: tiles cut along K on the register-staged kernel, their parts joined through
the workspace, against fp64 and against the same launch without a workspace (nothing is cut)."""
import pytest
import torch

import grouped_mm_bf16_amd.kernels as K_
from grouped_mm_bf16_amd import moe

pytestmark = pytest.mark.gpu
DEV = "cuda"


def launches(run, shape, dtype):
    """Cut twice, whole, cut: the cut results have to be equal bit for bit, and the workspace's counters zero again."""
    outs = []
    for cut in (True, True, False, True):
        out = torch.full(shape, float("nan"), device=DEV, dtype=dtype)
        with K_.tail_split(cut):
            run(out)
        assert K_.last_kernel() == "any" or not cut
        outs.append(out)
    torch.cuda.synchronize()
    stream = torch.cuda.current_stream().cuda_stream
    assert not K_._workspaces[(outs[0].device.index, stream)][:4096].any()
    bits = torch.int32 if dtype == torch.float32 else torch.int16
    for again in (outs[1], outs[3]):
        assert torch.equal(outs[0].view(bits), again.view(bits))
    return outs[0], outs[2]


def check(out, a, b):
    """|fl(sum) - sum| <= (n + 1) u sum |a||b| for n fp32 additions in any order (u = 2^-24), and a 16-bit result's rounding."""
    x, y = a.double(), b.double()
    want, size = x @ y, x.abs() @ y.abs()
    bound = (a.shape[1] + 1) * 2.0 ** -24 * size + (0 if out.dtype == torch.float32 else 2.0 ** -8) * want.abs()
    err = (out.double().cpu() - want).abs()
    assert (err <= bound).all()
    return float(err.norm())


def column(x, on):
    x = x.to(DEV)
    return x.transpose(-2, -1).contiguous().transpose(-2, -1) if on else x


# no element aligned: one tile and many parts, K just past the line, a remainder of one element, tiles at the most that are
# cut (fp32: 64 x 64), parts that make one and several clusters of eight; sizes None: equal products
@pytest.mark.parametrize("a_col,b_col", [(False, False), (False, True), (True, False)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("sizes,M,N,K", [(None, 1, 1, 1025), (None, 129, 127, 4097), ([3, 0, 1, 60, 17], 0, 131, 2049),
                                         ([70] * 3 + [0] * 66, 0, 67, 1601), (None, 33, 1030, 16500)])
def test_unaligned_products(sizes, M, N, K, dtype, a_col, b_col):
    gen = torch.Generator().manual_seed(K + N)
    if sizes is None:
        a, b = torch.randn(2, M, K, generator=gen).to(dtype), torch.randn(2, K, N, generator=gen).to(dtype)
        ad, bd = column(a, a_col), column(b, b_col)
        outs = launches(lambda out: K_.grouped_mm_3d3d(ad, bd, out), (2, M, N), dtype)
        errors = [sum(check(o[g], a[g], b[g]) for g in range(2)) for o in outs]
    else:
        ends = torch.tensor(sizes).cumsum(0).tolist()
        a, b = torch.randn(ends[-1] + 2, K, generator=gen).to(dtype), torch.randn(len(sizes), K, N, generator=gen).to(dtype)
        ad, bd, offs = column(a, a_col), column(b, b_col), torch.tensor(ends, dtype=torch.int32, device=DEV)
        outs = launches(lambda out: K_.grouped_mm_2d3d(ad, bd, offs, out), (ends[-1] + 2, N), dtype)
        errors = [sum(check(o[e - s:e], a[e - s:e], b[g]) for g, (s, e) in enumerate(zip(sizes, ends)) if s) for o in outs]
        assert all(o[ends[-1]:].isnan().all() for o in outs), "rows of no group were written"
    if outs[0].numel() > 1000:                 # cut sums are no further from fp64 than whole ones
        assert errors[0] <= 1.05 * errors[1]


# aligned, both sides of each line of the rule: parts of a tile 16, 8, 5, 4 and fewer; K; full and partly filled tiles
@pytest.mark.parametrize("variant,G,M,N,K,a_col,cut", [
    ("3d3d", 2, 96, 2048, 1032, False, True), ("3d3d", 2, 96, 2048, 1024, False, False), ("3d3d", 3, 104, 1408, 2056, False, True),
    ("3d3d", 3, 104, 1408, 2048, False, False), ("3d3d", 8, 104, 1152, 4096, False, True), ("3d3d", 8, 104, 1152, 4104, False, False),
    ("2d3d", 10, 120, 1280, 1032, False, True), ("2d3d", 10, 120, 1408, 1032, False, False), ("2d3d", 10, 120, 1280, 6152, False, False),
    ("2d3d", 2, 32, 1024, 14336, False, True), ("3d2d", 4, 40, 1024, 2560, True, True), ("3d2d", 4, 40, 1024, 2552, True, False),
    ("3d3d", 3, 520, 1664, 6144, True, True), ("3d3d", 3, 520, 1664, 6152, True, False), ("3d3d", 2, 136, 512, 1272, False, False),
    ("3d3d", 2, 136, 512, 1280, False, True), ("3d3d", 1, 1032, 1024, 3072, False, False), ("3d3d", 1, 1032, 1024, 3080, False, True),
    ("3d3d", 1, 1024, 1024, 2056, False, True), ("3d3d", 1, 1024, 1024, 5128, False, True)])
def test_aligned_products_at_the_lines_of_the_rule(variant, G, M, N, K, a_col, cut):
    gen = torch.Generator().manual_seed(G + K)
    r = lambda *s: torch.randn(*s, generator=gen).bfloat16()
    total = M if variant == "2d3d" else N
    ends = [total * (g + 1) // G // 8 * 8 for g in range(G)]
    offs = None if variant == "3d3d" else torch.tensor(ends, dtype=torch.int32, device=DEV)
    a, b = r(*((M, K) if variant == "2d3d" else (G, M, K))), r(*((K, N) if variant == "3d2d" else (G, K, N)))
    shape = (G, M, N) if variant == "3d3d" else (M, N)
    ad, bd = column(a, a_col), column(b, False)
    args = (ad, bd) if offs is None else (ad, bd, offs)
    out = torch.full(shape, float("nan"), device=DEV, dtype=torch.bfloat16)
    fn = getattr(K_, "grouped_mm_" + variant)
    fn(*args, out)
    assert (K_.last_kernel() == "any") == cut
    assert out.isfinite().all(), "something was not written"
    if cut:
        outs = launches(lambda o: fn(*args, o), shape, torch.bfloat16)
        assert torch.equal(out.view(torch.int16), outs[0].view(torch.int16))
    with K_.tail_split(False):
        fn(*args, torch.empty_like(out))
        assert K_.last_kernel() == "assembly"      # nothing to join the parts in
    for g in range(G):
        lo, hi = ([0] + ends)[g], ends[g]
        if variant == "3d3d":
            check(out[g], a[g], b[g])
        elif variant == "2d3d":
            check(out[lo:hi], a[lo:hi], b[g])
        else:
            check(out[:, lo:hi], a[g], b[:, lo:hi])


def test_gathered_rows_of_cut_tiles():
    """A decoding step's up projection: one row of each of eight groups, rows gathered, one index out of range."""
    gen = torch.Generator().manual_seed(9)
    a, b = torch.randn(3, 2048, generator=gen).bfloat16(), torch.randn(12, 2048, 1536, generator=gen).bfloat16()
    ends = [1, 1, 2, 3, 4, 5, 5, 6, 7, 7, 8, 8]
    idx = torch.tensor([0, 2, 1, 3, 0, 1, 2, 2], dtype=torch.int32)
    ad, bd, offs, rows = a.to(DEV), b.to(DEV), torch.tensor(ends, dtype=torch.int32, device=DEV), idx.to(DEV)
    outs = launches(lambda out: moe.grouped_mm_gathered(ad, rows, bd, offs, out=out), (8, 1536), torch.bfloat16)
    padded = torch.cat([a, torch.zeros(1, 2048).bfloat16()])
    for g, (lo, hi) in enumerate(zip([0] + ends, ends)):
        for out in outs:
            check(out[lo:hi], padded[idx[lo:hi].long()], b[g])
    assert (outs[0][3] == 0).all()


# the last round behind whole ones: 512 workgroups of 128 x 128 tiles, 1024 of 64 x 64 (fp32); tiles past it that are cut, that
# are too many to be cut, none at all; K at the line of 24 K tiles and below it
@pytest.mark.parametrize("dtype,G,M,N,K,cut", [
    (torch.bfloat16, 13, 130, 2570, 1537, True), (torch.float16, 26, 100, 2570, 1601, True), (torch.bfloat16, 16, 250, 2040, 1543, False),
    (torch.bfloat16, 13, 130, 2570, 1535, False), (torch.float32, 26, 130, 2500, 801, True), (torch.float32, 27, 130, 2500, 769, False)])
def test_last_round_behind_whole_ones(dtype, G, M, N, K, cut):
    gen = torch.Generator(device=DEV).manual_seed(K)
    a, b = (torch.randn(*s, device=DEV, generator=gen).to(dtype) for s in ((G, M, K), (G, K, N)))
    out, whole = launches(lambda o: K_.grouped_mm_3d3d(a, b, o), (G, M, N), dtype)
    differ = [not torch.equal(out[g], whole[g]) for g in range(G)]     # the last round's tiles are the last groups'
    assert out.isfinite().all() and any(differ) == cut and not any(differ[:G // 2])
    for g in range(G):
        if g % 5 == 0 or differ[g]:
            check(out[g, :, -700:], a[g].cpu(), b[g, :, -700:].cpu())
    bound = (K + 1) * 2.0 ** -23 * (a.float().abs() @ b.float().abs()) + (0 if dtype == torch.float32 else 2.0 ** -7) * whole.float().abs()
    assert ((out.float() - whole.float()).abs() <= bound).all()       # both within half of that of the exact sum


# 38 rows of 15 tiles, six groups empty; 33 rows of 48 tiles, every group shorter than one
@pytest.mark.parametrize("dtype,sizes,N", [(torch.float16, [256, 0, 41] * 6 + [256] * 7 + [42] * 5 + [43], 1841), (torch.bfloat16, [2, 3] * 13 + [0] + [2] * 7, 6037)])
def test_last_round_with_empty_and_with_short_groups(dtype, sizes, N):
    K, gen = 1601, torch.Generator(device=DEV).manual_seed(N)
    ends = torch.tensor(sizes).cumsum(0).tolist()
    offs = torch.tensor(ends, dtype=torch.int32, device=DEV)
    a, b = (torch.randn(*s, device=DEV, generator=gen).to(dtype) for s in ((ends[-1], K), (len(sizes), K, N)))
    out, whole = launches(lambda o: K_.grouped_mm_2d3d(a, b, offs, o), (ends[-1], N), dtype)
    assert out.isfinite().all() and not torch.equal(out.view(torch.int16), whole.view(torch.int16)), "nothing was cut"
    for g, (s, e) in enumerate(zip(sizes, ends)):
        if s:
            check(out[e - s:e, -400:], a[e - s:e].cpu(), b[g, :, -400:].cpu())
