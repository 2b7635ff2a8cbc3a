"""The register-staged kernel for operands of any alignment, at the sizes where its tiles, K tiles and 16-byte chunks
end: against the CPU oracle (16-bit) and against fp64 with the error bound of an fp32 sum (fp32)."""
import pytest
import torch

from grouped_mm_bf16_amd import kernels as K_
from grouped_mm_bf16_amd import moe
from oracle import grouped_mm_oracle as oracle

pytestmark = pytest.mark.gpu
DEV = "cuda"


def misaligned(t, col, pad):
    """The same values on the GPU, in storage that starts one element into an allocation and ends at the last element
    of the view: row-major (col False) or column-major, leading dimension `pad` elements longer than the row."""
    x = t.transpose(-2, -1) if col else t
    lead, cols = x.shape[:-1], x.shape[-1]
    ld = cols + pad
    rows = 1
    for d in lead:
        rows *= d
    flat = torch.full((1 + rows * ld - pad,), float("nan"), dtype=t.dtype, device=DEV)
    strides = [1]
    step = ld
    for d in reversed(lead):
        strides.insert(0, step)
        step *= d
    view = flat.as_strided(tuple(x.shape), tuple(strides), 1)
    view.copy_(x.to(DEV))
    return view.transpose(-2, -1) if col else view


def compare(got, a, b, offs, what):
    got = got.cpu()
    if a.dtype != torch.float32:
        want = oracle.grouped_mm(a, b, offs, out_dtype=got.dtype)
        assert torch.equal(torch.isnan(got.float()), torch.isnan(want.float())), "ownership differs " + what
        oracle.assert_close_grouped(got, want, a, b, offs, what=what)
        return
    want = oracle.grouped_mm(a, b, offs, out_dtype=torch.float32)
    owned = ~torch.isnan(want)
    assert torch.equal(torch.isnan(got), ~owned), "ownership differs " + what
    # |fl(sum) - sum| <= (K + 1) u sum |a||b| for products and sums in fp32 in any order (u = 2^-24), on both sides
    bound = 2 * (a.shape[-1] + 1) * 2.0 ** -24 * oracle.grouped_mm(a.abs(), b.abs(), offs, out_dtype=torch.float32)
    assert ((got - want).abs()[owned] <= bound[owned]).all(), what


# M / N at the edges of the 128 and 64 tiles and of a chunk, K at the edges of the K tiles (64 or 32 elements)
@pytest.mark.parametrize("a_col,b_col,pad", [(False, False, 0), (True, False, 1), (False, True, 3), (True, True, 0)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("M,K,N", [(129, 65, 127), (9, 1, 9), (63, 31, 257), (128, 129, 1), (1, 200, 65), (300, 33, 7)])
def test_edges_of_tiles_and_chunks(M, K, N, dtype, a_col, b_col, pad):
    gen = torch.Generator().manual_seed(M + K + N)
    a = torch.randn(3, M, K, generator=gen).to(dtype)
    b = torch.randn(3, K, N, generator=gen).to(dtype)
    ad, bd = misaligned(a, a_col, pad), misaligned(b, b_col, pad)
    out = torch.full((3, M, N), float("nan"), device=DEV, dtype=dtype)
    K_.grouped_mm_3d3d(ad, bd, out)
    torch.cuda.synchronize()
    assert K_.last_path() == "generic"
    compare(out, a, b, None, f"3d3d {M}x{K}x{N} {dtype}")


@pytest.mark.parametrize("variant", ["2d3d", "2d2d", "3d2d"])
@pytest.mark.parametrize("dtype,out_dtype", [(torch.bfloat16, torch.bfloat16), (torch.bfloat16, torch.float32),
                                             (torch.float32, torch.float32)])
def test_jagged_edges(variant, dtype, out_dtype):
    """Group boundaries at, before and behind the edges of tiles, K tiles and chunks; elements past the last offset
    belong to nobody and are NaN in every operand."""
    gen = torch.Generator().manual_seed(11)
    sizes = [0, 1, 63, 64, 65, 127, 129, 0, 7, 257]
    G, tot, extra = len(sizes), sum(sizes), 5
    offs = torch.tensor(sizes, dtype=torch.int64).cumsum(0).to(torch.int32)
    r = lambda *s: torch.randn(*s, generator=gen).to(dtype)
    if variant == "2d3d":
        a, b, shape, fn = r(tot + extra, 67), r(G, 67, 131), (tot + extra, 131), K_.grouped_mm_2d3d
        a[tot:] = float("nan")
    elif variant == "2d2d":
        a, b, shape, fn = r(131, tot + extra), r(tot + extra, 67), (G, 131, 67), K_.grouped_mm_2d2d
        a[:, tot:] = float("nan")
        b[tot:] = float("nan")
    else:
        a, b, shape, fn = r(G, 131, 67), r(67, tot + extra), (131, tot + extra), K_.grouped_mm_3d2d
        b[:, tot:] = float("nan")
    for a_col in (False, True):
        for b_col in (False, True):
            out = torch.full(shape, float("nan"), device=DEV, dtype=out_dtype)
            fn(misaligned(a, a_col, 1), misaligned(b, b_col, 1), offs.to(DEV), out)
            torch.cuda.synchronize()
            compare(out, a, b, offs, f"{variant} {dtype} a_col={a_col} b_col={b_col}")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_gathered_rows_without_alignment(dtype):
    """Row indices outside the source read as zeros, inside every tile of a group."""
    gen = torch.Generator().manual_seed(5)
    sizes, S, K, N = [130, 0, 3, 200], 77, 71, 133
    offs = torch.tensor(sizes, dtype=torch.int64).cumsum(0).to(torch.int32)
    a = torch.randn(S, K, generator=gen).to(dtype)
    b = torch.randn(4, K, N, generator=gen).to(dtype)
    idx = torch.randint(0, S, (sum(sizes),), generator=gen).to(torch.int32)
    idx[::17] = -1
    idx[5::41] = S
    rows = torch.zeros(sum(sizes), K, dtype=dtype)
    ok = (idx >= 0) & (idx < S)
    rows[ok] = a[idx[ok].long()]
    got = moe.grouped_mm_gathered(misaligned(a, False, 2), idx.to(DEV), misaligned(b, True, 1), offs.to(DEV))
    torch.cuda.synchronize()
    compare(got, rows, b, offs, f"gathered {dtype}")


def test_operands_smaller_than_a_chunk_and_strided_outputs():
    """Fewer than 8 elements in an operand: the element-wise kernel takes it; an output that is not contiguous along
    its columns goes out element by element."""
    a, b = torch.randn(1, 1, 3).bfloat16(), torch.randn(1, 3, 2).bfloat16()
    out = torch.full((1, 1, 2), float("nan"), device=DEV, dtype=torch.bfloat16)
    K_.grouped_mm_3d3d(a.to(DEV), b.to(DEV), out)
    compare(out, a, b, None, "tiny")
    a, b = torch.randn(2, 70, 33).bfloat16(), torch.randn(2, 33, 130).bfloat16()
    out = torch.full((2, 130, 70), float("nan"), device=DEV, dtype=torch.bfloat16).transpose(1, 2)
    K_.grouped_mm_3d3d(a.to(DEV), b.to(DEV), out)
    compare(out, a, b, None, "column-major output")


# both sides of each line of the rule that leaves small products with a very short contraction to the element-wise kernel:
# K 16 / 17, 256 / 257 tiles of 128 x 128, the operands' types
@pytest.mark.parametrize("G,M,K,N,a_col,dtype,kernel", [
    (16, 212, 5, 9, False, torch.bfloat16, "element"), (3, 129, 16, 131, False, torch.float16, "element"),
    (3, 129, 17, 131, False, torch.float16, "any"), (3, 129, 16, 131, True, torch.bfloat16, "element"), (3, 129, 17, 131, True, torch.bfloat16, "any"),
    (3, 129, 16, 131, False, torch.float32, "any"), (128, 129, 3, 65, False, torch.bfloat16, "element"),
    (257, 63, 3, 65, False, torch.bfloat16, "any"), (4, 2, 2, 3, False, torch.bfloat16, "element")])
def test_very_short_contractions(G, M, K, N, a_col, dtype, kernel):
    gen = torch.Generator().manual_seed(G + M + K + N)
    a, b = torch.randn(G, M, K, generator=gen).to(dtype), torch.randn(G, K, N, generator=gen).to(dtype)
    for b_col in (False, True):
        out = torch.full((G, M, N), float("nan"), device=DEV, dtype=dtype)
        K_.grouped_mm_3d3d(misaligned(a, a_col, 1), misaligned(b, b_col, 1), out)
        assert K_.last_kernel() == kernel
        compare(out, a, b, None, f"{G} of {M}x{K}x{N} {dtype}")


# both sides of each line of the rule that sends small aligned products to these kernels: K 384 / 392 (6 K tiles), rows per
# group 64 / 63 with more than 256 tiles, 128-row tiles times K tiles around 3072, first operand contiguous along M
@pytest.mark.parametrize("variant,G,M,K,N,a_col,small", [
    ("2d3d", 6, 32, 64, 48, False, True), ("2d3d", 3, 200, 384, 136, False, True), ("2d3d", 3, 200, 392, 136, False, False),
    ("2d3d", 70, 4480, 72, 640, False, True), ("2d3d", 70, 4472, 72, 640, False, False), ("2d3d", 70, 4472, 64, 640, False, True),
    ("3d3d", 48, 1000, 64, 1024, False, True), ("3d3d", 49, 1000, 64, 1024, False, False),
    ("3d3d", 4, 136, 1032, 264, True, True), ("3d3d", 3, 40, 2056, 72, True, False),
    ("3d2d", 5, 264, 384, 1000, False, True), ("3d2d", 5, 264, 776, 1000, True, True)])
@pytest.mark.parametrize("dtype,out_dtype", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32)])
def test_small_aligned_products_take_these_kernels(variant, G, M, K, N, a_col, small, dtype, out_dtype):
    gen = torch.Generator().manual_seed(G + M + K + N)
    r = lambda *s: torch.randn(*s, generator=gen).to(dtype)
    col = lambda x, c: x.to(DEV).transpose(-2, -1).contiguous().transpose(-2, -1) if c else x.to(DEV)
    offs = None
    if variant != "3d3d":
        tot = M if variant == "2d3d" else N
        cuts = torch.randint(0, tot + 1, (G,), generator=gen).sort().values
        cuts[-1] = tot - 3                                # the last three rows or columns belong to nobody
        offs = cuts.clamp(max=tot - 3).to(torch.int32)
    if variant == "2d3d":
        a, b, shape, fn = r(M, K), r(G, K, N), (M, N), K_.grouped_mm_2d3d
    elif variant == "3d3d":
        a, b, shape, fn = r(G, M, K), r(G, K, N), (G, M, N), K_.grouped_mm_3d3d
    else:
        a, b, shape, fn = r(G, M, K), r(K, N), (M, N), K_.grouped_mm_3d2d
    for b_col in (False, True):
        ad, bd = col(a, a_col), col(b, b_col)
        args = (ad, bd) if offs is None else (ad, bd, offs.to(DEV))

        def launch():
            out = torch.full(shape, float("nan"), device=DEV, dtype=out_dtype)
            fn(*args, out)
            return out

        got = launch()
        assert K_.last_path() == "mfma" and K_.last_kernel() == ("any" if small else "assembly")
        if small:                                         # the same kernel, so the same bits
            with K_.forced_path("generic"):
                same = launch()
            bits = torch.int32 if out_dtype == torch.float32 else torch.int16
            assert torch.equal(got.view(bits), same.view(bits))
        compare(got, a, b, offs, f"{variant} {dtype} b_col={b_col}")
