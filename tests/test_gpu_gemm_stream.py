"""GPU parity of the weight-streaming form of the grouped GEMM (few rows per expert) at the edges of its tiles.

Operands are small integers, so every product and every partial sum is a whole number below 2^24 and the fp32 result is the
same in any order of summation: the outputs have to equal an int64 matmul exactly, no tolerance.  The form computes launches
of few rows per expert, up to four on average or where the panel tiles are not the faster ones, in which few experts have more than 32
rows; `gemm_launch_info` tells, and each test asks it."""
import ctypes

import pytest
import torch

from flux_amd import capi

pytestmark = pytest.mark.gpu
DT = {"bf16": torch.bfloat16, "f16": torch.float16, "fp8": torch.float8_e4m3fn}


def small_ints(gen, *shape):
    return torch.randint(-3, 4, shape, generator=gen)


def expected(a, w, splits, rows_of=None):
    out = torch.zeros(sum(splits), w.shape[1], dtype=torch.int64)
    at = 0
    for e, n in enumerate(splits):
        src = a[at:at + n] if rows_of is None else a[rows_of[at:at + n].long()]
        out[at:at + n] = src @ w[e].t()
        at += n
    return out


def sparse(splits):
    """As many experts without rows as make it four rows per expert on average, which no other form for few rows takes."""
    return splits + [0] * ((sum(splits) + 3) // 4 - len(splits))


def streams(dtype, splits, n, k, block_scaled=False, **kw):
    """The launch's description; no panel tiles, and the streaming form computes it unless too many experts have more than 32 rows."""
    about = dict(block_scaled=block_scaled, **kw)
    assert capi.gemm_launch_info(DT[dtype], len(splits), sum(splits), n, k, panel=True, **about).cols == 0
    info = capi.gemm_launch_info(DT[dtype], len(splits), sum(splits), n, k, splits=splits, **about)
    active, chunks = sum(r > 0 for r in splits), sum((r + 31) // 32 for r in splits)
    few = chunks <= active + (active // 4 if active >= 16 else 0)
    assert info.form == (capi.GEMM_STREAM if few else capi.GEMM_MACRO_TILES) and info.stream_cols in (32, 64)
    return info


# (splits, N, K), all of them on 32-column tiles: one row; 15, 16 and 17 rows; empty experts and more than 64 of them; column tiles
# cut off at 4 columns; K shorter than a line, ending inside one, and over many lines per wave (eight waves).  The macro tiles
# compute the cases with an expert of more than 32 rows: same results where the two forms meet.
CASES = [
    ([1], 4, 16), ([1, 0, 2], 64, 128), (sparse([15, 16, 17]), 100, 272), (sparse([33, 0, 64, 65, 2]), 132, 1040),
    ([0] * 70 + [3, 1] + [0] * 8 + [9], 68, 400), ([7, 5], 1028, 8192 + 48), ([2, 3, 1, 4, 2, 0, 1, 5], 4224, 2064),
    (sparse([40, 1, 22, 30]), 704, 176),
]


@pytest.mark.parametrize("dtype", ["bf16", "f16", "fp8"])
@pytest.mark.parametrize("splits,n,k", CASES)
def test_stream_form_is_exact_on_integers(dtype, splits, n, k):
    print(f"[case] stream gemm {dtype} splits={splits[:6]} n={n} k={k}", flush=True)
    assert streams(dtype, splits, n, k).stream_cols == 32
    g = torch.Generator().manual_seed(n + k)
    m, e = sum(splits), len(splits)
    a, w = small_ints(g, m, k), small_ints(g, e, n, k)
    ad, wd = a.to(torch.float32).to(DT[dtype]).cuda(), w.to(torch.float32).to(DT[dtype]).cuda()
    sp = torch.tensor(splits, dtype=torch.int32, device="cuda")
    ref = expected(a, w, splits)
    got, kind = capi.grouped_gemm(ad, wd, sp, out_dtype=torch.float32, want_kind=True)
    assert kind == 1
    assert torch.equal(got.cpu().long(), ref)
    # rows picked by a gather, results put elsewhere, every scale factor (powers of two) and a second weight tensor
    perm = torch.randperm(m, generator=g).to(torch.int32)
    row_scale = 2.0 ** torch.randint(-1, 2, (m,), generator=g)
    alpha = 2.0 ** torch.randint(-1, 2, (e,), generator=g)
    out = torch.full((m, n), -7.0, device="cuda")
    capi.grouped_gemm(ad, wd, sp, out=out, gather_a=perm.cuda(), scatter_d=perm.flip(0).contiguous().cuda(),
                      row_scale=row_scale.cuda(), alpha=alpha.cuda())
    per_row = torch.repeat_interleave(alpha, torch.tensor(splits)) * row_scale
    want = torch.empty(m, n, dtype=torch.float64)
    want[perm.flip(0).long()] = expected(a, w, splits, perm).double() * per_row[:, None].double()
    assert torch.equal(out.cpu().double(), want)
    two = capi.grouped_gemm_multi(ad, [wd, wd.flip(0).contiguous()] if dtype != "fp8" else [wd, wd], sp, out_dtype=torch.float32)
    assert torch.equal(two[0].cpu().long(), ref)
    assert torch.equal(two[1].cpu().long(), expected(a, w.flip(0) if dtype != "fp8" else w, splits))


@pytest.mark.parametrize("splits,n,k", [([1], 128, 128), (sparse([16, 0, 17, 2]), 256, 384), (sparse([33, 31, 5]), 384, 2048), ([2, 1], 132, 8192)])
@pytest.mark.parametrize("a_layout", [capi.ASCALE_BLOCK128, capi.ASCALE_EXPERT_K_M])
@pytest.mark.parametrize("b_layout", [capi.BSCALE_N_K, capi.BSCALE_K_N])
def test_stream_form_block_scaled_is_exact_on_integers(splits, n, k, a_layout, b_layout):
    print(f"[case] stream gemm block-scaled splits={splits} n={n} k={k} layouts {a_layout} {b_layout}", flush=True)
    streams("fp8", splits, n, k, block_scaled=True)
    g = torch.Generator().manual_seed(n + k)
    m, e, kb, nb = sum(splits), len(splits), k // 128, (n + 127) // 128
    a, w = small_ints(g, m, k), small_ints(g, e, n, k)
    sa = 2.0 ** torch.randint(-1, 2, (m, kb), generator=g)
    sb = 2.0 ** torch.randint(-1, 2, (e, nb, kb), generator=g)
    if a_layout == capi.ASCALE_BLOCK128:
        pad = torch.zeros((m + 127) // 128 * 128, kb)
        pad[:m] = sa
        sad = pad.view(-1, 128, kb).permute(0, 2, 1).contiguous()
    else:
        at, parts = 0, []
        for r in splits:
            parts.append(sa[at:at + r].t().contiguous().flatten())
            at += r
        sad = torch.cat(parts)
    sbd = sb if b_layout == capi.BSCALE_N_K else sb.transpose(1, 2).contiguous()
    got = capi.grouped_gemm_blockscale(a.float().to(DT["fp8"]).cuda(), w.float().to(DT["fp8"]).cuda(),
                                       torch.tensor(splits, dtype=torch.int32, device="cuda"), sad.cuda(), sbd.cuda(), a_layout,
                                       b_layout, out_dtype=torch.float32)
    af = a.double() * torch.repeat_interleave(sa.double(), 128, dim=1)
    wf = w.double() * torch.repeat_interleave(torch.repeat_interleave(sb.double(), 128, dim=1)[:, :n], 128, dim=2)
    at = 0
    for i, r in enumerate(splits):
        assert torch.equal(got[at:at + r].cpu().double(), af[at:at + r] @ wf[i].t()), f"expert {i}"
        at += r


# The 64-column form: more than four rows per expert on average (block-scaled: any), at least 512 column tiles in all, and rows of 4 KiB in
# at least 1024 tiles of 128 columns or too few columns for the panel tiles.  One block and two blocks of 16 rows, rows that do not fill
# them, experts of several chunks of 32 rows; columns cut off at 4; K that ends inside a line and numbers of lines that four waves with
# two lines in flight do not divide; more than 64 experts.  (splits, N, bytes of K)
WIDE = [([32, 0, 31, 17, 16, 1, 2, 9] * 8, 2052, 4096), (([65, 7, 9, 5, 3, 30, 1, 8, 2, 64, 17] + [2] * 8) * 4, 1732, 4096),
        ([32, 0, 31, 17, 16, 1, 2, 9, 5, 20] * 52, 60, 544), ([16, 0, 31, 17, 16, 1, 2, 9, 5, 33] * 52, 60, 4112)]


@pytest.mark.parametrize("dtype", ["bf16", "f16", "fp8"])
@pytest.mark.parametrize("splits,n,kbytes", WIDE)
def test_stream_form_64_columns(dtype, splits, n, kbytes):
    k = kbytes // (1 if dtype == "fp8" else 2)
    print(f"[case] stream gemm, 64 columns {dtype} splits={splits[:6]} n={n} k={k}", flush=True)
    info = streams(dtype, splits, n, k)
    assert (info.form, info.stream_cols, info.stream_waves) == (capi.GEMM_STREAM, 64, 4)
    g = torch.Generator(device="cuda").manual_seed(n + k)
    m, e = sum(splits), len(splits)
    a = torch.randint(-3, 4, (m, k), generator=g, device="cuda").float().to(DT[dtype])
    w = torch.randint(-3, 4, (e, n, k), generator=g, device="cuda", dtype=torch.int8).float().to(DT[dtype])
    sp = torch.tensor(splits, dtype=torch.int32, device="cuda")
    perm = torch.randperm(m, generator=g, device="cuda").to(torch.int32)
    ends = torch.tensor(splits).cumsum(0).tolist()

    def product(a, reverse=False):
        rows = [(end - r, end, i) for r, end, i in zip(splits, ends, range(e)) if r > 0]
        return torch.cat([a[lo:hi].double() @ w[e - 1 - i if reverse else i].double().t().contiguous() for lo, hi, i in rows])

    want = product(a)
    assert torch.equal(capi.grouped_gemm(a, w, sp, out_dtype=torch.float32).double(), want)
    row_scale = 2.0 ** torch.randint(-1, 2, (m,), generator=g, device="cuda").float()
    picked = product(a[perm.long()]) * row_scale.double()[:, None]
    for margin in (0, 40, 1000):
        out = torch.full((m, n), -7.0, device="cuda")
        capi.grouped_gemm(a, w, sp, out=out, gather_a=perm, scatter_d=perm, row_scale=row_scale, cu_margin=margin)
        assert torch.equal(out[perm.long()].double(), picked), f"margin {margin}"
    two = capi.grouped_gemm_multi(a, [w, w.view(torch.uint8).flip(0).contiguous().view(w.dtype)], sp, out_dtype=torch.float32)
    assert torch.equal(two[0].double(), want) and torch.equal(two[1].double(), product(a, reverse=True))


@pytest.mark.parametrize("splits,n,k", [([32, 0, 31, 17, 16, 1, 2, 9], 4164, 384), ([3] * 70 + [0, 32, 1], 516, 1152),
                                        ([65, 7, 9, 5, 3, 30, 1, 8, 2, 64, 17] + [2] * 8, 2052, 384), ([3] * 66 + [70, 33, 0, 96], 580, 256)])
@pytest.mark.parametrize("a_layout", [capi.ASCALE_BLOCK128, capi.ASCALE_EXPERT_K_M])
@pytest.mark.parametrize("b_layout", [capi.BSCALE_N_K, capi.BSCALE_K_N])
def test_stream_form_64_columns_block_scaled(splits, n, k, a_layout, b_layout):
    info = streams("fp8", splits, n, k, block_scaled=True)
    assert (info.form, info.stream_cols) == (capi.GEMM_STREAM, 64)
    test_stream_form_block_scaled_is_exact_on_integers(splits, n, k, a_layout, b_layout)


@pytest.mark.parametrize("dtype", ["bf16", "f16", "fp8"])
@pytest.mark.parametrize("splits,form", [([32, 7, 0, 20, 32, 1], 2), ([33, 7, 0, 20, 31, 1], 1), ([33] * 4 + [0, 1] + [3] * 12, 2),
                                         ([33] * 5 + [0, 1] + [3] * 10, 1), ([130, 0] + [2] * 15, 2), ([0, 0, 0, 0, 0, 90], 1), ([1] * 70 + [600], 1),
                                         ([1] * 70 + [90, 64, 33], 2), ([9, 3, 0, 20], 2)])
def test_one_form_computes_a_launch(dtype, splits, form):
    """Which form runs is decided on the device; every result is computed, and added to a sum, exactly once."""
    print(f"[case] form by splits {dtype} {splits[-6:]}", flush=True)
    splits = sparse(splits)
    n, k, m, e = 260, 272, sum(splits), len(splits)
    assert streams(dtype, splits, n, k).form == form
    assert capi.gemm_launch_info(DT[dtype], e, m, n, k).form == (capi.GEMM_BY_SPLITS if m > 32 else capi.GEMM_STREAM)
    g = torch.Generator().manual_seed(m)
    a, w = small_ints(g, m, k), small_ints(g, e, n, k)
    ad, wd = a.float().to(DT[dtype]).cuda(), w.float().to(DT[dtype]).cuda()
    sp = torch.tensor(splits, dtype=torch.int32, device="cuda")
    ref = expected(a, w, splits)
    assert torch.equal(capi.grouped_gemm(ad, wd, sp, out_dtype=torch.float32).cpu().long(), ref)
    token = torch.randint(0, m // 2 + 1, (m,), generator=g).to(torch.int32)
    sums = torch.zeros(m // 2 + 1, n, dtype=torch.int64).index_add_(0, token.long(), ref)
    out = capi.grouped_gemm_topk_reduce(ad, wd, sp, token.cuda(), m // 2 + 1)
    assert torch.equal(out.cpu(), sums.float().to(out.dtype))


def test_form_follows_the_splits_of_each_replay():
    """A captured launch holds both forms; every replay runs the one that its row counts ask for, as an eager call does."""
    g = torch.Generator().manual_seed(7)
    x = torch.randn(90, 400, generator=g).to(torch.bfloat16).cuda()
    w = (torch.randn(24, 516, 400, generator=g) * 0.05).to(torch.bfloat16).cuda()
    sp, out = torch.zeros(24, dtype=torch.int32, device="cuda"), torch.zeros(90, 516, device="cuda")
    capi.grouped_gemm(x, w, sp, out=out)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        capi.grouped_gemm(x, w, sp, out=out)
    for splits in ([32, 0, 8, 20, 30, 0], [33, 0, 7, 20, 30, 0], [15] * 6, [0, 0, 90, 0, 0, 0], [32, 0, 8, 20, 30, 0]):
        streams("bf16", splits + [0] * 18, 516, 400)
        sp[:6].copy_(torch.tensor(splits, dtype=torch.int32))
        want = capi.grouped_gemm(x, w, sp, out_dtype=torch.float32)
        out.fill_(-1)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)


@pytest.mark.parametrize("dtype", ["bf16", "fp8"])
@pytest.mark.parametrize("splits,n,k", [([9, 10, 8, 11, 7, 9, 10, 10], 2048, 4096), ([2, 0, 3, 1], 4100, 8192 + 16)])
def test_stream_form_weight_groups_have_the_bits_of_one_launch_each(dtype, splits, n, k):
    """One group alone is less than 512 column tiles, the groups together are more."""
    print(f"[case] stream gemm groups {dtype} splits={splits} n={n} k={k}", flush=True)
    g = torch.Generator().manual_seed(n + k)
    x = torch.randn(sum(splits), k, generator=g).to(DT[dtype]).cuda()
    ws = [(torch.randn(len(splits), n, k, generator=g) * 0.05).to(DT[dtype]).cuda() for _ in range(4)]
    sp = torch.tensor(splits, dtype=torch.int32, device="cuda")
    alone = [capi.grouped_gemm(x, w, sp, out_dtype=torch.float32) for w in ws]
    for groups in (2, 3, 4):
        for got, want in zip(capi.grouped_gemm_multi(x, ws[:groups], sp, out_dtype=torch.float32), alone):
            assert torch.equal(got, want)


@pytest.mark.parametrize("kblocks,rows,n,experts", [(1, 3, 128, 1), (3, 3, 128, 1), (7, 3, 256, 2), (8, 3, 128, 1), (9, 3, 128, 1),
                                                    (65, 3, 128, 1), (3, 4, 2176, 24), (9, 4, 2176, 24)])
def test_stream_form_block_scaled_infinite_scales(kblocks, rows, n, experts):
    """An infinite product of scales (each of them finite, or one infinite) makes a result infinite, not NaN, whatever K is
    padded to inside the kernel.  Codes 1 ... 3, so every block's sum is positive; fp32 results, exact integers or +inf."""
    print(f"[case] stream gemm infinite scales kblocks={kblocks} rows={rows} n={n} experts={experts}", flush=True)
    k, m = kblocks * 128, rows * experts
    streams("fp8", [rows] * experts, n, k, block_scaled=True)
    g = torch.Generator().manual_seed(kblocks)
    a, w = torch.randint(1, 4, (m, k), generator=g), torch.randint(1, 4, (experts, n, k), generator=g)
    sa, sb = torch.ones(m, kblocks), torch.ones(experts, n // 128, kblocks)
    sa[1::rows, 0], sb[:, 0, 0] = 2.0 ** 100, 2.0 ** 100  # each row 1 of an expert overflows in its first 128 columns
    sa[2::rows, kblocks - 1] = float("inf")              # each row 2 is infinite everywhere
    pad = torch.zeros((m + 127) // 128 * 128, kblocks)
    pad[:m] = sa
    got = capi.grouped_gemm_blockscale(a.float().to(DT["fp8"]).cuda(), w.float().to(DT["fp8"]).cuda(),
                                       torch.full((experts,), rows, dtype=torch.int32, device="cuda"),
                                       pad.view(-1, 128, kblocks).permute(0, 2, 1).contiguous().cuda(), sb.cuda(),
                                       out_dtype=torch.float32).cpu()
    blocks = torch.einsum("erkc,enkc->ernk", a.view(experts, rows, kblocks, 128).float(), w.view(experts, n, kblocks, 128).float())
    scale = sa.view(experts, rows, 1, kblocks) * torch.repeat_interleave(sb, 128, dim=1).unsqueeze(1)  # fp32: overflows here
    ref = (blocks * scale).sum(-1).view(m, n)
    assert torch.isinf(ref[1, 0]) and torch.isinf(ref[2]).all() and torch.isfinite(ref[0]).all()
    inf = torch.isinf(ref)
    assert torch.equal(torch.isinf(got) & (got > 0), inf)
    assert torch.allclose(got[~inf].double(), ref[~inf].double(), rtol=1e-5, atol=0)


@pytest.mark.parametrize("margin", [1, 100, 255, 1000])
@pytest.mark.parametrize("splits,n,k", [([2, 3, 1, 4, 2, 0, 1, 5], 4224, 2064), ([33, 0, 64, 65, 2], 4096, 528), ([1] * 80, 1028, 400)])
def test_stream_form_leaves_compute_units_and_changes_no_bit(splits, n, k, margin):
    """With `cu_margin` few workgroups walk all items (down to one workgroup); the second case is the panel tiles'."""
    print(f"[case] stream gemm margin={margin} splits={splits[:6]} n={n} k={k}", flush=True)
    g = torch.Generator().manual_seed(n + k)
    a = torch.randn(sum(splits), k, generator=g).to(torch.bfloat16).cuda()
    w = (torch.randn(len(splits), n, k, generator=g) * 0.05).to(torch.bfloat16).cuda()
    sp = torch.tensor(splits, dtype=torch.int32, device="cuda")
    base = capi.grouped_gemm(a, w, sp)
    assert torch.equal(capi.grouped_gemm(a, w, sp, cu_margin=margin), base)


@pytest.mark.parametrize("margin", [1, 249, 1000])
@pytest.mark.parametrize("dtype,splits,n,k", [("fp8", [32, 0, 31, 17, 16, 1, 2, 9], 4164, 272), ("f16", [32, 0, 31, 17, 16, 1, 2, 9], 4164, 272),
                                              ("bf16", [7, 33, 2], 516, 1040), ("fp8", [5, 0, 2], 516, 8192), ("bs", [32, 0, 31, 17, 16, 1, 2, 9], 4160, 384),
                                              ("bs", [3, 1], 260, 8192)])
def test_margin_changes_no_bit_of_any_form(dtype, splits, n, k, margin):
    print(f"[case] stream gemm margin={margin} {dtype} splits={splits} n={n} k={k}", flush=True)
    g = torch.Generator().manual_seed(n + k)
    m, e = sum(splits), len(splits)
    td = DT["fp8" if dtype == "bs" else dtype]
    a = torch.randn(m, k, generator=g).to(td).cuda()
    w = (torch.randn(e, n, k, generator=g) * 0.05).to(td).cuda()
    sp = torch.tensor(splits, dtype=torch.int32, device="cuda")
    if dtype != "bs":
        assert torch.equal(capi.grouped_gemm(a, w, sp, cu_margin=margin), capi.grouped_gemm(a, w, sp))
        return
    sa = torch.rand((m + 127) // 128, k // 128, 128, generator=g).cuda()
    sb = torch.rand(e, (n + 127) // 128, k // 128, generator=g).cuda()
    args, out = capi._gemm_args(a, w, sp, None, None, None, None, None, None, 1.0, None, None, torch.float32, margin, 0, 0)
    capi._check(capi.load().fluxmi_grouped_gemm_blockscale(ctypes.byref(args), capi._ptr(sa), capi.ASCALE_BLOCK128, capi._ptr(sb),
                                                           capi.BSCALE_N_K, capi._stream()), "fluxmi_grouped_gemm_blockscale")
    assert torch.equal(out, capi.grouped_gemm_blockscale(a, w, sp, sa, sb, out_dtype=torch.float32))
