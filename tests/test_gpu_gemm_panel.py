"""GPU parity of the panel tiles of the grouped GEMM (up to about 96 rows per expert) at the edges of their tiles.

Operands are small integers and scales powers of two, so every product and every partial sum is a whole multiple of a power of two
below 2^24 steps: the fp32 result is the same in any order of summation and has to equal a float64 matmul exactly, no tolerance."""
import ctypes
import random

import pytest
import torch

from flux_amd import capi

pytestmark = pytest.mark.gpu
DT = {"bf16": torch.bfloat16, "f16": torch.float16, "fp8": torch.float8_e4m3fn, "bs": torch.float8_e4m3fn}


def spread(lo, hi, experts, seed):
    rng = random.Random(seed)
    return [lo, hi] + [rng.randint(lo, hi) for _ in range(experts - 2)]


# (name, splits, N, K, columns, rows of a chunk): every instance of the tiles, with chunks at both sides of 32, 64, 96 and 128 rows, empty
# experts and more than 64 of them, columns cut off at 4 (the last wave's moved back, also past a whole wave), K shorter than a line,
# ending inside one, and of as many lines as the rings have stages and more.
CASES = [
    ("64 columns, 32 rows", [32, 0, 31, 17, 16, 1, 2, 9], 4164, 272, 64, 32),
    ("64 columns, 32 rows, lines in pairs", [32, 0, 31, 17, 16, 1, 2, 9], 4164, 3216, 64, 32),
    ("128 columns, 32 rows", [1, 32, 16, 17] + [0] * 3 + [5] * 123, 1028, 144, 128, 32),
    ("64 columns, 64 rows", [64, 65, 1, 0, 16, 97, 33, 130], 132, 272, 64, 64),
    ("64 columns, 64 rows, all on one", [0, 0, 300, 0], 68, 16, 64, 64),
    ("64 columns, 128 rows, small", [150, 129, 300, 1, 128], 132, 272, 64, 128),
    ("128 columns, 64 rows", spread(1, 64, 70, 1), 580, 400, 128, 64),
    ("256 columns", spread(33, 128, 70, 2), 1540, 400, 256, 128),
    ("256 columns, short K", [64, 96, 128, 65, 97, 48] + [50] * 64, 1540, 48, 256, 128),
    ("128 columns, 128 rows", spread(1, 128, 24, 3), 1412, 1040, 128, 128),
    ("64 columns, 128 rows", [32, 33, 64, 65, 96, 97, 128, 0], 1092, 8192 + 16, 64, 128),
]
# In none of these K is whole lines of 128 bytes; in the same ones with K cut to a multiple of 128 (one line at least) it is, in every type, and
# the weights' loads are the non-temporal ones.
LINES = [(name + ", whole lines", splits, n, max(128, k // 128 * 128), cols, chunk) for name, splits, n, k, cols, chunk in CASES]


def made(splits, n, k, dtype, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    m, e = sum(splits), len(splits)
    a = torch.randint(-3, 4, (m, k), generator=g, device="cuda").float()
    w = torch.randint(-3, 4, (e, n, k), generator=g, device="cuda").float()
    return a, w, torch.tensor(splits, dtype=torch.int32, device="cuda"), g


def product(a, w, splits):
    out, at = [], 0
    for e, r in enumerate(splits):
        out.append(a[at:at + r].double() @ w[e].double().t().contiguous())
        at += r
    return torch.cat(out)


@pytest.mark.parametrize("dtype", ["bf16", "f16", "fp8"])
@pytest.mark.parametrize("name,splits,n,k,cols,chunk", CASES + LINES, ids=[c[0] for c in CASES + LINES])
def test_panel_tiles_are_exact_on_integers(name, splits, n, k, cols, chunk, dtype):
    print(f"[case] panel gemm {dtype} {name} n={n} k={k}", flush=True)
    assert (k * DT[dtype].itemsize % 128 == 0) == name.endswith("whole lines")
    m, e = sum(splits), len(splits)
    info = capi.gemm_launch_info(DT[dtype], e, m, n, k, splits=splits, panel=True)
    assert (info.cols, info.chunk_rows, info.computes) == (cols, chunk, 1)
    a, w, sp, g = made(splits, n, k, dtype, n + k)
    ad, wd = a.to(DT[dtype]), w.to(DT[dtype])
    assert torch.equal(capi.grouped_gemm(ad, wd, sp, out_dtype=torch.float32).double(), product(a, w, splits))
    # rows picked by a gather, results put elsewhere, every scale factor, a second weight tensor, margins
    perm = torch.randperm(m, generator=g, device="cuda").to(torch.int32)
    to = perm.flip(0).contiguous()
    row_scale = 2.0 ** torch.randint(-1, 2, (m,), generator=g, device="cuda").float()
    col_scale = 2.0 ** torch.randint(-1, 2, (e, n), generator=g, device="cuda").float()
    alpha = 2.0 ** torch.randint(-1, 2, (e,), generator=g, device="cuda").float()
    expert = torch.repeat_interleave(torch.arange(e, device="cuda"), sp.long())
    want = torch.empty(m, n, dtype=torch.float64, device="cuda")
    want[to.long()] = product(a[perm.long()], w, splits) * (alpha[expert] * row_scale).double()[:, None] * col_scale[expert].double()
    for margin in (0, 40, 250, 1000):
        out = torch.full((m, n), -7.0, device="cuda")
        capi.grouped_gemm(ad, wd, sp, out=out, gather_a=perm, scatter_d=to, row_scale=row_scale, col_scale=col_scale, alpha=alpha, cu_margin=margin)
        assert torch.equal(out.double(), want), f"margin {margin}"
    two = capi.grouped_gemm_multi(ad, [wd, wd.flip(0).contiguous()] if dtype != "fp8" else [wd, wd], sp, out_dtype=torch.float32)
    assert torch.equal(two[0].double(), product(a, w, splits))
    assert torch.equal(two[1].double(), product(a, w.flip(0) if dtype != "fp8" else w, splits))
    # added to sums: every result once
    token = torch.randint(0, m // 2 + 1, (m,), generator=g, device="cuda")
    sums = torch.zeros(m // 2 + 1, n, dtype=torch.float64, device="cuda").index_add_(0, token, product(a, w, splits))
    assert torch.equal(capi.grouped_gemm_topk_reduce(ad, wd, sp, token.to(torch.int32), m // 2 + 1), sums.float().to(capi._half_out(ad.dtype)))


BLOCK_SCALED = [
    ("64 columns, 32 rows", [32, 0, 31, 17, 16, 1, 2, 9], 4160, 384, 64, 32),
    ("64 columns, 32 rows, lines in pairs", [32, 0, 31, 17, 16, 1, 2, 9], 4160, 6272, 64, 32),
    ("128 columns, 32 rows", [1, 32, 16, 17] + [0] * 3 + [5] * 123, 1088, 256, 128, 32),
    ("64 columns, 64 rows", [64, 65, 1, 0, 16, 97, 33, 130], 192, 384, 64, 64),
    ("128 columns, 64 rows", spread(1, 64, 70, 1), 640, 640, 128, 64),
    ("128 columns, 128 rows", spread(1, 128, 24, 3), 1408, 1152, 128, 128),
    ("64 columns, 128 rows", [32, 33, 64, 65, 96, 97, 128, 0], 1088, 8192, 64, 128),
]


def block_scales(m, e, n, k, splits, a_layout, b_layout, g):
    kb, nb = k // 128, (n + 127) // 128
    sa = 2.0 ** torch.randint(-1, 2, (m, kb), generator=g, device="cuda").float()
    sb = 2.0 ** torch.randint(-1, 2, (e, nb, kb), generator=g, device="cuda").float()
    if a_layout == capi.ASCALE_BLOCK128:
        pad = torch.zeros((m + 127) // 128 * 128, kb, device="cuda")
        pad[:m] = sa
        sad = pad.view(-1, 128, kb).permute(0, 2, 1).contiguous()
    else:
        at, parts = 0, []
        for r in splits:
            parts.append(sa[at:at + r].t().contiguous().flatten())
            at += r
        sad = torch.cat(parts)
    return sa, sb, sad, (sb if b_layout == capi.BSCALE_N_K else sb.transpose(1, 2).contiguous())


@pytest.mark.parametrize("name,splits,n,k,cols,chunk", BLOCK_SCALED, ids=[c[0] for c in BLOCK_SCALED])
@pytest.mark.parametrize("a_layout", [capi.ASCALE_BLOCK128, capi.ASCALE_EXPERT_K_M])
@pytest.mark.parametrize("b_layout", [capi.BSCALE_N_K, capi.BSCALE_K_N])
def test_panel_tiles_block_scaled_are_exact_on_integers(name, splits, n, k, cols, chunk, a_layout, b_layout):
    print(f"[case] panel gemm block-scaled {name} n={n} k={k} layouts {a_layout} {b_layout}", flush=True)
    m, e = sum(splits), len(splits)
    info = capi.gemm_launch_info(DT["bs"], e, m, n, k, splits=splits, panel=True, block_scaled=True)
    if name != "64 columns, 128 rows":
        assert (info.cols, info.chunk_rows, info.computes) == (cols, chunk, 1)
    a, w, sp, g = made(splits, n, k, "fp8", n + k)
    sa, sb, sad, sbd = block_scales(m, e, n, k, splits, a_layout, b_layout, g)
    af = a * torch.repeat_interleave(sa, 128, dim=1)
    wf = w * torch.repeat_interleave(torch.repeat_interleave(sb, 128, dim=1)[:, :n], 128, dim=2)
    want = product(af, wf, splits)
    ad, wd = a.to(DT["bs"]), w.to(DT["bs"])
    assert torch.equal(capi.grouped_gemm_blockscale(ad, wd, sp, sad, sbd, a_layout, b_layout, out_dtype=torch.float32).double(), want)
    if a_layout == capi.ASCALE_BLOCK128:  # rows, and their scales, picked by a gather
        perm = torch.randperm(m, generator=g, device="cuda").to(torch.int32)
        got = capi.grouped_gemm_blockscale(ad, wd, sp, sad, sbd, a_layout, b_layout, out_dtype=torch.float32, gather_a=perm)
        assert torch.equal(got.double(), product(af[perm.long()], wf, splits))
    for margin in (40, 1000):
        args, out = capi._gemm_args(ad, wd, sp, None, None, None, None, None, None, 1.0, None, None, torch.float32, margin, 0, 0)
        capi._check(capi.load().fluxmi_grouped_gemm_blockscale(ctypes.byref(args), capi._ptr(sad), a_layout, capi._ptr(sbd), b_layout, capi._stream()),
                    "fluxmi_grouped_gemm_blockscale")
        assert torch.equal(out.double(), want), f"margin {margin}"


@pytest.mark.parametrize("kblocks,rows,n,experts", [(1, 40, 128, 4), (2, 40, 640, 70), (3, 70, 1408, 24), (9, 90, 192, 3), (17, 5, 2176, 24), (49, 5, 2176, 24)])
def test_panel_tiles_infinite_scales(kblocks, rows, n, experts):
    """An infinite product of scales makes a result infinite, not NaN, whatever K is padded to inside the kernel."""
    print(f"[case] panel gemm infinite scales kblocks={kblocks} rows={rows} n={n} experts={experts}", flush=True)
    k, m = kblocks * 128, rows * experts
    assert capi.gemm_launch_info(DT["bs"], experts, m, n, k, panel=True, block_scaled=True).cols > 0
    g = torch.Generator(device="cuda").manual_seed(kblocks)
    a, w = (torch.randint(1, 4, s, generator=g, device="cuda").float() for s in ((m, k), (experts, n, k)))
    sa, sb = torch.ones(m, kblocks, device="cuda"), torch.ones(experts, (n + 127) // 128, kblocks, device="cuda")
    sa[1::rows, 0], sb[:, 0, 0] = 2.0 ** 100, 2.0 ** 100  # row 1 of an expert overflows in its first 128 columns
    sa[2::rows, kblocks - 1] = float("inf")              # row 2 is infinite everywhere
    pad = torch.zeros((m + 127) // 128 * 128, kblocks, device="cuda")
    pad[:m] = sa
    got = capi.grouped_gemm_blockscale(a.to(DT["bs"]), w.to(DT["bs"]), torch.full((experts,), rows, dtype=torch.int32, device="cuda"),
                                       pad.view(-1, 128, kblocks).permute(0, 2, 1).contiguous(), sb, out_dtype=torch.float32)
    assert not torch.isnan(got).any()
    inf = torch.zeros(experts, rows, n, dtype=torch.bool, device="cuda")
    inf[:, 1, :128] = True
    inf[:, 2] = True
    assert torch.equal(torch.isinf(got) & (got > 0), inf.view(m, n))


MORE_ROWS = [c for c in CASES + LINES if sum(c[1]) > 32 * len(c[1])]  # (with fewer rows they have the streaming form's bits, below)


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("name,splits,n,k,cols,chunk", MORE_ROWS, ids=[c[0] for c in MORE_ROWS])
def test_panel_tiles_have_the_bits_of_the_macro_tiles(name, splits, n, k, cols, chunk, dtype):
    """16-bit operands: the same rows among so many others that the macro tiles compute the launch."""
    print(f"[case] panel gemm bits {dtype} {name} n={n} k={k}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(n)
    more = [r + 200 for r in splits]
    assert capi.gemm_launch_info(DT[dtype], len(splits), sum(more), n, k, panel=True).cols == 0
    x = torch.randn(sum(more), k, generator=g, device="cuda").to(DT[dtype])
    w = (torch.randn(len(splits), n, k, generator=g, device="cuda") * 0.05).to(DT[dtype])
    starts = torch.tensor([0] + more).cumsum(0)[:-1]
    rows = torch.cat([torch.arange(s, s + r) for s, r in zip(starts.tolist(), splits)]).cuda()
    many = capi.grouped_gemm(x, w, torch.tensor(more, dtype=torch.int32, device="cuda"), out_dtype=torch.float32)
    few = capi.grouped_gemm(x[rows], w, torch.tensor(splits, dtype=torch.int32, device="cuda"), out_dtype=torch.float32)
    assert torch.equal(few, many[rows])


# (name, splits, N, bytes of K, columns, rows of a chunk, waves over which the streaming form splits K): launches of few rows per
# expert, which both forms take.  Numbers of lines that four and eight sums do not divide.
FEW_ROWS = [
    ("64 columns, 32 rows", [32, 0, 31, 17, 16, 1, 2, 9], 4164, 544, 64, 32, 4),
    ("64 columns, 32 rows, lines in pairs", [32, 0, 31, 17, 16, 1, 2, 9], 4164, 6432, 64, 32, 4),
    ("128 columns, 32 rows", [1, 32, 16, 17] + [0] * 3 + [5] * 123, 1028, 800, 128, 32, 4),
    ("64 columns, 64 rows", [20, 32, 17, 26], 192, 2080, 64, 64, 4),
    ("128 columns, 64 rows", [20] * 62 + [17, 32], 2052, 800, 128, 64, 4),
    ("64 columns, 64 rows, eight sums, small", [20, 24, 28, 18], 192, 16416, 64, 64, 8),
    ("64 columns, 64 rows, eight sums", [20, 24, 28, 18], 4096, 16416, 64, 64, 8),
]
FEW_ROWS += [(name + ", whole lines", splits, n, kbytes // 128 * 128, *form) for name, splits, n, kbytes, *form in FEW_ROWS]


def random_operands(splits, n, k, dtype, groups=1):
    """x, w for each group, and run(rows, splits, weights): the fp32 results of these rows of x."""
    g = torch.Generator(device="cuda").manual_seed(n + k)
    m, e = sum(splits), len(splits)
    x = torch.randn(m, k, generator=g, device="cuda").to(DT[dtype])
    ws = [(torch.randn(e, n, k, generator=g, device="cuda") * (1.0 if dtype in ("fp8", "bs") else 0.05)).to(DT[dtype]) for _ in range(groups)]
    sa = torch.rand(m, k // 128, generator=g, device="cuda") + 0.5
    sb = torch.rand(e, (n + 127) // 128, k // 128, generator=g, device="cuda") + 0.5

    def run(rows, counts, w):
        sp = torch.tensor(counts, dtype=torch.int32, device="cuda")
        if dtype != "bs":
            return capi.grouped_gemm(x[rows], w, sp, out_dtype=torch.float32)
        pad = torch.zeros((len(rows) + 127) // 128 * 128, k // 128, device="cuda")
        pad[:len(rows)] = sa[rows]
        return capi.grouped_gemm_blockscale(x[rows], w, sp, pad.view(-1, 128, k // 128).permute(0, 2, 1).contiguous(), sb, out_dtype=torch.float32)

    return x, ws, run


@pytest.mark.parametrize("dtype", ["bf16", "f16", "fp8", "bs"])
@pytest.mark.parametrize("name,splits,n,kbytes,cols,chunk,waves", FEW_ROWS, ids=[c[0] for c in FEW_ROWS])
def test_few_rows_have_the_bits_of_the_streaming_form(name, splits, n, kbytes, cols, chunk, waves, dtype):
    """A result is the same sum of partial sums over K in both forms (one chain would be less precise): the rows, four of each expert at a
    time, in launches that the streaming form computes."""
    k = kbytes // (2 if dtype in ("bf16", "f16") else 1)
    if dtype == "bs":
        n, k = (n + 127) // 128 * 128, (k + 127) // 128 * 128
    print(f"[case] panel gemm, streaming form's bits {dtype} {name} n={n} k={k}", flush=True)
    m, e, bs = sum(splits), len(splits), dtype == "bs"
    info = capi.gemm_launch_info(DT[dtype], e, m, n, k, splits=splits, panel=True, block_scaled=bs)
    assert (info.cols, info.chunk_rows, info.computes) == (cols, chunk, 1)
    _, (w,), run = random_operands(splits, n, k, dtype)
    got = run(torch.arange(m, device="cuda"), splits, w)
    starts = torch.tensor([0] + splits).cumsum(0).tolist()
    for first in range(0, max(splits), 4):
        counts = [max(0, min(4, r - first)) for r in splits]
        rows = torch.cat([torch.arange(s + first, s + first + c) for s, c in zip(starts, counts)]).cuda()
        assert capi.gemm_launch_info(DT[dtype], e, len(rows), n, k, panel=True, block_scaled=bs).cols == 0
        part = capi.gemm_launch_info(DT[dtype], e, len(rows), n, k, splits=counts, block_scaled=bs)
        assert (part.form, part.stream_waves) == (capi.GEMM_STREAM, waves)
        assert torch.equal(got[rows], run(rows, counts, w)), f"rows {first} to {first + 3} of each expert"


@pytest.mark.parametrize("dtype,splits,n,k", [("bf16", [9] * 64, 1408, 2048), ("bf16", [8] * 32, 2048, 2048), ("fp8", [9] * 64, 1408, 4096),
                                              ("bf16", [20] * 32, 1024, 512), ("f16", [20, 24, 28, 18], 192, 8208),
                                              ("fp8", [60] * 16, 2048, 2048), ("fp8", [300] + [30] * 15, 2048, 2048), ("bf16", [44] * 8, 2048, 2048)])
def test_several_weight_groups_have_the_bits_of_one_launch_each(dtype, splits, n, k):
    """The number of weight groups may choose between panel tiles and the streaming form, with more rows between them and the macro tiles."""
    print(f"[case] panel gemm groups {dtype} n={n} k={k}", flush=True)
    x, ws, run = random_operands(splits, n, k, dtype, groups=4)
    sp = torch.tensor(splits, dtype=torch.int32, device="cuda")
    alone = [run(torch.arange(len(x), device="cuda"), splits, w) for w in ws]
    for groups in (2, 3, 4):
        for got, want in zip(capi.grouped_gemm_multi(x, ws[:groups], sp, out_dtype=torch.float32), alone):
            assert torch.equal(got, want)


@pytest.mark.parametrize("dtype", ["bf16", "f16", "fp8"])
@pytest.mark.parametrize("name,splits,n,k,cols,chunk", LINES, ids=[c[0] for c in LINES])
def test_panel_tiles_same_bits_where_weights_do_not_start_on_lines(name, splits, n, k, cols, chunk, dtype):
    """The cache policy of the weights' loads follows their alignment to 128 bytes; results do not."""
    print(f"[case] panel gemm, weights off a line {dtype} {name} n={n} k={k}", flush=True)
    a, w, sp, _ = made(splits, n, k, dtype, n + k)
    ad, wd = a.to(DT[dtype]), w.to(DT[dtype])
    assert k * wd.element_size() % 128 == 0 and wd.data_ptr() % 128 == 0
    raw = wd.view(torch.uint8).reshape(-1)
    store = torch.empty(raw.numel() + 128, dtype=torch.uint8, device="cuda")
    store[16:16 + raw.numel()] = raw
    moved = store[16:16 + raw.numel()].view(DT[dtype]).view(wd.shape)
    assert moved.data_ptr() % 128 == 16 and moved.is_contiguous()
    want = capi.grouped_gemm(ad, wd, sp, out_dtype=torch.float32)
    assert torch.equal(capi.grouped_gemm(ad, moved, sp, out_dtype=torch.float32), want)
    assert torch.equal(want.double(), product(a, w, splits))


@pytest.mark.parametrize("dtype", ["bf16", "fp8", "bs"])
@pytest.mark.parametrize("splits,computes", [([129] + [40] * 15 + [30] * 8, 1), ([600, 600] + [10] * 22, 0), ([64] * 5 + [0] * 19, 1)])
def test_splits_choose_between_panel_and_macro_tiles(dtype, splits, computes):
    """Both are launched; every result is computed, and added to a sum, exactly once, also by a captured launch whose splits change."""
    n, k, m, e = 1408, 1152, sum(splits), len(splits)
    print(f"[case] panel gemm by splits {dtype} {splits[:3]}", flush=True)
    rows = 24 * 60  # on average, whatever the splits
    info = capi.gemm_launch_info(DT[dtype], e, rows, n, k, splits=splits, panel=True, block_scaled=dtype == "bs")
    assert (info.macro_tiles_too, info.computes) == (1, computes)
    a, w, sp, g = made(splits, n, k, dtype, m)
    a = torch.cat([a, a.new_zeros(rows - m, k)])
    ad, wd = a.to(DT[dtype]), w.to(DT[dtype])
    want = product(a, w, splits)
    if dtype == "bs":
        sad, sbd = torch.ones((rows + 127) // 128, k // 128, 128, device="cuda"), torch.ones(e, n // 128, k // 128, device="cuda")
        run = lambda out: capi.grouped_gemm_blockscale(ad, wd, sp, sad, sbd, out=out)
    else:
        run = lambda out: capi.grouped_gemm(ad, wd, sp, out=out)
        token = torch.randint(0, m // 2 + 1, (rows,), generator=g, device="cuda")
        sums = torch.zeros(m // 2 + 1, n, dtype=torch.float64, device="cuda").index_add_(0, token[:m], want)
        got = capi.grouped_gemm_topk_reduce(ad, wd, sp, token.to(torch.int32), m // 2 + 1)
        assert torch.equal(got, sums.float().to(got.dtype))
    out = torch.full((rows, n), -1.0, device="cuda")
    run(out)
    assert torch.equal(out[:m].double(), want) and bool((out[m:] == -1).all())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run(out)
    for s in (splits, [0] * (e - 1) + [300], [20] * e, splits):
        sp.copy_(torch.tensor(s, dtype=torch.int32))
        out.fill_(-1)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out[:sum(s)].double(), product(a, w, s)) and bool((out[sum(s):] == -1).all())


@pytest.mark.parametrize("splits,computes", [([128] + [50] * 23, 1), ([129] + [50] * 23, 0), ([129] + [50] * 22 + [0], 1)])
def test_block_scaled_rounds_choose_between_panel_and_macro_tiles(splits, computes):
    """24 experts of 21 column tiles are two rounds, a chunk more is a third: both launches agree on which of them computes."""
    n, k, m, e = 2688, 256, sum(splits), len(splits)
    print(f"[case] panel gemm, rounds {splits[:3]}", flush=True)
    assert capi.gemm_launch_info(DT["bs"], e, m, n, k, splits=splits, panel=True, block_scaled=True).computes == computes
    a, w, sp, _ = made(splits, n, k, "bs", m)
    sad, sbd = torch.ones((m + 127) // 128, k // 128, 128, device="cuda"), torch.ones(e, n // 128, k // 128, device="cuda")
    out = torch.full((m, n), -1.0, device="cuda")
    capi.grouped_gemm_blockscale(a.to(DT["bs"]), w.to(DT["bs"]), sp, sad, sbd, out=out)
    assert torch.equal(out.double(), product(a, w, splits))


@pytest.mark.parametrize("dtype", ["bf16", "fp8", "bs"])
@pytest.mark.parametrize("splits,n,k,done", [([7, 0, 30, 1], 1024, 8192, 1), ([12, 3, 9, 20, 17, 0, 31, 8], 4160, 384, 1), ([70, 64, 1, 0], 192, 256, 1),
                                             ([-3, 20, 600, 5], 192, 256, 1), ([129] + [40] * 15 + [30] * 8, 1408, 1152, 1),
                                             ([600, 600] + [10] * 22, 1408, 1152, 0), ([300, 200], 1024, 1024, 0), ([4] * 129, 1024, 384, 0)])
def test_row_counts_known_on_the_host(dtype, splits, n, k, done):
    """One kernel with the counts in its arguments has the bits of the ordinary call; otherwise nothing is launched."""
    print(f"[case] host splits {dtype} {splits[:4]} n={n} k={k}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(n + k)
    m, e = sum(max(0, r) for r in splits), len(splits)
    x = torch.randn(m, k, generator=g, device="cuda").to(DT[dtype])
    w = (torch.randn(e, n, k, generator=g, device="cuda") * 0.05).to(DT[dtype])
    sa = torch.rand((m + 127) // 128, k // 128, 128, generator=g, device="cuda")
    sb = torch.rand(e, (n + 127) // 128, k // 128, generator=g, device="cuda")
    r1, r2 = (torch.rand(m, generator=g, device="cuda") + 0.5 for _ in range(2))
    sp = torch.tensor(splits, dtype=torch.int32, device="cuda")
    kw = {} if dtype == "bs" else {"row_scale": r1 * r2}
    want = torch.full((m, n), -1.0, device="cuda")
    if dtype == "bs": capi.grouped_gemm_blockscale(x, w, sp, sa, sb, out=want)
    else: capi.grouped_gemm(x, w, sp, out=want, **kw)
    args, out = capi._gemm_args(x, w, sp, None, None, None, None, None if dtype == "bs" else r1, None, 1.0, None, None, torch.float32, 0, 0, 0)
    host, on_device = (ctypes.c_int32 * e)(*splits), args.splits
    scales = [capi._ptr(sa), capi.ASCALE_BLOCK128, capi._ptr(sb), capi.BSCALE_N_K] if dtype == "bs" else [None, 0, None, 0]
    call = lambda second: capi.load().fluxmi_grouped_gemm_host_splits(ctypes.byref(args), host, second, *scales, capi._stream())
    args.splits = None
    out.fill_(-1)
    assert call(None if dtype == "bs" else capi._ptr(r2)) == done
    assert torch.equal(out, want) if done else bool((out == -1).all())
    args.splits, r12 = on_device, r1 * r2  # with the counts on the device as well
    if dtype != "bs": args.row_scale = r12.data_ptr()
    out.fill_(-1)
    assert call(None) == 1
    assert torch.equal(out, want)


@pytest.mark.parametrize("dtype", ["bf16", "f16", "fp8"])
@pytest.mark.parametrize("splits,n,kbytes", [([64, 0, 33, 17], 192, b) for b in (64, 128, 256, 384, 640, 720, 896, 1664)] +
                         [([30, 34, 20, 17, 30, 0, 3, 26], 64, 8192), ([20, 17, 30, 0], 256, 768), ([96, 80, 1, 64], 1024, 1152), ([0, 0, 0], 192, 256)])
def test_a_ring_in_pairs_for_one_workgroup_to_a_unit(dtype, splits, n, kbytes):
    """Launches with no more items than compute units, as the host's row counts say: odd and even numbers of lines of K, fewer than the ring holds,
    a part of a line, one, four and eight sums, no rows at all.  Integers, so any order of summation is exact."""
    k, m, e = kbytes // DT[dtype].itemsize, max(1, sum(splits)), len(splits)
    print(f"[case] panel gemm in pairs {dtype} {splits} n={n} k={k}", flush=True)
    a, w, sp, _ = made(splits, n, k, dtype, n + k) if sum(splits) else made([1] + splits[1:], n, k, dtype, n + k)
    ad, wd = a.to(DT[dtype]), w.to(DT[dtype])
    args, out = capi._gemm_args(ad, wd, sp, None, None, None, None, None, None, 1.0, None, None, torch.float32, 0, 0, 0)
    args.splits = None
    out.fill_(-1)
    host = (ctypes.c_int32 * e)(*splits)
    assert capi.load().fluxmi_grouped_gemm_host_splits(ctypes.byref(args), host, None, None, 0, None, 0, capi._stream()) == 1
    if sum(splits): assert torch.equal(out.double(), product(a, w, splits))
    else: assert bool((out == -1).all())
