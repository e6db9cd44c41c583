"""GPU parity of the dual tiles of the grouped GEMM (256 x 256 on eight waves that take turns) at the edges of their tiles.

Operands are small integers and scales powers of two, so every product and every partial sum is a whole multiple of a power of two
below 2^24 steps: the fp32 result is the same in any order of summation and has to equal a float64 matmul exactly, no tolerance."""
import ctypes

import pytest
import torch

from flux_amd import capi
from test_gpu_gemm_panel import DT, block_scales, made, product

pytestmark = pytest.mark.gpu

# Rows on both sides of a wave's 64, of both halves of a tile and of one, two and more tiles, empty experts, up to 128 experts; columns that end
# in each group of 32 and after the first half of a tile; the fewest steps of K, odd and even numbers of them, and more than the ring holds;
# tiles of a last round cut in four, in two and whole, and several rounds.
CASES = [
    ("heights", [255, 256, 257, 64, 65, 128, 129, 193, 321, 0, 1, 1000, 190], 392, 384),
    ("two steps", [300], 136, 256),
    ("128 experts", [200, 0, 450] + [190] * 124 + [700], 264, 256),
    ("long K, cut in two", [313, 511, 300, 248, 192], 2312, 2176),
    ("cut in four", [600, 1], 1032, 1152),
    ("several rounds", [1100, 900, 1300, 1024], 4104, 640),
]


def is_dual(dtype, splits, n, k, **kw):
    m, e = sum(splits), len(splits)
    info = capi.gemm_launch_info(DT[dtype], e, m, n, k, splits=splits, block_scaled=dtype == "bs")
    return info.form == capi.GEMM_MACRO_TILES and capi.gemm_dual_tiles(DT[dtype], e, m, n, k, block_scaled=dtype == "bs", **kw)


@pytest.mark.parametrize("dtype", ["bf16", "f16", "fp8"])
@pytest.mark.parametrize("name,splits,n,k", CASES, ids=[c[0] for c in CASES])
def test_dual_tiles_are_exact_on_integers(name, splits, n, k, dtype):
    print(f"[case] dual gemm {dtype} {name} n={n} k={k}", flush=True)
    m, e = sum(splits), len(splits)
    assert is_dual(dtype, splits, n, k)
    assert not is_dual(dtype, splits, n, k, sched_flags=capi.SCHED_HALF_LINE_FILLS)
    a, w, sp, g = made(splits, n, k, dtype, n + k)
    ad, wd = a.to(DT[dtype]), w.to(DT[dtype])
    want = product(a, w, splits)
    assert torch.equal(capi.grouped_gemm(ad, wd, sp), want.float().to(capi._half_out(ad.dtype)))
    perm = torch.randperm(m, generator=g, device="cuda").to(torch.int32)
    to = perm.flip(0).contiguous()
    row_scale = 2.0 ** torch.randint(-1, 2, (m,), generator=g, device="cuda").float()
    col_scale = 2.0 ** torch.randint(-1, 2, (e, n), generator=g, device="cuda").float()
    alpha = 2.0 ** torch.randint(-1, 2, (e,), generator=g, device="cuda").float()
    expert = torch.repeat_interleave(torch.arange(e, device="cuda"), sp.long())
    picked = torch.empty_like(want)
    picked[to.long()] = product(a[perm.long()], w, splits) * (alpha[expert] * row_scale).double()[:, None] * col_scale[expert].double()
    for margin, flags in ((0, 0), (40, capi.SCHED_WHOLE_TAIL_TILES), (253, 0)):
        out = torch.full((m, n), -7.0, device="cuda")
        capi.grouped_gemm(ad, wd, sp, out=out, gather_a=perm, scatter_d=to, row_scale=row_scale, col_scale=col_scale, alpha=alpha, cu_margin=margin,
                          sched_flags=flags, raster_rows=margin // 40)
        assert torch.equal(out.double(), picked), f"margin {margin}"
    other = -w.flip(0)  # (negated too: a single expert flipped is itself)
    two = capi.grouped_gemm_multi(ad, [wd, other.to(DT[dtype])], sp, out_dtype=torch.float32)
    assert torch.equal(two[0].double(), want)
    assert torch.equal(two[1].double(), product(a, other, splits))


@pytest.mark.parametrize("dtype", ["bf16", "f16", "fp8"])
@pytest.mark.parametrize("out_dtype", ["half", "fp32"])
def test_dual_tiles_odd_indices_scalars_and_weights_off_lines(dtype, out_dtype):
    """Gathered rows outside A are its first or last row, scattered rows outside D are not stored; a scalar from the host and one from the
    device; weights that start 16 bytes past a line.  Experts of one row tile and of two."""
    splits, n, k = [250, 256, 0, 300, 230], 392, 384
    print(f"[case] dual gemm odd indices {dtype} {out_dtype}", flush=True)
    m, e, a_rows = sum(splits), len(splits), 77
    assert is_dual(dtype, splits, n, k, gathered=True) and is_dual(dtype, splits, n, k, gathered=True, d_fp32=True)
    a, w, sp, g = made(splits, n, k, dtype, 11)
    a = a[:a_rows]
    raw = torch.zeros(w.numel() * DT[dtype].itemsize + 256, dtype=torch.uint8, device="cuda")
    at = -raw.data_ptr() % 128 + 16
    wd = raw[at:at + w.numel() * DT[dtype].itemsize].view(DT[dtype]).view(e, n, k)
    wd.copy_(w.to(DT[dtype]))
    assert wd.data_ptr() % 128 == 16
    gather = torch.randint(-90, 200, (m,), generator=g, device="cuda").to(torch.int32)
    to = torch.randperm(m, generator=g, device="cuda").to(torch.int32)
    outside = torch.randperm(m, generator=g, device="cuda")[:200]
    to[outside[:100]] = torch.randint(-(1 << 31), 0, (100,), generator=g, device="cuda").to(torch.int32)
    to[outside[100:]] = torch.randint(m, (1 << 31) - 1, (100,), generator=g, device="cuda").to(torch.int32)
    kept = (to >= 0) & (to < m)
    want = torch.full((m, n), -7.0, device="cuda", dtype=torch.float64)
    rows = product(a[gather.long().clamp(0, a_rows - 1)], w, splits) * (0.5 * 4.0)
    want[to[kept].long()] = rows[kept]
    kind = torch.float32 if out_dtype == "fp32" else capi._half_out(DT[dtype])
    out = torch.full((m, n), -7.0, device="cuda", dtype=kind)
    capi.grouped_gemm(a.to(DT[dtype]), wd, sp, out=out, gather_a=gather, scatter_d=to, scalar_scale=0.5,
                      scalar_scale_dev=torch.tensor([4.0], device="cuda"), max_rows=m)
    assert torch.equal(out, want.to(torch.float32).to(kind))


@pytest.mark.parametrize("dtype", ["bf16", "fp8"])
def test_dual_tiles_fp32_results_beyond_half_a_gigabyte(dtype):
    """Such launches store non-temporally.  Most rows are not any expert's: they keep what they held."""
    splits, n, k, m = [300, 0, 256, 129, 64, 700] + [0] * 10, 5640, 256, 24000
    print(f"[case] dual gemm non-temporal stores {dtype}", flush=True)
    assert m * n * 4 > 512 << 20 and capi.gemm_dual_tiles(DT[dtype], len(splits), m, n, k, d_fp32=True)
    a, w, sp, _ = made([sum(splits)] + [0] * 15, n, k, dtype, 5)
    wide = torch.zeros(m, k, device="cuda", dtype=DT[dtype])
    wide[:a.shape[0]] = a.to(DT[dtype])
    sp = torch.tensor(splits, dtype=torch.int32, device="cuda")
    out = torch.full((m, n), -7.0, device="cuda")
    capi.grouped_gemm(wide, w.to(DT[dtype]), sp, out=out)
    assert torch.equal(out[:a.shape[0]].double(), product(a, w, splits)) and bool((out[a.shape[0]:] == -7).all())


@pytest.mark.parametrize("k", [256, 384, 1152])
def test_dual_tiles_block_scaled_infinite_and_nan_scales(k):
    """A scale that is infinite or not a number reaches the results of its row, or of its 128 columns of one expert, and no others; in the
    first block of K, where nothing has been summed yet, and in the last.  Positive operands: no infinity meets its opposite or a zero."""
    splits, n = [300, 129, 64, 250], 392
    print(f"[case] dual gemm block-scaled, scales that are not finite K={k}", flush=True)
    m, e, kb = sum(splits), len(splits), k // 128
    assert is_dual("bs", splits, n, k)
    g = torch.Generator(device="cuda").manual_seed(k)
    a = torch.randint(1, 4, (m, k), generator=g, device="cuda").float()
    w = torch.randint(1, 4, (e, n, k), generator=g, device="cuda").float()
    sp = torch.tensor(splits, dtype=torch.int32, device="cuda")
    sa, sb, _, _ = block_scales(m, e, n, k, splits, capi.ASCALE_BLOCK128, capi.BSCALE_N_K, g)
    sa[5, 0], sa[70, kb - 1], sa[310, 0], sa[440, kb - 1] = float("inf"), float("inf"), float("nan"), float("nan")
    sb[1, 1, 0], sb[3, 3, kb - 1] = float("inf"), float("nan")
    pad = torch.zeros((m + 127) // 128 * 128, kb, device="cuda")
    pad[:m] = sa
    want = product(a * torch.repeat_interleave(sa, 128, dim=1),
                   w * torch.repeat_interleave(torch.repeat_interleave(sb, 128, dim=1)[:, :n], 128, dim=2), splits)
    got = capi.grouped_gemm_blockscale(a.to(DT["bs"]), w.to(DT["bs"]), sp, pad.view(-1, 128, kb).permute(0, 2, 1).contiguous(), sb,
                                       out_dtype=torch.float32).double()
    assert torch.isnan(want).any() and torch.isinf(want).any() and torch.isfinite(want).any()
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(torch.nan_to_num(got), torch.nan_to_num(want))


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("splits,n,k", [([200, 300, 64, 511], 1040, 2112), ([900, 700], 520, 1024), ([128, 470, 77], 2304, 8192)])
def test_dual_tiles_have_the_macro_tiles_bits(splits, n, k, dtype):
    print(f"[case] dual gemm bits {dtype} n={n} k={k}", flush=True)
    assert is_dual(dtype, splits, n, k)
    g = torch.Generator(device="cuda").manual_seed(k)
    a = torch.randn(sum(splits), k, generator=g, device="cuda").to(DT[dtype])
    w = torch.randn(len(splits), n, k, generator=g, device="cuda").to(DT[dtype])
    sp = torch.tensor(splits, dtype=torch.int32, device="cuda")
    for out in (torch.float32, DT[dtype]):
        assert torch.equal(capi.grouped_gemm(a, w, sp, out_dtype=out),
                           capi.grouped_gemm(a, w, sp, out_dtype=out, sched_flags=capi.SCHED_HALF_LINE_FILLS))


@pytest.mark.parametrize("name,splits,n,k", CASES, ids=[c[0] for c in CASES])
@pytest.mark.parametrize("a_layout", [capi.ASCALE_BLOCK128, capi.ASCALE_EXPERT_K_M])
@pytest.mark.parametrize("b_layout", [capi.BSCALE_N_K, capi.BSCALE_K_N])
def test_dual_tiles_block_scaled_are_exact_on_integers(name, splits, n, k, a_layout, b_layout):
    print(f"[case] dual gemm block-scaled {name} n={n} k={k} layouts {a_layout} {b_layout}", flush=True)
    m, e = sum(splits), len(splits)
    assert is_dual("bs", splits, n, k)
    a, w, sp, g = made(splits, n, k, "fp8", n + k)
    sa, sb, sad, sbd = block_scales(m, e, n, k, splits, a_layout, b_layout, g)
    af = a * torch.repeat_interleave(sa, 128, dim=1)
    wf = w * torch.repeat_interleave(torch.repeat_interleave(sb, 128, dim=1)[:, :n], 128, dim=2)
    want = product(af, wf, splits)
    ad, wd = a.to(DT["bs"]), w.to(DT["bs"])
    for margin in (0, 40, 253):
        args, out = capi._gemm_args(ad, wd, sp, None, None, None, None, None, None, 1.0, None, None, torch.float32, margin, 0, 0)
        capi._check(capi.load().fluxmi_grouped_gemm_blockscale(ctypes.byref(args), capi._ptr(sad), a_layout, capi._ptr(sbd), b_layout, capi._stream()),
                    "fluxmi_grouped_gemm_blockscale")
        assert torch.equal(out.double(), want), f"margin {margin}"
    half = capi.grouped_gemm_blockscale(ad, wd, sp, sad, sbd, a_layout, b_layout)
    assert torch.equal(half, want.float().to(torch.bfloat16))
    if a_layout == capi.ASCALE_BLOCK128:  # rows, and their scales, picked by a gather; results put elsewhere, with every factor
        perm = torch.randperm(m, generator=g, device="cuda").to(torch.int32)
        to = perm.flip(0).contiguous()
        row_scale = 2.0 ** torch.randint(-1, 2, (m,), generator=g, device="cuda").float()
        col_scale = 2.0 ** torch.randint(-1, 2, (e, n), generator=g, device="cuda").float()
        alpha = 2.0 ** torch.randint(-1, 2, (e,), generator=g, device="cuda").float()
        expert = torch.repeat_interleave(torch.arange(e, device="cuda"), sp.long())
        picked = torch.empty_like(want)
        picked[to.long()] = product(af[perm.long()], wf, splits) * (alpha[expert] * row_scale).double()[:, None] * col_scale[expert].double()
        got = capi.grouped_gemm_blockscale(ad, wd, sp, sad, sbd, a_layout, b_layout, out_dtype=torch.float32, gather_a=perm, scatter_d=to,
                                           row_scale=row_scale, col_scale=col_scale, alpha=alpha)
        assert torch.equal(got.double(), picked)


def test_dual_tiles_do_not_touch_rows_past_the_splits():
    """Rows beyond sum(splits), and negative and too large counts: clamped like everywhere else."""
    print("[case] dual gemm block-scaled, counts past the rows", flush=True)
    splits, n, k, m = [400, -7, 300, 5000], 264, 512, 1000
    a, w, _, g = made([m], n, k, "fp8", 3)
    w = torch.randint(-3, 4, (4, n, k), generator=g, device="cuda").float()
    sad, sbd = torch.ones((m + 127) // 128, k // 128, 128, device="cuda"), torch.ones(4, 3, k // 128, device="cuda")
    out = torch.full((m + 8, n), -5.0, device="cuda")
    call = lambda s: capi.grouped_gemm_blockscale(a.to(DT["bs"]), w.to(DT["bs"]), torch.tensor(s, dtype=torch.int32, device="cuda"), sad, sbd, out=out)
    call(splits)
    assert torch.equal(out[:m].double(), product(a, w, [400, 0, 300, 300])) and bool((out[m:] == -5).all())
    out.fill_(-5)
    call([400, 0, 300, 0])
    assert torch.equal(out[:700].double(), product(a[:700], w, [400, 0, 300, 0])) and bool((out[700:] == -5).all())


@pytest.mark.parametrize("dtype,splits,n,k,done", [(d, *c) for d in ("bf16", "f16", "fp8", "bs") for c in (
    ([600, 0, 500, 557], 392, 384, 1), ([-3, 700, 900, 1], 264, 256, 1), ([600, 500, 700], 136, 256, 1), ([250] * 128, 264, 256, 1),
    ([250] * 129, 264, 256, 0), ([700, 600], 264, 320, 0)) if d != "bs" or c[2] % 128 == 0])
def test_dual_tiles_take_row_counts_from_the_host(dtype, splits, n, k, done):
    """Counts and a second factor per row in the kernel's arguments: the bits of the ordinary call with the factors' product.  Not for more
    experts than the arguments hold nor (K = 320, in fp8 no whole lines) for other forms; nothing is launched then."""
    print(f"[case] dual gemm, counts in the arguments {dtype} {splits[:4]} n={n} k={k}", flush=True)
    if dtype != "fp8" and k == 320:
        done = 1
    if dtype == "bs":
        n = (n + 127) // 128 * 128
    g = torch.Generator(device="cuda").manual_seed(n + k)
    m, e = sum(max(0, r) for r in splits) - (100 if splits == [600, 500, 700] else 0), len(splits)  # or fewer rows than the counts say
    x = torch.randn(m, k, generator=g, device="cuda").to(DT[dtype])
    w = (torch.randn(e, n, k, generator=g, device="cuda") * 0.05).to(DT[dtype])
    sa, sb = torch.rand((m + 127) // 128, k // 128, 128, generator=g, device="cuda"), torch.rand(e, (n + 127) // 128, k // 128, generator=g, device="cuda")
    r1, r2 = (torch.rand(m, generator=g, device="cuda") + 0.5 for _ in range(2))
    sp = torch.tensor(splits, dtype=torch.int32, device="cuda")
    want = torch.full((m, n), -1.0, device="cuda")
    if dtype == "bs": capi.grouped_gemm_blockscale(x, w, sp, sa, sb, out=want)
    else: capi.grouped_gemm(x, w, sp, out=want, row_scale=r1 * r2)
    args, out = capi._gemm_args(x, w, sp, None, None, None, None, None if dtype == "bs" else r1, None, 1.0, None, None, torch.float32, 0, 0, 0)
    host, on_device = (ctypes.c_int32 * e)(*splits), args.splits
    scales = [capi._ptr(sa), capi.ASCALE_BLOCK128, capi._ptr(sb), capi.BSCALE_N_K] if dtype == "bs" else [None, 0, None, 0]
    call = lambda entry, second: getattr(capi.load(), entry)(ctypes.byref(args), host, second, *scales, capi._stream())
    args.splits = None
    out.fill_(-1)
    second = None if dtype == "bs" else capi._ptr(r2)
    assert call("fluxmi_grouped_gemm_host_splits", second) == 0
    assert bool((out == -1).all())
    assert call("fluxmi_grouped_gemm_host_counts", second) == done
    assert torch.equal(out, want) if done else bool((out == -1).all())
    args.splits, r12 = on_device, r1 * r2  # with the counts on the device as well
    if dtype != "bs": args.row_scale = r12.data_ptr()
    out.fill_(-1)
    assert call("fluxmi_grouped_gemm_host_counts", None) == 1
    assert torch.equal(out, want)


@pytest.mark.parametrize("dtype", ["bf16", "f16", "fp8"])
@pytest.mark.parametrize("splits,n,k", [([700], 264, 384), ([300, 257, 512], 520, 512), ([513, 0, 470, 256, 300], 1032, 640), ([290] * 9, 1800, 256)])
def test_fewer_tiles_than_compute_units(splits, n, k, dtype):
    """Grids of more workgroups than tiles: one to four tiles to an XCD, cut in four, in two and whole, grids off the eight XCDs, in both forms of
    256 x 256 tiles.  Integers, exact."""
    print(f"[case] few tiles {dtype} {splits[:4]} n={n} k={k}", flush=True)
    assert is_dual(dtype, splits, n, k)
    a, w, sp, _ = made(splits, n, k, dtype, n + k)
    ad, wd, want = a.to(DT[dtype]), w.to(DT[dtype]), product(a, w, splits)
    for flags in (0, capi.SCHED_WHOLE_TAIL_TILES, capi.SCHED_HALF_LINE_FILLS, capi.SCHED_HALF_LINE_FILLS | capi.SCHED_NO_SKINNY_TAIL):
        for margin in (0, 100, 219):
            out = torch.full((sum(splits), n), -7.0, device="cuda")
            capi.grouped_gemm(ad, wd, sp, out=out, sched_flags=flags, cu_margin=margin)
            assert torch.equal(out.double(), want), f"flags {flags} margin {margin}"
