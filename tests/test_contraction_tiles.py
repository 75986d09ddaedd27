"""GPU: every tile of the contraction kernels.

One code object per group takes the row count M at launch and runs the tile
the lowering chooses for it (16x16 ... 256x128); N = 1040 leaves every tile a
ragged last column tile, K ends in half a 128-byte slice, and the row counts
sit on and beside the tiles' edges.  Groups of N = 4016 and whole slices of K
reach the 256x256 ring, which takes no half slice.  Whole-number sums are
exact; 16-bit floats are held to the f32 summation bound K 2^-24 sum|ab| plus
half an ulp of the output; block-scaled results to the matrix core's bars.
"""
import numpy as np
import pytest

import hfusion_mi355x as hf
import group_catalog as cat
from helpers import run_gpu
from test_dynamic import _call
from test_matmul_mx import TOL_FP4, fp4_case, fp4_products

I = hf.inputs
N = 1040
ROWS = [1, 16, 17, 33, 64, 65, 100, 129, 200, 2000, 3500, 5900]


def test_alternatives_by_row_count():
    """The manifest lists the kernels by ascending row count, each with the
    grid of its tile, and they are what a static group of that M gets."""
    for name, k, layout in (("tiles_w8a8_nk_rt", 1088, "nk"), ("tiles_w8a8_kn_rt", 1088, "kn")):
        art = hf.compile(cat.get(name), options="dyn=runtime")
        alts = [ln.split()[1:] for ln in open(art.manifest) if ln.startswith("alt ")]
        rows = [int(a[1]) for a in alts]
        assert rows == sorted(set(rows)) and len(alts) >= 5
        for kern, top, rb, rc, threads in alts:
            tm, tn = (int(v) for v in kern.rsplit("_", 1)[1].split("k")[0].split("x"))
            assert int(rb) == tm and int(rc) == (-(-N // tn) + 7) // 8 * 8 and int(threads) <= 1024
            blk = hf.compile(hf.groups.w8a8_dequant(int(top), N, k, b_layout=layout), options="emit=hip").blocks[0]
            assert f"{tm}x{tn} tiles" in blk["variant"]
            assert blk["grid"][0] == -(-int(top) // tm) * int(rc)


def test_tile_where_large_ones_queue():
    """Sizes a little past whole rounds of 256x256 tiles, and few wide columns:
    the 256x256 ring, or the largest tile that fills the chip."""
    g = hf.groups
    ring = "LDS DMA ring (128-byte slices, 2 waves/SIMD"
    for ir, want in [(g.w8a8_dequant(5000, 4096, 4096), ring), (g.w8a8_dequant(5000, 4096, 4096, b_layout="kn"), ring),
                     (g.bf16_mmad(5000, 4096, 4096), ring), (g.bf16_mmad(3000, 11008, 4096, b_layout="kn"), ring),
                     (g.w8a8_dequant(1536, 14336, 4096), ring), (g.matmul_mx(5000, 4096, 4096), "mfma_scale"),
                     (g.bf16_mmad(5000, 1024, 4096), "256x128 tiles"), (g.w8a8_dequant(5000, 1024, 4096, b_layout="kn"), "256x128 tiles"),
                     (g.w8a8_dequant(2048, 4096, 4096), "256x128 tiles"), (g.w8a8_dequant(1024, 4096, 4096), "128x128 tiles")]:
        b = hf.compile(ir, options="emit=hip").blocks[0]
        assert want in b["variant"], b["variant"]
    for fmt in ("e4m3", "e2m1"):
        b = hf.compile(g.matmul_mx(5000, 4096, 4096, fa=fmt, fb=fmt, via="format"), options="emit=hip").blocks[0]
        assert b["grid"][0] == 20 * 16 and b["block"][0] == 512


TILES = {"nk": {"16x16", "32x16", "32x32", "64x32", "64x64k2", "64x64", "128x64", "128x128", "256x128"},
         "kn": {"16x16", "32x16", "32x32", "32x64", "64x64k2", "64x64", "64x128k2", "128x64", "128x128", "256x128"},
         "mx_e4m3": {"32x64", "64x64", "64x128", "128x128"}, "mx_e2m1": {"32x64", "64x64", "64x128", "128x128"}}
# groups that between them run every tile of a family: (name, N, K)
TILE_GROUPS = {("nk", "w8a8"): [("tiles_w8a8_nk_k2112_rt", 1040, 2112)], ("nk", "bf16"): [("tiles_bf16_nk_k1056_rt", 1040, 1056)],
               ("kn", "w8a8"): [("tiles_w8a8_kn_k2112_rt", 1040, 2112), ("tiles_w8a8_kn_rt", 1040, 1088), ("tiles_w8a8_kn_n2064_rt", 2064, 4160)],
               ("kn", "bf16"): [("tiles_bf16_kn_k1056_rt", 1040, 1056), ("tiles_bf16_kn_k544_rt", 1040, 544), ("tiles_bf16_kn_n2064_rt", 2064, 2080)],
               ("mx_e4m3", ""): [("tiles_mx_e4m3_rt", 1040, 640)], ("mx_e2m1", ""): [("tiles_mx_e2m1_rt", 1040, 1280)]}
MOST_ROWS = 6000
RING_GROUPS = ["ring_w8a8_nk_rt", "ring_w8a8_kn_rt", "ring_bf16_kn_rt", "ring_mx_e4m3_rt", "ring_mx_e2m1_rt"]


def _alts(name, **kw):
    """(kernel, largest row count, rows a tile) of each alternative, ascending."""
    art = hf.compile(cat.get(name), options="dyn=runtime", **kw)
    rows = [ln.split()[1:] for ln in open(art.manifest) if ln.startswith("alt ")]
    return [(r[0], int(r[1]), int(r[2])) for r in rows]


def _rows_of_tiles(name, **kw):
    """{tile: the first and the last row count of its first range}."""
    out, low = {}, 0
    for kern, top, _ in _alts(name, **kw):
        out.setdefault(kern.rsplit("_", 1)[1], (low + 1, top))
        low = top
    return out


def _ring_rows(name, **kw):
    """Row counts that run the main kernel (the ring): the first and the last
    of its first range as an alternative, and one past every alternative."""
    alts, low, rows = _alts(name, **kw), 0, []
    for kern, top, tm in alts:
        if tm == 256 and "_256x" not in kern and not rows:
            rows = [low + 1, top]
        low = top
    return rows + [low + 1, low + 300]


@pytest.mark.parametrize("family", list(TILE_GROUPS))
def test_every_tile_is_picked(family):
    """The groups run every tile that the lowering can pick, each within the
    row counts that the GPU test takes."""
    run = {t for name, _, _ in TILE_GROUPS[family] for t, ends in _rows_of_tiles(name).items() if ends[0] <= MOST_ROWS}
    assert run - {"256x256"} == TILES[family[0]]


def test_ring_rows_run_the_ring():
    for name in RING_GROUPS:
        b = hf.compile(cat.get(name), options="dyn=runtime").blocks[0]
        assert b["rows_dyn"][1] == 256 and b["rows_dyn"][2] == -(-4016 // 256) and b["block"][0] == 512, name
        assert len(_ring_rows(name)) >= 2 and max(_ring_rows(name)) < 20000


def _whole(name, m, n, k, gpu, seed):
    """A group over whole numbers whose sums are exact in any order, checked
    against the 64-bit product."""
    import torch
    gen = torch.Generator(device=gpu).manual_seed(seed)
    ints = lambda lo, hi, *sh: torch.randint(lo, hi + 1, sh, device=gpu, generator=gen)
    kind = "mx" if "_mx_" in name else "bf16" if "_bf16_" in name else "w8a8"
    dg = hf.DynamicGroup(cat.get(name), require_cached=True, runtime=True)
    if kind == "mx":
        # e4m3 0 .. 7 and e2m1 0 .. 6 by magnitude, scales 1/2, 1 and 2 per 32 k:
        # multiples of 1/4 with |sum| <= 196 K < 2^22 of them
        fp4 = "e2m1" in name
        code = torch.tensor([0x0, 0x2, 0x4, 0x5, 0x6, 0x7] if fp4 else [0x00, 0x38, 0x40, 0x44, 0x48, 0x4A, 0x4C, 0x4E], device=gpu)
        val = torch.tensor([0, 1, 2, 3, 4, 6] if fp4 else [0, 1, 2, 3, 4, 5, 6, 7], dtype=torch.float64, device=gpu)
        def operand(*sh):
            i, neg = ints(0, len(code) - 1, *sh), ints(0, 1, *sh)
            return code[i] + neg * (8 if fp4 else 128), val[i] * (1 - 2 * neg)
        (ca, va), (cb, vb) = operand(m, k), operand(k, n)
        sa, sb = ints(126, 128, m, k // 32), ints(126, 128, n, k // 32)
        ref = (va * torch.exp2(sa.double() - 127).repeat_interleave(32, 1)) @ (vb * torch.exp2(sb.double() - 127).repeat_interleave(32, 1).t())
        if fp4:
            ca, cb = ca[:, 0::2] | ca[:, 1::2] << 4, cb[0::2] | cb[1::2] << 4
        by = lambda t: t.to(torch.uint8).view(torch.int8).contiguous()
        return dg(by(ca), by(cb), by(sa), by(sb)).double(), ref
    lim = 127 if kind == "w8a8" else 3
    a, b = ints(-lim, lim, m, k), ints(-lim, lim, *((n, k) if "_nk_" in name else (k, n)))
    c = a.double() @ (b.double().t() if "_nk_" in name else b.double())
    if kind == "bf16":
        out = dg(a.bfloat16(), b.bfloat16(), torch.empty(m, n, dtype=torch.bfloat16, device=gpu))
        return out, c.bfloat16()
    # (scales are powers of two: one rounding, to bf16; |c| <= 127^2 K rounds to f32 first)
    st, sc = torch.exp2(ints(-6, 0, m).float()), torch.exp2(ints(-6, 0, n).float())
    out = dg(a.to(torch.int8), b.to(torch.int8), st, sc, torch.empty(m, n, dtype=torch.bfloat16, device=gpu))
    return out, ((c.float() * st[:, None]) * sc[None, :]).bfloat16()


@pytest.mark.gpu
@pytest.mark.parametrize("name,n,k", [g for v in TILE_GROUPS.values() for g in v])
def test_gpu_every_tile(gpu, name, n, k):
    """Every tile of a group at the ends of its first range of row counts,
    ragged in N, K and M."""
    import torch
    for tile, ends in _rows_of_tiles(name, require_cached=True).items():
        for m in ends:
            if m > MOST_ROWS:
                continue
            print(f"[case] {name} {tile} M={m}", flush=True)
            out, ref = _whole(name, m, n, k, gpu, 91 + m)
            assert torch.equal(out, ref), (tile, m)


@pytest.mark.gpu
@pytest.mark.parametrize("name", RING_GROUPS)
def test_gpu_ring_launch_time_rows(gpu, name):
    """The 256x256 ring with a launch-time row count, where the alternatives
    hand over to it and past them."""
    import torch
    k = {"w8a8": 640, "bf16": 320, "e4m3": 640, "e2m1": 1280}[name.split("_")[2 if "_mx_" in name else 1]]
    for m in _ring_rows(name, require_cached=True):
        print(f"[case] {name} M={m}", flush=True)
        out, ref = _whole(name, m, 4016, k, gpu, 92 + m)
        assert torch.equal(out, ref), m
        del out, ref


def _mm(rng, m, k, layout):
    a = rng.integers(-127, 128, (m, k), dtype=np.int8)
    b = rng.integers(-127, 128, (N, k) if layout == "nk" else (k, N), dtype=np.int8)
    bt = b.T if layout == "nk" else b
    return a, b, (a.astype(np.float64) @ bt.astype(np.float64)).astype(np.int64)


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["nk", "kn"])
def test_gpu_tiles_w8a8(gpu, layout):
    rng = np.random.default_rng(77)
    # (past 16384 rows the main kernel)
    for m in ROWS + [16500] * (layout == "kn"):
        print(f"[case] tiles_w8a8_{layout}_rt M={m}", flush=True)
        a, b, c = _mm(rng, m, 1088, layout)
        st, sc = rng.uniform(0.001, 0.02, m).astype(np.float32), rng.uniform(0.001, 0.02, N).astype(np.float32)
        out, = _call(f"tiles_w8a8_{layout}_rt", [a, b, st, sc, np.zeros((m, N), np.uint16)], gpu)
        ref = I.f32_to_bf16_bits((c.astype(np.float32) * st[:, None]) * sc[None, :])
        assert np.array_equal(out.view(np.uint16), ref)


@pytest.mark.gpu
@pytest.mark.parametrize("m", [150, 257, 960, 1100, 1791])
@pytest.mark.parametrize("layout", ["nk", "kn"])
def test_gpu_tiles_two_slices(gpu, layout, m):
    """Two slices of K a stage: 8.5 slices, the last stage of the second wave
    group past the end; whole-number values, exact sums."""
    print(f"[case] two slices {layout} M={m}", flush=True)
    rng, k = np.random.default_rng(79), 544
    fa, fb = rng.integers(-3, 4, (m, k)).astype(np.float32), rng.integers(-3, 4, (N, k) if layout == "nk" else (k, N)).astype(np.float32)
    out, = _call(f"tiles_bf16_{layout}_k544_rt", [I.f32_to_bf16_bits(fa), I.f32_to_bf16_bits(fb), np.zeros((m, N), np.uint16)], gpu)
    # (|sum| <= 9 * 544 < 2^24: every order of adding gives it, rounded once)
    assert np.array_equal(out.view(np.uint16), I.f32_to_bf16_bits(fa @ (fb.T if layout == "nk" else fb)))
    a, b, c = _mm(rng, m, 1088, layout)
    st, sc = rng.uniform(0.001, 0.02, m).astype(np.float32), rng.uniform(0.001, 0.02, N).astype(np.float32)
    out, = _call(f"tiles_w8a8_{layout}_rt", [a, b, st, sc, np.zeros((m, N), np.uint16)], gpu)
    assert np.array_equal(out.view(np.uint16), I.f32_to_bf16_bits((c.astype(np.float32) * st[:, None]) * sc[None, :]))


@pytest.mark.gpu
@pytest.mark.parametrize("elem,layout", [("bf16", "nk"), ("bf16", "kn"), ("f16", "kn")])
def test_gpu_tiles_16bit(gpu, elem, layout):
    rng, k = np.random.default_rng(78), 224
    for m in ROWS:
        print(f"[case] tiles_{elem}_{layout}_rt M={m}", flush=True)
        fa, fb = rng.normal(0, 1, (m, k)).astype(np.float32), rng.normal(0, 1, (N, k) if layout == "nk" else (k, N)).astype(np.float32)
        if elem == "bf16":
            a, b = I.f32_to_bf16_bits(fa), I.f32_to_bf16_bits(fb)
            fa, fb, up = I.bf16_bits_to_f32(a), I.bf16_bits_to_f32(b), 2.0 ** -8
        else:
            a, b = fa.astype(np.float16), fb.astype(np.float16)
            fa, fb, up = a.astype(np.float32), b.astype(np.float32), 2.0 ** -11
            a, b = a.view(np.uint16), b.view(np.uint16)
        fa, fb = fa.astype(np.float64), (fb.T if layout == "nk" else fb).astype(np.float64)
        out, = _call(f"tiles_{elem}_{layout}_rt", [a, b, np.zeros((m, N), np.uint16)], gpu)
        got = (I.bf16_bits_to_f32(out.view(np.uint16)) if elem == "bf16" else out.view(np.float16)).astype(np.float64)
        ref, bound = fa @ fb, k * 2.0 ** -24 * (np.abs(fa) @ np.abs(fb))
        # the f32 sum is within `bound`, and rounding it moves it by up to half
        # an ulp: 2^-8 of the value with bf16's 8 significant bits, 2^-11 with
        # f16's 11
        assert np.all(np.abs(got - ref) <= bound + up * (np.abs(ref) + bound) + 2.0 ** -25)


@pytest.mark.gpu
def test_gpu_tiles_mx_fp8(gpu):
    rng, k = np.random.default_rng(79), 640
    codes = np.array([c for c in range(256) if c & 0x7F != 0x7F], np.uint8)
    import torch
    dec = lambda u: torch.from_numpy(u).view(torch.float8_e4m3fn).float().numpy().astype(np.float64)
    for m in ROWS[:-1]:
        print(f"[case] tiles_mx_e4m3_rt M={m}", flush=True)
        a, b = rng.choice(codes, (m, k)), rng.choice(codes, (k, N))
        sa, sb = rng.integers(120, 131, (m, k // 32), dtype=np.uint8), rng.integers(120, 131, (N, k // 32), dtype=np.uint8)
        out, = _call("tiles_mx_e4m3_rt", [a, b, sa, sb], gpu)
        fa = dec(a) * np.repeat(np.exp2(sa.astype(np.float64) - 127), 32, axis=1)
        fb = dec(b) * np.repeat(np.exp2(sb.astype(np.float64) - 127), 32, axis=1).T
        assert np.all(np.abs(out - fa @ fb) <= 2.0 ** -11 * (np.abs(fa) @ np.abs(fb)))


@pytest.mark.gpu
def test_gpu_tiles_mx_fp4(gpu):
    rng, k = np.random.default_rng(80), 1280
    for m in ROWS[:-1]:
        print(f"[case] tiles_mx_e2m1_rt M={m}", flush=True)
        a, b, sa, sb, ca, cb = fp4_case(rng, m, N, k)
        out, = _call("tiles_mx_e2m1_rt", [a, b, sa, sb], gpu)
        mag, ref = fp4_products(ca, cb, sa, sb)
        assert np.all(np.abs(out.astype(np.float64) - ref) <= TOL_FP4 * mag + 1e-30)


@pytest.mark.gpu
@pytest.mark.parametrize("name,k,layout", [("ring_w8a8_nk_k128", 128, "nk"), ("ring_w8a8_kn_k256", 256, "kn"),
                                           ("ring_w8a8_nk_k384", 384, "nk"), ("ring_mx_e4m3_k128", 128, "mx")])
def test_gpu_ring_short_k(gpu, name, k, layout):
    """The alternating wave groups with fewer slices than they keep in
    flight: re-read slices must not reach a result."""
    print(f"[case] {name}", flush=True)
    rng, m, n = np.random.default_rng(81), 4000, 4016
    if layout == "mx":
        # small whole numbers in e4m3 (0 .. 7 and -7 .. 0) with unit scales: exact sums
        code = np.array([0x00, 0x38, 0x40, 0x44, 0x48, 0x4A, 0x4C, 0x4E], np.uint8)
        ia, ib = rng.integers(-7, 8, (m, k)), rng.integers(-7, 8, (k, n))
        enc = lambda v: (code[np.abs(v)] | np.where(v < 0, 0x80, 0).astype(np.uint8))
        sc = [np.full((r, k // 32), 127, np.uint8) for r in (m, n)]
        out, = run_gpu(name, [enc(ia), enc(ib)] + sc, gpu)
        assert np.array_equal(out.astype(np.float64), ia.astype(np.float64) @ ib.astype(np.float64))
        return
    a = rng.integers(-127, 128, (m, k), dtype=np.int8)
    b = rng.integers(-127, 128, (n, k) if layout == "nk" else (k, n), dtype=np.int8)
    c = a.astype(np.float64) @ (b.T if layout == "nk" else b).astype(np.float64)
    st, sc = rng.uniform(0.001, 0.02, m).astype(np.float32), rng.uniform(0.001, 0.02, n).astype(np.float32)
    out, = run_gpu(name, [a, b, st, sc, np.zeros((m, n), np.uint16)], gpu)
    assert np.array_equal(out.view(np.uint16), I.f32_to_bf16_bits((c.astype(np.float32) * st[:, None]) * sc[None, :]))
