"""The copy kernels' forms at the sizes where they change: rows narrower and
wider than a vector, multiples of 16 bytes or not, merged and split bands of
columns, dense and strided destinations, misaligned objects, tiles that start
and end in the middle of a row, a last vector that is not whole, RECAST and
ZERO pieces, rows 2 GiB apart.  Every case is byte movement or one rounding:
exact against torch, with the bytes around each destination untouched."""
import ctypes

import pytest
import torch

from suika_amd import _lib

pytestmark = pytest.mark.gpu

DT = {"u8": (_lib.SR_DT_U8, torch.uint8), "bf16": (_lib.SR_DT_BF16, torch.bfloat16),
      "f32": (_lib.SR_DT_F32, torch.float32), "f64": (_lib.SR_DT_F64, torch.float64)}
COPY, RECAST, ZERO = _lib.SR_PIECE_COPY, _lib.SR_PIECE_RECAST, _lib.SR_PIECE_ZERO
GUARD = 64       # elements around each object
POISON = 0xA7


class Obj:
    """A [rows, cols] object `shift` elements into a guarded allocation."""

    def __init__(self, rows, cols, dt, shift=0, seed=None):
        self.rows, self.cols, self.dt = rows, cols, dt
        tdt = DT[dt][1]
        self.buf = torch.empty(rows * cols + 2 * GUARD, dtype=tdt, device="cuda")
        self.bytes = self.buf.view(torch.uint8)
        self.at = GUARD + shift
        self.es = self.buf.element_size()
        if seed is None:
            self.bytes.fill_(POISON)
        else:
            g = torch.Generator("cuda").manual_seed(seed)
            if tdt.is_floating_point:
                self.buf.copy_(torch.randn(self.buf.shape, generator=g, device="cuda"))
            else:
                self.buf.copy_(torch.randint(0, 256, self.buf.shape, generator=g, device="cuda"))
        self.t = self.buf[self.at:self.at + rows * cols].view(rows, cols)

    def check(self, want, what):
        got = self.t.contiguous().view(torch.uint8)
        assert torch.equal(got, want.contiguous().view(torch.uint8)), what
        lo, hi = self.at * self.es, (self.at + self.rows * self.cols) * self.es
        assert bool((self.bytes[:lo] == POISON).all()) and bool((self.bytes[hi:] == POISON).all()), f"{what}: guard"


def _gather(src, dst, pieces, tile_bytes=0, flags=0, noalloc=False, max_blocks=0):
    L = _lib.lib()
    S = (_lib.SrTensor * max(1, len(src)))(*[_lib.SrTensor(o.rows, o.cols, DT[o.dt][0], 0) for o in src])
    D = (_lib.SrTensor * len(dst))(*[_lib.SrTensor(o.rows, o.cols, DT[o.dt][0], 0) for o in dst])
    P = (_lib.SrPiece * len(pieces))(*[_lib.SrPiece(*p) for p in pieces])
    opt = _lib.SrPlanOptions(tile_bytes, max_blocks, flags, 0)
    h = ctypes.c_void_p()
    _lib.check(L.sr_plan_create(S, len(src), D, len(dst), 1, P, len(pieces), ctypes.byref(opt), ctypes.byref(h)), "plan")
    try:
        vp = ctypes.c_void_p
        sp = (vp * max(1, len(src)))(*[o.t.data_ptr() for o in src])
        dp = (vp * len(dst))(*[o.t.data_ptr() for o in dst])
        call = L.sr_gather_noalloc if noalloc else L.sr_gather
        _lib.check(call(h, sp, dp, vp(torch.cuda.current_stream().cuda_stream)), "gather")
        torch.cuda.synchronize()
    finally:
        L.sr_plan_destroy(h)


def copy(si, di, rows, cols, sc=0, dc=0, sr=0, dr=0):
    return (COPY, 0, si, di, -1, 0, rows, cols, sr, sc, dr, dc)


# bytes per row: below a vector, around 16, around the widths where short rows
# end (64, 384, 400, 512), around a wave's and a tile's vectors
ROWS = [1, 2, 3, 6, 8, 12, 15, 16, 17, 24, 33, 48, 63, 64, 66, 96, 128, 192, 382, 384, 398, 400, 402, 510, 512, 514,
        1022, 1024, 1028, 2730, 5460, 16382, 16384, 16400]


@pytest.mark.parametrize("tile_bytes", [0, 4096, 1 << 16])
@pytest.mark.parametrize("dt", sorted(DT))
def test_bands_of_columns(dt, tile_bytes):
    """Two bands merged side by side and split apart, at every row width that
    is whole elements."""
    es = torch.empty(0, dtype=DT[dt][1]).element_size()
    for k, width in enumerate(w for w in ROWS if w % es == 0):
        c = width // es
        rows = max(3, min(5000, 150000 // width))
        print(f"[copy forms] {dt} rows of {width} B, tile {tile_bytes}", flush=True)
        a, b = Obj(rows, c, dt, seed=3 * k), Obj(rows, c, dt, seed=3 * k + 1)
        d = Obj(rows, 2 * c, dt)
        _gather([a, b], [d], [copy(0, 0, rows, c), copy(1, 0, rows, c, dc=c)], tile_bytes)
        d.check(torch.cat([a.t, b.t], 1), f"merge {width}")
        s = Obj(rows, 2 * c, dt, seed=3 * k + 2)
        x, y = Obj(rows, c, dt), Obj(rows, c, dt)
        _gather([s], [x, y], [copy(0, 0, rows, c), copy(0, 1, rows, c, sc=c)], tile_bytes, noalloc=tile_bytes == 4096)
        x.check(s.t[:, :c], f"split {width}")
        y.check(s.t[:, c:], f"split {width}")


@pytest.mark.parametrize("shift", [(0, 0), (1, 0), (0, 1), (3, 1)])
@pytest.mark.parametrize("dt", sorted(DT))
def test_contiguous_pieces_at_any_alignment(dt, shift):
    es = torch.empty(0, dtype=DT[dt][1]).element_size()
    sizes = {1, 2, 3, 15, 16, 17, 16384 // es - 1, 16384 // es, 16384 // es + 1, 16384 // es + 3, 40000 // es + 1,
             (8 * 16384 + 5 * es) // es}
    for n in sorted(sizes):
        print(f"[copy forms] {dt} contiguous {n}, shift {shift}", flush=True)
        a, d = Obj(1, n, dt, shift[0], seed=n), Obj(1, n, dt, shift[1])
        _gather([a], [d], [copy(0, 0, 1, n)])
        d.check(a.t, n)
        z = Obj(1, n, dt, shift[1])
        _gather([], [z], [(ZERO, 0, -1, 0, -1, 0, 1, n, 0, 0, 0, 0)])
        z.check(torch.zeros_like(z.t), n)


@pytest.mark.parametrize("flags", [0, _lib.SR_OPT_TEMPORAL | _lib.SR_OPT_NO_XCD_INTERLEAVE])
@pytest.mark.parametrize("shift", [0, 1])
def test_recast_and_zero_rows(shift, flags):
    """RECAST bands with and without the f32 copy, beside ZERO bands."""
    for c in (1, 3, 4, 5, 16, 20, 32, 33, 64, 96, 100, 257, 683, 4096, 4100):
        rows = max(3, min(3000, 40000 // c))
        print(f"[copy forms] recast rows of {c}, shift {shift}", flush=True)
        a, b = Obj(rows, c, "f32", shift, seed=c), Obj(rows, 2 * c, "f32", seed=c + 1)
        d, h = Obj(rows, 3 * c, "f32", shift), Obj(rows, 3 * c, "bf16", shift)
        x, y = Obj(rows, c, "f32"), Obj(rows, c, "bf16")
        n = Obj(rows, 2 * c, "bf16", shift)
        _gather([a, b], [d, h, x, y, n],
                [(RECAST, 0, 0, 0, 1, 0, rows, c, 0, 0, 0, 0), (RECAST, 0, 1, 0, 1, 0, rows, c, 0, c, 0, c),
                 (ZERO, 0, -1, 0, -1, 0, rows, c, 0, 0, 0, 2 * c), (ZERO, 0, -1, 1, -1, 0, rows, c, 0, 0, 0, 2 * c),
                 (RECAST, 0, 1, 2, 3, 0, rows, c, 0, 0, 0, 0),
                 (RECAST, 0, 0, -1, 4, 0, rows, c, 0, 0, 0, 0), (RECAST, 0, 1, -1, 4, 0, rows, c, 0, 0, 0, c)],
                flags=flags)
        want = torch.cat([a.t, b.t[:, c:], torch.zeros_like(a.t)], 1)
        d.check(want, c)
        h.check(want.to(torch.bfloat16), c)
        x.check(b.t[:, :c], c)
        y.check(b.t[:, :c].to(torch.bfloat16), c)
        n.check(torch.cat([a.t, b.t[:, :c]], 1).to(torch.bfloat16), c)


@pytest.mark.parametrize("size,count,tile_bytes,max_blocks", [
    (7168, 40, 0, 0), (7169, 40, 0, 0),             # mean bytes of a tile: 256 lanes up to 7 KiB,
    (12288, 40, 0, 0), (12289, 40, 0, 0),           # 512 up to 12 KiB
    (16384, 5120, 0, 0), (16384, 5121, 0, 0),       # 512 up to 5120 tiles, 1024 above
    (16384, 6000, 0, 512), (16384, 6000, 0, 513),   # and for grids capped at 512
    (100, 3000, 4096, 0), (90000, 300, 65536, 0), (90001, 300, 65536, 24), (65539, 7, 16384, 5)])
def test_workgroups_by_tile_size(size, count, tile_bytes, max_blocks):
    """`count` contiguous pieces of `size` bytes in reverse order, a band of
    columns of as many bytes, split off and with both RECAST copies, beside
    zeros: on both sides of each line where the workgroups change."""
    print(f"[copy forms] {count} pieces of {size}, tile {tile_bytes}, {max_blocks} blocks", flush=True)
    a, d = Obj(count, size, "u8", seed=size), Obj(count, size, "u8")
    flat = [(COPY, 0, 0, 0, -1, 0, 1, size, count - 1 - k, 0, k, 0) for k in range(count)]
    _gather([a], [d], flat, tile_bytes, max_blocks=max_blocks)
    d.check(a.t.flip(0), "pieces")
    rows, c = 64, max(1, size * count // 64 // 4)
    b, x, y, h, z = (Obj(rows, 2 * c, "f32", seed=size + 1), Obj(rows, c, "f32"), Obj(rows, c, "f32"),
                     Obj(rows, c, "bf16"), Obj(rows, c, "f32", 1))
    _gather([b], [x, y, h, z], [copy(0, 0, rows, c), (RECAST, 0, 0, 1, 2, 0, rows, c, 0, c, 0, 0),
                                (ZERO, 0, -1, 3, -1, 0, rows, c, 0, 0, 0, 0)], tile_bytes, max_blocks=max_blocks)
    x.check(b.t[:, :c], "split")
    y.check(b.t[:, c:], "recast: f32")
    h.check(b.t[:, c:].to(torch.bfloat16), "recast: bf16")
    z.check(torch.zeros_like(z.t), "zeros")


@pytest.mark.parametrize("bands,rows,tile_bytes", [(300, 256, 4096), (100, 4096, 0), (5, 40000, 0)])
def test_items_read_ahead(bands, rows, tile_bytes):
    """Bands of 64 columns, an item each, split off and merged again: tiles of
    many items, of the last ones and of single items."""
    print(f"[copy forms] {bands} bands of {rows} rows, tile {tile_bytes}", flush=True)
    w = Obj(rows, 64 * bands, "f32", seed=bands)
    parts = [Obj(rows, 64, "f32") for _ in range(bands)]
    _gather([w], parts, [copy(0, k, rows, 64, sc=64 * k) for k in range(bands)], tile_bytes)
    for k, p in enumerate(parts):
        p.check(w.t[:, 64 * k:64 * k + 64], f"band {k}")
    d = Obj(rows, 64 * bands, "f32")
    _gather(parts, [d], [copy(k, 0, rows, 64, dc=64 * k) for k in range(bands)], tile_bytes)
    d.check(w.t, "merged")


@pytest.mark.parametrize("rows,tile_bytes", [(300, 0), (20400, 0), (20800, 0), (66000, 0), (1400, 65536)])
def test_streamed_lines(rows, tile_bytes):
    """A band of 1024 columns of wider rows beside a ZERO band, the rest of
    the rows untouched, and whole rows, in phases of few tiles, of a middling
    number (5121 to 16383) and of more."""
    print(f"[copy forms] bands of {rows} rows, tile {tile_bytes}", flush=True)
    a, d = Obj(rows, 1024, "f32", seed=rows), Obj(rows, 3072, "f32")
    flat, e = Obj(1, 1024 * (rows // 8), "f32", seed=1), Obj(1, 1024 * (rows // 8), "f32")
    _gather([a, flat], [d, e], [copy(0, 0, rows, 1024, dc=1024), (ZERO, 0, -1, 0, -1, 0, rows, 1024, 0, 0, 0, 2048),
                                copy(1, 1, 1, flat.cols)], tile_bytes, flags=_lib.SR_OPT_SKIP_COVERAGE)
    assert bool((d.t[:, :1024].contiguous().view(torch.uint8) == POISON).all()), "columns before the band"
    d.t[:, :1024] = 0
    d.check(torch.cat([torch.zeros_like(a.t), a.t, torch.zeros_like(a.t)], 1), "band")
    e.check(flat.t, "whole rows")


@pytest.mark.parametrize("rows,tile_bytes", [(19000, 4096), (66000, 0), (5000, 0)])
@pytest.mark.parametrize("cols", [1026, 1025, 1032, 33])
def test_two_pass_records(cols, rows, tile_bytes):
    """Bands in large phases, where rows in 8-byte vectors and RECAST into bf16
    alone have records of two passes, and in a small one: split, merged, and
    rounded, side by side with pieces of one pass."""
    print(f"[copy forms] bands of {cols}, {rows} rows, tile {tile_bytes}", flush=True)
    rows = rows * (31 if cols == 33 else 1)
    w = Obj(rows, 2 * cols, "f32", seed=cols)
    x, h, d, f = Obj(rows, cols, "f32"), Obj(rows, cols, "bf16"), Obj(rows, 2 * cols, "bf16"), Obj(rows, cols, "f32")
    _gather([w], [x, h, f], [copy(0, 0, rows, cols, sc=cols), (RECAST, 0, 0, -1, 1, 0, rows, cols, 0, 0, 0, 0),
                             copy(0, 2, rows, cols)], tile_bytes)
    x.check(w.t[:, cols:], "split")
    h.check(w.t[:, :cols].to(torch.bfloat16), "rounded")
    e = Obj(rows, 2 * cols, "f32")
    _gather([x, f], [d, e], [(RECAST, 0, 1, -1, 0, 0, rows, cols, 0, 0, 0, 0),
                             (RECAST, 0, 0, -1, 0, 0, rows, cols, 0, 0, 0, cols), copy(1, 1, rows, cols),
                             copy(0, 1, rows, cols, dc=cols)], tile_bytes)
    d.check(w.t.to(torch.bfloat16), "merged, rounded")
    e.check(w.t, "merged")


def test_rows_two_gib_apart():
    """Rows so long that a tile's rows span 2 GiB: 64-bit offsets, beside a
    band of the same rows that is near enough within a smaller tile."""
    rows, cols = 3, 900_000_001
    print("[copy forms] rows 0.9 GB apart", flush=True)
    src = torch.zeros(rows * cols, dtype=torch.uint8, device="cuda").view(rows, cols)
    bands = {0: 7, 1000: 16, 5000: 200, cols - 40001: 40001}
    g = torch.Generator("cuda").manual_seed(1)
    for at, w in bands.items():
        src[:, at:at + w] = torch.randint(0, 256, (rows, w), generator=g, device="cuda", dtype=torch.uint8)

    class Whole:
        pass
    s = Whole()
    s.rows, s.cols, s.dt, s.t = rows, cols, "u8", src
    dst = [Obj(rows, w, "u8") for w in bands.values()]
    _gather([s], dst, [copy(0, k, rows, w, sc=at) for k, (at, w) in enumerate(bands.items())])
    for d, (at, w) in zip(dst, bands.items()):
        d.check(src[:, at:at + w], f"band at {at}")
    del s, src
    torch.cuda.empty_cache()
