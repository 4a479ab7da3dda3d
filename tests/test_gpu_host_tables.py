"""Small phases: tables written by the host at the first launch on new
pointers, device tables from the second.  Around the tile count where the
other route begins, both give torch's bytes, also where bindings take turns
without a host synchronisation, and where launches of one binding are on two
streams.  All exact."""
import ctypes

import pytest
import torch

from suika_amd import _lib

pytestmark = pytest.mark.gpu

LIMIT = 2048     # tiles up to which the host writes the tables
TILE = 4096
vp = ctypes.c_void_p


class Plan:
    """[rows, cols] f32 source: columns split off as f32, the rest recast into
    f32 + bf16, zero-filled rows, and whole rows up to `tiles` tiles."""

    def __init__(self, tiles, cols=333, rows=40, split=100):
        self.rows, self.cols, self.split = rows, cols, split
        piece = _lib.SrPiece
        small = -(-rows * split * 4 // TILE) + -(-rows * (cols - split) * 4 // TILE) + 1
        self.fill = (tiles - small) * TILE // 4
        assert self.fill > 0
        f32, bf16 = _lib.SR_DT_F32, _lib.SR_DT_BF16
        T = _lib.SrTensor
        S = (T * 2)(T(rows, cols, f32, 0), T(1, self.fill, f32, 0))
        D = (T * 4)(T(rows + 3, split, f32, 0), T(rows, cols - split, f32, 0), T(rows, cols - split, bf16, 0),
                    T(1, self.fill, f32, 0))
        P = [piece(_lib.SR_PIECE_COPY, 0, 0, 0, -1, 0, rows, split, 0, 0, 0, 0),
             piece(_lib.SR_PIECE_ZERO, 0, -1, 0, -1, 0, 3, split, 0, 0, rows, 0),
             piece(_lib.SR_PIECE_RECAST, 0, 0, 1, 2, 0, rows, cols - split, 0, split, 0, 0),
             piece(_lib.SR_PIECE_COPY, 0, 1, 3, -1, 0, 1, self.fill, 0, 0, 0, 0)]
        opt = _lib.SrPlanOptions(TILE, 0, 0, 0)
        self.h = vp()
        self.L = _lib.lib()
        _lib.check(self.L.sr_plan_create(S, 2, D, 4, 1, (piece * 4)(*P), 4, ctypes.byref(opt), ctypes.byref(self.h)),
                   "plan")
        n = ctypes.c_uint64()
        _lib.check(self.L.sr_plan_peer_bytes(self.h, 0, ctypes.byref(n)), "peer bytes")
        self.peer_bytes = n.value

    def src(self, seed):
        g = torch.Generator("cuda").manual_seed(seed)
        return [torch.randn(self.rows, self.cols, generator=g, device="cuda"),
                torch.randn(1, self.fill, generator=g, device="cuda")]

    def dst(self):
        w = self.cols - self.split
        return [torch.full((self.rows + 3, self.split), 7.0, device="cuda"),
                torch.full((self.rows, w), 7.0, device="cuda"),
                torch.full((self.rows, w), 7.0, device="cuda", dtype=torch.bfloat16),
                torch.full((1, self.fill), 7.0, device="cuda")]

    def gather(self, src, dst):
        self._call(self.L.sr_gather, src, dst)

    def _call(self, fn, a, b):
        A, B = (vp * len(a))(*[t.data_ptr() for t in a]), (vp * len(b))(*[t.data_ptr() for t in b])
        _lib.check(fn(self.h, A, B, vp(torch.cuda.current_stream().cuda_stream)), "call")

    def exchange(self, src, buf, dst):
        self._call(self.L.sr_pack, src, [buf])
        self._call(self.L.sr_unpack, [buf], dst)

    def check(self, src, dst):
        want = [torch.cat([src[0][:, :self.split], src[0].new_zeros(3, self.split)]), src[0][:, self.split:],
                src[0][:, self.split:].to(torch.bfloat16), src[1]]
        for k, (a, b) in enumerate(zip(dst, want)):
            assert torch.equal(a, b), f"destination {k}"

    def close(self):
        torch.cuda.synchronize()
        self.L.sr_plan_destroy(self.h)


@pytest.mark.parametrize("cols,split", [(333, 100), (336, 96), (40, 3)])
@pytest.mark.parametrize("tiles", [64, LIMIT - 1, LIMIT, LIMIT + 1])
def test_bindings_in_turn(tiles, cols, split):
    print(f"[gpu host tables] {tiles} tiles, {cols} columns at {split}", flush=True)
    p = Plan(tiles, cols=cols, split=split)
    try:
        srcs, dsts = [p.src(i) for i in range(3)], [p.dst() for _ in range(3)]
        for i in (0, 1, 2, 1, 1, 1, 0, 2, 2):   # first, second and third launches of a binding, and returns to it
            for t in dsts[i]:
                t.fill_(7)
            p.gather(srcs[i], dsts[i])
        for s, d in zip(srcs, dsts):
            p.check(s, d)
        bufs = [torch.empty(p.peer_bytes, dtype=torch.uint8, device="cuda") for _ in range(2)]
        for i in (0, 1, 1, 0):
            for t in dsts[i]:
                t.fill_(7)
            p.exchange(srcs[i], bufs[i], dsts[i])
        for i in range(2):
            p.check(srcs[i], dsts[i])
    finally:
        p.close()


@pytest.mark.parametrize("tiles", [64, LIMIT, LIMIT + 1])
@pytest.mark.parametrize("first", [1, 2, 3])
def test_two_streams(tiles, first):
    """Launches of one binding on a stream that is held up by other work and
    then on a free one, where other bindings follow, with no host wait; then a
    plan destroyed while its first stream still runs, and its table memory in
    another plan's hands."""
    print(f"[gpu host tables] two streams, {tiles} tiles, {first} launches on the first", flush=True)
    p, a, b = Plan(tiles), Plan(tiles), Plan(tiles)
    srcs, dsts = [p.src(i) for i in range(3)], [p.dst() for _ in range(3)]
    last_src, last_dst = [p.src(i) for i in (3, 4)], [p.dst() for _ in range(2)]
    held = torch.randn(1 << 28, device="cuda")
    copy = torch.empty_like(held)
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    try:
        with torch.cuda.stream(s1):
            p.gather(srcs[2], dsts[2])
            for _ in range(8):
                copy.copy_(held)
            for _ in range(first):
                p.gather(srcs[0], dsts[0])
        with torch.cuda.stream(s2):
            p.gather(srcs[0], dsts[0])
            for i in (1, 1, 2, 2, 1):
                p.gather(srcs[i], dsts[i])
        with torch.cuda.stream(s1):
            for _ in range(8):
                copy.copy_(held)
            for _ in range(first):
                a.gather(last_src[0], last_dst[0])
        with torch.cuda.stream(s2):
            a.gather(last_src[0], last_dst[0])
        a.L.sr_plan_destroy(a.h)
        with torch.cuda.stream(s2):
            for _ in range(2):
                b.gather(last_src[1], last_dst[1])
        torch.cuda.synchronize()
        for s, d in zip(srcs + last_src, dsts + last_dst):
            p.check(s, d)
    finally:
        p.close()
        b.close()


def test_graph_capture_stays_refused():
    """A plan that has run is refused on a capturing stream before any device
    work: the capture stays valid, and so does the plan."""
    print("[gpu host tables] capture refused", flush=True)
    p = Plan(64)
    try:
        src, dst = p.src(0), p.dst()
        mark = torch.zeros(64, device="cuda")
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            for _ in range(2):   # bound by the host, then on the device
                p.gather(src, dst)
                stream.synchronize()
                g = torch.cuda.CUDAGraph()
                with torch.cuda.graph(g, stream=stream):
                    mark.add_(1.0)
                    with pytest.raises(_lib.ReshardError, match="cannot be captured"):
                        p.gather(src, dst)
                for _ in range(2):
                    g.replay()
            src[0].add_(1.0)
            p.gather(src, dst)
            stream.synchronize()
        p.check(src, dst)
        assert torch.equal(mark, torch.full_like(mark, 4.0))
    finally:
        p.close()


def test_first_use_in_a_capture():
    """A small phase whose first use is captured has tables that the graph's
    launches build on the device: each replay gives the bytes of the sources
    as they then are, with other plans' launches and host waits between."""
    print("[gpu host tables] first use captured", flush=True)
    p, q, other = Plan(64), Plan(64), Plan(64)
    src, dst, back = p.src(0), p.dst(), p.dst()
    buf = torch.empty(q.peer_bytes, dtype=torch.uint8, device="cuda")
    new = [p.src(i) for i in (1, 2, 3)]
    busy = p.dst()
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    try:
        with torch.cuda.stream(stream):
            with torch.cuda.graph(g, stream=stream, capture_error_mode="relaxed"):
                p.gather(src, dst)
                q.exchange(src, buf, back)
            for fresh in new:
                for a, b in zip(src, fresh):
                    a.copy_(b)
                for t in dst + back:
                    t.fill_(7)
                buf.fill_(0xA5)
                g.replay()
                other.gather(fresh, busy)
                torch.cuda.synchronize()
                p.check(fresh, dst)
                p.check(fresh, back)
                other.check(fresh, busy)
    finally:
        torch.cuda.synchronize()
        del g
        for plan in (p, q, other):
            plan.close()


@pytest.mark.parametrize("cols", [512, 513, 514, 516])
@pytest.mark.parametrize("rows", [700, 5000])
def test_device_tables_rebound(rows, cols):
    """Above the limit, in phases of a few and of many thousand tiles: columns
    put together, and the same rounded, in row groups, and zero-filled rows,
    with bindings taking turns and no host wait."""
    parts, zeros = 3, 2
    print(f"[gpu host tables] {parts} x [{rows}, {cols}] put together, pointers in turn", flush=True)
    L, T, piece = _lib.lib(), _lib.SrTensor, _lib.SrPiece
    f32, bf16 = _lib.SR_DT_F32, _lib.SR_DT_BF16
    S = (T * parts)(*[T(rows, cols, f32, 0)] * parts)
    D = (T * 2)(T(rows + zeros, parts * cols, f32, 0), T(rows, parts * cols, bf16, 0))
    P = [piece(_lib.SR_PIECE_COPY, 0, k, 0, -1, 0, rows, cols, 0, 0, 0, k * cols) for k in range(parts)]
    P += [piece(_lib.SR_PIECE_RECAST, 0, k, -1, 1, 0, rows, cols, 0, 0, 0, k * cols) for k in range(parts)]
    P.append(piece(_lib.SR_PIECE_ZERO, 0, -1, 0, -1, 0, zeros, parts * cols, 0, 0, rows, 0))
    h, n = vp(), ctypes.c_uint64()
    _lib.check(L.sr_plan_create(S, parts, D, 2, 1, (piece * len(P))(*P), len(P),
                                ctypes.byref(_lib.SrPlanOptions(TILE, 0, 0, 0)), ctypes.byref(h)), "plan")

    def call(fn, a, b):
        A, B = (vp * len(a))(*[t.data_ptr() for t in a]), (vp * len(b))(*[t.data_ptr() for t in b])
        _lib.check(fn(h, A, B, vp(torch.cuda.current_stream().cuda_stream)), "call")

    try:
        _lib.check(L.sr_plan_peer_bytes(h, 0, ctypes.byref(n)), "peer bytes")
        assert 2 * parts * rows * cols * 4 // TILE > LIMIT
        g = torch.Generator("cuda").manual_seed(cols)
        srcs = [[torch.randn(rows, cols, generator=g, device="cuda") for _ in range(parts)] for _ in range(3)]
        dsts = [[torch.empty(rows + zeros, parts * cols, device="cuda"),
                 torch.empty(rows, parts * cols, device="cuda", dtype=torch.bfloat16)] for _ in range(3)]
        bufs = [torch.empty(n.value, dtype=torch.uint8, device="cuda") for _ in range(3)]
        for route in ("gather", "exchange"):
            for i in (0, 1, 2, 1, 1, 0, 2, 2, 0):
                for t in dsts[i]:
                    t.fill_(7)
                if route == "gather":
                    call(L.sr_gather, srcs[i], dsts[i])
                else:
                    bufs[i].fill_(0xA5)
                    call(L.sr_pack, srcs[i], [bufs[i]])
                    call(L.sr_unpack, [bufs[i]], dsts[i])
            for i, (s, d) in enumerate(zip(srcs, dsts)):
                want = torch.cat(s, 1)
                assert torch.equal(d[0], torch.cat([want, want.new_zeros(zeros, parts * cols)])), (route, i, "copy")
                assert torch.equal(d[1], want.to(torch.bfloat16)), (route, i, "rounded")
    finally:
        torch.cuda.synchronize()
        L.sr_plan_destroy(h)
