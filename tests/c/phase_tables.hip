// The engine's host code over a model of the HIP runtime, on the CPU.
//
// The program includes the engine's source, compiled for the host only, and
// defines the runtime calls that it makes.  Streams hold their work back: an
// operation runs when something waits for it, or at the end in an order that
// the scenario picks, so whatever the streams and events do not order shows as
// wrong bytes.  Kernels run as plain loops over the tables that the launch
// names.  Every allocation ends in a guard that is checked after each call.
//
// Usage: phase_tables SCENARIO; prints "ok" and exits 0, or says what differs.
#include "../../suika_amd/csrc/reshard.hip"

#include <cstdlib>
#include <functional>
#include <map>
#include <set>

namespace model {

[[noreturn]] void die(const char* what) {
  std::printf("FAILED: %s\n", what);
  std::exit(1);
}

// ---- memory
constexpr size_t kGuard = 65536;
struct Alloc {
  size_t bytes;
};
std::map<unsigned char*, Alloc> allocs;

void* alloc(size_t bytes) {
  unsigned char* p = static_cast<unsigned char*>(std::aligned_alloc(4096, (bytes + kGuard + 4095) / 4096 * 4096));
  std::memset(p, 0xEE, bytes);
  std::memset(p + bytes, 0xC3, kGuard);
  allocs[p] = {bytes};
  return p;
}

void check_guards(const char* when) {
  static const std::vector<unsigned char> whole(kGuard, 0xC3);
  for (auto& [p, a] : allocs)
    if (std::memcmp(p + a.bytes, whole.data(), kGuard)) {
      std::printf("a block of %zu bytes was written past its end (%s)\n", a.bytes, when);
      die("guard");
    }
}

// ---- work
struct Work {
  std::function<void()> run;
  std::vector<int> after;
  bool done = false;
};
std::vector<Work> work;

struct Stream {
  int last = -1;
  bool capturing = false;
};
struct Event {
  int at = -1;
};
Stream streams[8];   // 0: the null stream
int n_streams = 4;   // further ones are made by the engine

Stream* of(hipStream_t s) { return s ? reinterpret_cast<Stream*>(s) : &streams[0]; }
hipStream_t handle(int i) { return i ? reinterpret_cast<hipStream_t>(&streams[i]) : nullptr; }

void add(hipStream_t s, std::function<void()> run, int also = -1) {
  Stream* st = of(s);
  Work w;
  w.run = std::move(run);
  if (st->last >= 0) w.after.push_back(st->last);
  if (also >= 0) w.after.push_back(also);
  work.push_back(std::move(w));
  st->last = int(work.size()) - 1;
}

void finish(int i) {
  if (i < 0 || work[i].done) return;
  for (int d : work[i].after) finish(d);
  work[i].done = true;
  if (work[i].run) work[i].run();
}

// Everything still held back, streams in the given order.
void drain(std::initializer_list<int> order) {
  for (int s : order) finish(streams[s].last);
  for (int s = 0; s < 8; ++s) finish(streams[s].last);
}

bool capturing() {
  for (const Stream& s : streams)
    if (s.capturing) return true;
  return false;
}

// ---- kernels, one operation each
struct Launch {
  const void* fn;
  void** args;
  template <typename T> T arg(int i) const { return *static_cast<T*>(args[i]); }
};

// The objects that the launches of the present call write.
typedef std::vector<std::pair<uint64_t, uint64_t>> Spans;
Spans writes;

void check_write(const Spans& spans, uint64_t to, size_t n) {
  for (const auto& [lo, hi] : spans)
    if (to >= lo && to + n <= hi) return;
  die("a launch whose tables are no longer those of its call");
}

void copy_tiles(const DevItem* items, const DevTile* tiles, uint32_t n, const Spans& spans) {
  for (uint32_t i = 0; i < n; ++i) {
    const DevTile& t = tiles[i];
    const DevItem& it = items[t.item];
    const uint32_t nbytes = t.info & kTileBytesMask, kind = it.flags & 0xfu;
    for (uint32_t b = 0, run; b < nbytes; b += run) {   // the bytes of one row
      uint64_t from = t.src + b, to = t.dst ? t.dst + b : 0, half = it.dst2 + ((from - it.src) >> 1);
      run = nbytes;
      if (it.row_bytes) {
        const uint64_t x = t.dst + b, row = t.src + x / it.row_bytes, col = x % it.row_bytes;
        from = it.src + row * it.src_stride + col;
        to = it.dst ? it.dst + row * it.dst_stride + col : 0;
        half = it.dst2 + row * it.dst2_stride + (col >> 1);
        run = uint32_t(std::min<uint64_t>(nbytes - b, it.row_bytes - col));
      }
      if (to) check_write(spans, to, run);
      if (to && kind == kKindZero) std::memset(reinterpret_cast<void*>(to), 0, run);
      if (to && kind != kKindZero) std::memcpy(reinterpret_cast<void*>(to), reinterpret_cast<void*>(from), run);
      if (kind != kKindRecast) continue;
      check_write(spans, half, run / 2);
      for (uint32_t k = 0; k < run; k += 4) {
        uint32_t u;
        std::memcpy(&u, reinterpret_cast<void*>(from + k), 4);
        const uint16_t h = uint16_t((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
        std::memcpy(reinterpret_cast<void*>(half + k / 2), &h, 2);
      }
    }
  }
}

std::function<void()> body(const Launch& l, dim3 grid, dim3 block) {
  if (l.fn == reinterpret_cast<const void*>(sr_table_copy_kernel)) {
    auto from = l.arg<const unsigned char*>(0);
    auto to = l.arg<unsigned char*>(1);
    const size_t bytes = size_t(l.arg<uint32_t>(2)) * 16;
    if (size_t(grid.x) * block.x * 16 < bytes) die("table copy: grid too small");
    return [=] { std::memcpy(to, from, bytes); };
  }
  if (l.fn == reinterpret_cast<const void*>(sr_offsets_kernel)) {
    auto begin = l.arg<const uint32_t*>(0);
    auto list = l.arg<const uint32_t*>(1);
    auto payload = l.arg<const uint64_t*>(2);
    auto offset = l.arg<uint64_t*>(3);
    const uint32_t peers = grid.x;
    return [=] {
      for (uint32_t p = 0; p < peers; ++p) {
        uint64_t at = 0;
        for (uint32_t i = begin[p]; i < begin[p + 1]; ++i) {
          offset[list[i]] = at;
          at += (payload[list[i]] + kBufAlign - 1) / kBufAlign * kBufAlign;
        }
      }
    };
  }
  if (l.fn == reinterpret_cast<const void*>(sr_tile_emit_kernel)) {
    auto rel = l.arg<const DevRel*>(0);
    auto base = l.arg<const uint64_t*>(1);
    auto chunks = l.arg<const EmitChunk*>(2);
    const uint32_t n_chunks = l.arg<uint32_t>(3);
    auto tiles = l.arg<DevTile*>(4);
    auto ptrs = l.arg<const uint64_t*>(5);
    auto offset = l.arg<const uint64_t*>(6);
    auto items = l.arg<DevItem*>(7);
    return [=] {
      for (uint32_t c = 0; c < n_chunks; ++c) {
        const DevRel& h = rel[chunks[c].item];
        uint32_t op;
        const DevItem item = bind_item(h, ptrs, offset, op);
        items[chunks[c].item] = item;
        const uint64_t cnt = base[chunks[c].item + 1] - base[chunks[c].item];
        const uint64_t first = base[chunks[c].item] - h.group_index * cnt + h.group_index;
        const uint64_t j0 = uint64_t(chunks[c].chunk) * kEmitTiles;
        for (uint64_t j = j0; j < std::min<uint64_t>(cnt, j0 + kEmitTiles); ++j)
          tiles[first + j * h.group_size] = tile_record(item, h, chunks[c].item, op, j);
      }
    };
  }
#define PHASES(NT, B, U)                                          \
  reinterpret_cast<const void*>(sr_pack_kernel<NT, B, U>),        \
      reinterpret_cast<const void*>(sr_unpack_kernel<NT, B, U>),  \
      reinterpret_cast<const void*>(sr_gather_kernel<NT, B, U>)
  static const std::set<const void*> copies = {PHASES(true, 1024, 1),  PHASES(true, 512, 2),  PHASES(true, 256, 1),
                                               PHASES(true, 1024, 2),  PHASES(false, 1024, 1), PHASES(false, 512, 2),
                                               PHASES(false, 256, 1), PHASES(false, 1024, 2)};
  if (copies.count(l.fn)) {
    auto items = l.arg<const DevItem*>(0);
    auto tiles = l.arg<const DevTile*>(1);
    const uint32_t n = l.arg<uint32_t>(2);
    if (uint64_t(grid.x) * block.x > 0xffffffffu || n > l.arg<uint32_t>(4)) die("copy: grid");
    return [=, spans = writes] { copy_tiles(items, tiles, n, spans); };
  }
  die("unknown kernel");
}

}  // namespace model

extern "C" {

hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error of the model"; }
hipError_t hipMalloc(void** p, size_t n) {
  if (model::capturing()) return *p = nullptr, hipErrorStreamCaptureUnsupported;
  return *p = model::alloc(n), hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return hipMalloc(p, n); }
hipError_t hipFree(void* p) {
  model::check_guards("free");
  model::drain({});
  model::allocs.erase(static_cast<unsigned char*>(p));
  return std::free(p), hipSuccess;
}
hipError_t hipHostFree(void* p) { return hipFree(p); }
hipError_t hipGetSymbolAddress(void** p, const void*) {
  static void* scratch_memory = model::alloc(SR_SCRATCH_BYTES);
  return *p = scratch_memory, hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  return *e = reinterpret_cast<hipEvent_t>(new model::Event()), hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) { return delete reinterpret_cast<model::Event*>(e), hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  return reinterpret_cast<model::Event*>(e)->at = model::of(s)->last, hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  return model::finish(reinterpret_cast<model::Event*>(e)->at), hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  const int at = reinterpret_cast<model::Event*>(e)->at;
  if (at >= 0) model::add(s, nullptr, at);
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  return *s = model::handle(model::n_streams++), hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* c) {
  return *c = model::of(s)->capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone, hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t s) {
  const int last = model::of(s)->last;
  return last < 0 || model::work[last].done ? hipSuccess : hipErrorNotReady;
}
hipError_t hipStreamSynchronize(hipStream_t s) { return model::finish(model::of(s)->last), hipSuccess; }
hipError_t hipMemcpyAsync(void* to, const void* from, size_t n, hipMemcpyKind, hipStream_t s) {
  if (model::of(s)->capturing) return hipSuccess;   // a node of the graph
  bool pinned = false;
  for (auto& [p, a] : model::allocs) pinned |= from >= p && from < p + a.bytes;
  model::add(s, [=] { std::memcpy(to, from, n); });
  if (!pinned) model::finish(model::of(s)->last);
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* fn, dim3 grid, dim3 block, void** args, size_t, hipStream_t s) {
  auto run = model::body(model::Launch{fn, args}, grid, block);
  if (!model::of(s)->capturing) model::add(s, std::move(run));
  return hipSuccess;
}

static struct {
  dim3 grid, block;
  size_t shmem;
  hipStream_t stream;
} g_call;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t m, hipStream_t s) {
  return g_call = {g, b, m, s}, hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* m, hipStream_t* s) {
  return *g = g_call.grid, *b = g_call.block, *m = g_call.shmem, *s = g_call.stream, hipSuccess;
}
void** __hipRegisterFatBinary(const void*) { return nullptr; }
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*, void*, int*) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void**) {}

}  // extern "C"

// ------------------------------------------------------------------ scenarios

namespace {

using model::check_guards;
using model::die;
using model::drain;
using model::handle;

void ok(int rc, const char* what) {
  if (rc != SR_OK) {
    std::printf("%s: %s\n", what, sr_last_error());
    die("call");
  }
  check_guards(what);
}

// A plan of four pieces of [rows, 2 * cols] f32 tensors -- a copied band, a
// zeroed band, a band rounded on the way, a whole tensor -- of about `tiles`
// records in each phase, with its objects (several sets of them).
struct Job {
  static constexpr uint32_t kTile = 4096;
  uint64_t rows, cols, fill;
  sr_plan* plan = nullptr;
  std::vector<std::vector<std::vector<unsigned char>>> src, dst;
  std::vector<std::vector<unsigned char>> bufs;

  explicit Job(uint64_t tiles, int sets, uint64_t cols_ = 25, int seed = 1) : rows(40), cols(cols_) {
    const uint64_t band = (rows * cols * 4 + kTile - 1) / kTile;
    fill = (tiles - 3 * band) * kTile;
    const sr_tensor s[2] = {{rows, 2 * cols, SR_DT_F32, 0}, {1, fill, SR_DT_U8, 0}};
    const sr_tensor d[4] = {{rows, 2 * cols, SR_DT_F32, 0}, {rows, cols, SR_DT_F32, 0}, {rows, cols, SR_DT_BF16, 0},
                            {1, fill, SR_DT_U8, 0}};
    const sr_piece p[4] = {{SR_PIECE_COPY, 0, 0, 0, -1, 0, rows, cols, 0, cols, 0, 0},
                           {SR_PIECE_ZERO, 0, -1, 0, -1, 0, rows, cols, 0, 0, 0, cols},
                           {SR_PIECE_RECAST, 0, 0, 1, 2, 0, rows, cols, 0, 0, 0, 0},
                           {SR_PIECE_COPY, 0, 1, 3, -1, 0, 1, fill, 0, 0, 0, 0}};
    sr_plan_options opt{};
    opt.tile_bytes = kTile;
    ok(sr_plan_create(s, 2, d, 4, 1, p, 4, &opt, &plan), "plan");
    uint64_t n = 0;
    ok(sr_plan_peer_bytes(plan, 0, &n), "peer bytes");
    uint32_t x = uint32_t(seed);
    for (int k = 0; k < sets; ++k) {
      src.push_back({std::vector<unsigned char>(rows * 2 * cols * 4), std::vector<unsigned char>(fill)});
      for (size_t i = 0; i + 4 <= src[k][0].size(); i += 4) {
        const float f = float((x = x * 1664525u + 1013904223u) >> 8) / 65536.0f - 128.0f;
        std::memcpy(&src[k][0][i], &f, 4);
      }
      for (unsigned char& c : src[k][1]) c = (unsigned char)((x = x * 1664525u + 1013904223u) >> 24);
      dst.push_back({std::vector<unsigned char>(rows * 2 * cols * 4), std::vector<unsigned char>(rows * cols * 4),
                     std::vector<unsigned char>(rows * cols * 2), std::vector<unsigned char>(fill)});
      bufs.push_back(std::vector<unsigned char>(n + 32));
      clear(k);
    }
  }
  ~Job() { close(); }
  void close() {
    sr_plan_destroy(plan);
    plan = nullptr;
    check_guards("destroy");
  }

  void clear(int k) {
    for (auto& v : dst[k]) std::fill(v.begin(), v.end(), 0x77);
  }
  unsigned char* buf(int k) {
    return reinterpret_cast<unsigned char*>((reinterpret_cast<uintptr_t>(bufs[k].data()) + 15) & ~uintptr_t(15));
  }
  void writes_dst(int k) {
    model::writes.clear();
    for (const auto& v : dst[k]) {
      const uint64_t at = reinterpret_cast<uintptr_t>(v.data());
      model::writes.push_back({at, at + v.size()});
    }
  }
  int gather(int k, int stream) {
    const void* s[2] = {src[k][0].data(), src[k][1].data()};
    void* d[4] = {dst[k][0].data(), dst[k][1].data(), dst[k][2].data(), dst[k][3].data()};
    writes_dst(k);
    return sr_gather(plan, s, d, handle(stream));
  }
  int pack(int k, int stream) {
    const void* s[2] = {src[k][0].data(), src[k][1].data()};
    void* b[1] = {buf(k)};
    const uint64_t at = reinterpret_cast<uintptr_t>(buf(k));
    model::writes = {{at, at + bufs[k].size() - 16}};
    return sr_pack(plan, s, b, handle(stream));
  }
  int unpack(int k, int stream) {
    const void* b[1] = {buf(k)};
    void* d[4] = {dst[k][0].data(), dst[k][1].data(), dst[k][2].data(), dst[k][3].data()};
    writes_dst(k);
    return sr_unpack(plan, b, d, handle(stream));
  }
  void check(int k, const char* what) {
    bool same = dst[k][3] == src[k][1];
    for (uint64_t r = 0; r < rows; ++r)
      for (uint64_t c = 0; c < cols; ++c) {
        const unsigned char* row = src[k][0].data() + r * 2 * cols * 4;
        const unsigned char zero[4] = {};
        same &= !std::memcmp(&dst[k][0][(r * 2 * cols + c) * 4], row + (cols + c) * 4, 4);
        same &= !std::memcmp(&dst[k][0][(r * 2 * cols + cols + c) * 4], zero, 4);
        same &= !std::memcmp(&dst[k][1][(r * cols + c) * 4], row + c * 4, 4);
        uint32_t u;
        std::memcpy(&u, row + c * 4, 4);
        const uint16_t h = uint16_t((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
        same &= !std::memcmp(&dst[k][2][(r * cols + c) * 2], &h, 2);
      }
    if (!same) {
      std::printf("set %d: %s\n", k, what);
      die("bytes");
    }
  }
};

constexpr uint64_t kFew = 64, kMost = kHostTableTiles, kMany = kHostTableTiles + 40;

// Every route gives the same bytes: first, second and third launches of a
// binding and returns to it, gather and pack + unpack.
void routes() {
  for (uint64_t tiles : {kFew, kMost, kMany})
    for (uint64_t cols : {3, 16, 25, 64}) {
      Job j(tiles, 3, cols);
      for (int k : {0, 1, 2, 1, 1, 1, 0, 2, 2}) {
        j.clear(k);
        ok(j.gather(k, 1), "gather");
        drain({});
        j.check(k, "gather");
      }
      for (int k : {0, 1, 1, 2, 0}) {
        j.clear(k);
        ok(j.pack(k, 1), "pack");
        ok(j.unpack(k, 1), "unpack");
        drain({});
        j.check(k, "pack and unpack");
      }
    }
}

// A first use on a capturing stream that fails after its table memory was
// taken (from blocks that plans before it left), then the same calls again.
void capture_fails() {
  { Job before(kFew, 1); ok(before.gather(0, 1), "gather"); ok(before.gather(0, 1), "gather"); drain({}); }
  Job j(kMost, 1);
  model::streams[1].capturing = true;
  if (j.pack(0, 1) != SR_EHIP) die("a pack whose buffer offsets find no memory in a capture");
  check_guards("failed capture");
  model::streams[1].capturing = false;
  for (int i = 0; i < 3; ++i) {
    j.clear(0);
    ok(j.pack(0, 1), "pack");
    ok(j.unpack(0, 1), "unpack");
    drain({});
    j.check(0, "after a failed capture");
  }
}

// Launches of one binding on two streams, then other bindings, all while the
// first stream's work is held back; at last the plan goes, and its memory to
// another plan.
void two_streams(uint64_t tiles, int first, int repeats) {
  Job j(tiles, 3);
  ok(j.gather(2, 1), "gather");   // a binding before, so that this one is not the plan's first
  for (int i = 0; i < first; ++i) ok(j.gather(0, 1), "gather");
  for (int i = 0; i < repeats; ++i) ok(j.gather(0, 2), "gather");
  for (int k : {1, 2, 1})
    for (int i = 0; i < 2; ++i) ok(j.gather(k, 2), "gather");
  drain({2, 1});
  for (int k = 0; k < 3; ++k) j.check(k, "two streams");

  Job a(tiles, 2);
  ok(a.gather(1, 1), "gather");
  for (int i = 0; i < first; ++i) ok(a.gather(0, 1), "gather");
  ok(a.gather(0, 2), "gather");
  a.close();
  Job b(tiles, 1, 25, 9);
  for (int i = 0; i < 2; ++i) ok(b.gather(0, 3), "gather");
  drain({3, 2, 1});
  a.check(0, "destroyed while a stream still runs");
  b.check(0, "memory of a destroyed plan");
}

}  // namespace

int main(int argc, char** argv) {
  const std::string what = argc > 1 ? argv[1] : "";
  if (what == "routes") routes();
  else if (what == "capture_fails") capture_fails();
  else if (what == "two_streams_small") for (int first : {1, 2, 3}) for (int n : {0, 1, 2}) two_streams(kFew, first, n);
  else if (what == "two_streams_large") for (int first : {1, 2, 3}) for (int n : {0, 1, 2}) two_streams(kMany, first, n);
  else die("no such scenario");
  check_guards("end");
  std::puts("ok");
  return 0;
}
