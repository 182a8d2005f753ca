// gsofa_copy.hip -- copies between host arrays and the device through pinned
// staging, and the small host-side pools behind them (host code, one kernel).
//
// Callers' arrays are pageable.  The runtime's own pageable copies take 115 us
// for 256 KB and 400 us for 1 MB, where a pinned one takes 13 and 26, and each
// copy is a call and a wait of its own.  So all arrays of a call go together:
//   small totals (a matrix of thousands of rows) by one kernel between the
//     arrays and one pinned buffer: the fetch of a 16 x 16 grid 160 -> 17 us,
//     its upload 60 -> 19;
//   the rest in chunks of at most 4 MB, each moved by a kernel while the thread
//     copies the previous one out.  (A copy of the runtime's is a kernel too,
//     but 10 us apart from the next and one for each array.)  A single thread
//     that first touches the destination moves 14 GB/s, so larger totals take
//     up to kThreads threads.
// Vertex numbers make up nearly all of a result, and neighbouring ones are
// close: rows are sorted and follow each other.  They cross the link as 16-bit
// offsets, 64 to a base, and the thread that would copy them adds the base
// (host rate of either: 120 GB/s at eight threads, twice the link's); a block of
// a wider range, as where a row of far-spread columns ends, crosses as it is.
// Fetch us by pageable copies / through pinned buffers by the runtime's copies /
// by kernels / as 16-bit offsets: 64 x 64 grid (2.2 MB) 230 / 250 / 97 / 77;
// band of 11,948 (9.9 MB) 2230 / 900 / 310 / 220; 27^3 grid (49 MB) 4170 / 1570
// / 1290 / 1110; 33^3 (127 MB) 9490 / 3300 / 2900 / 2250; 48^3 (874 MB) 22200 /
// 18900 / 17200 / 10000, where the link alone took 15300.  Eight threads instead
// of 12: 2.40 and 11.3 ms; 16: the same.  16 MB buffers: 33^3 6.8 ms.
// Result arrays start on 2 MB boundaries with transparent huge pages requested,
// since their first touch is in this path.
#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

#include <sys/mman.h>

#include "gsofa_internal.h"

namespace gsofa {

namespace {

constexpr uint32_t kBlock = 64;             // indexes that share a base
constexpr size_t kChunkMost = 4u << 20;    // bytes of result in a chunk, and what they take as
                                           // bases, 16-bit offsets and room for whole blocks
constexpr size_t kStageBytes = kChunkMost / (4 * kBlock) * (4 + 6 * kBlock) + (16u << 10);
// Making and releasing the buffers of one large copy takes over 2 ms, so they
// are kept and no copy makes more than it must: with kStageMost out (four large
// copies') a further one has a single thread's two.  So at most
// kStageMost + 1 + 2 * callers exist, all kept while plans live for up to 15
// callers at a time (a server has 16 workers at most); after the last plan's
// release kStageRest, one copy's (153 MB).
constexpr size_t kStageMost = 96;
constexpr size_t kStageKeep = kStageMost + 32;
constexpr size_t kStageRest = 24;
constexpr size_t kKernelMost = 512u << 10; // totals up to here: one kernel
constexpr size_t kPerThread = 2u << 20;     // bytes per copy thread, at least
constexpr int kThreads = 12;
constexpr size_t kChunkMin = 1u << 20;
constexpr size_t kChunks = 4;              // chunks a thread, at least
constexpr size_t kHugePage = 2u << 20;
constexpr size_t kHugeMin = 1u << 20;

std::mutex g_mu;
std::vector<void*> g_stage;                // idle staging buffers
size_t g_out = 0;                          // buffers in use
uint64_t g_made = 0;                       // made so far
struct IdleStream {
    int device;
    hipStream_t s;
};
std::vector<IdleStream> g_streams;
constexpr size_t kStreamKeep = 16;
constexpr size_t kStreamRest = 2;
size_t g_live = 0;                         // streams handed out: live plans
std::vector<Ctrl*> g_ctrl;                 // idle pinned counter blocks, made a page at a time
constexpr size_t kCtrlSlots = 4096 / sizeof(Ctrl);

// A buffer; null if none can be made, or for one that the call can do without
// (`more`) when enough are out.
void* stage_get(bool more) {
    {
        std::lock_guard<std::mutex> lk(g_mu);
        if (more && g_out >= kStageMost) return nullptr;
        g_out++;
        if (!g_stage.empty()) {
            void* p = g_stage.back();
            g_stage.pop_back();
            return p;
        }
        g_made++;
    }
    void* p = nullptr;
    if (hipHostMalloc(&p, kStageBytes, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        std::lock_guard<std::mutex> lk(g_mu);
        g_out--;
        return nullptr;
    }
    return p;
}

void stage_put(void* p) {
    if (!p) return;
    {
        std::lock_guard<std::mutex> lk(g_mu);
        g_out--;
        if (g_stage.size() < kStageKeep) {
            g_stage.push_back(p);
            return;
        }
    }
    (void)hipHostFree(p);
}

struct Pieces {
    static constexpr int MAX = 16;
    uint32_t* dst[MAX];
    const uint32_t* src[MAX];
    uint32_t words[MAX];
    bool index[MAX];  // packed on the way out: dst is the piece's bases
    int count;
};

// An index piece in a staging buffer: a word for every block (its smallest
// value, or WIDE), then the blocks' 16-bit offsets, then their places as they
// are, used by blocks of a wider range only.
constexpr uint32_t WIDE = 0x80000000u;
__host__ __device__ constexpr uint32_t blocks_of(uint32_t words) { return (words + kBlock - 1) / kBlock; }
__host__ __device__ constexpr size_t offsets_at(uint32_t words) { return ((size_t)blocks_of(words) * 4 + 15) & ~(size_t)15; }
__host__ __device__ constexpr size_t wide_at(uint32_t words) {
    return offsets_at(words) + (size_t)blocks_of(words) * kBlock * 2;
}
constexpr size_t index_bytes(uint32_t words) { return wide_at(words) + (size_t)blocks_of(words) * kBlock * 4; }

struct __attribute__((packed, aligned(4))) Quad {
    uint32_t x, y, z, w;
};

// Eight lanes a block, eight values a lane.
__device__ void pack_piece(uint32_t* bases, const uint32_t* src, uint32_t words, uint32_t t, uint32_t step) {
    char* const b = reinterpret_cast<char*>(bases);
    uint4* const offs = reinterpret_cast<uint4*>(b + offsets_at(words));
    uint4* const wide = reinterpret_cast<uint4*>(b + wide_at(words));
    const uint32_t lanes = blocks_of(words) * (kBlock / 8u);
    for (uint32_t i = t; i < lanes; i += step) {  // the lanes of a block stay together
        const uint32_t e = i * 8u;
        uint32_t v[8];
        if (e + 8u <= words) {
            const Quad a = *reinterpret_cast<const Quad*>(src + e), c = *reinterpret_cast<const Quad*>(src + e + 4u);
            v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w;
            v[4] = c.x, v[5] = c.y, v[6] = c.z, v[7] = c.w;
        } else {
#pragma unroll
            for (uint32_t k = 0; k < 8u; k++) v[k] = e + k < words ? src[e + k] : src[words - 1u];
        }
        uint32_t lo = v[0], hi = v[0];
#pragma unroll
        for (uint32_t k = 1; k < 8u; k++) {
            lo = v[k] < lo ? v[k] : lo;
            hi = v[k] > hi ? v[k] : hi;
        }
#pragma unroll
        for (int d = 1; d < 8; d <<= 1) {
            const uint32_t ol = __shfl_xor(lo, d, 8), oh = __shfl_xor(hi, d, 8);
            lo = ol < lo ? ol : lo;
            hi = oh > hi ? oh : hi;
        }
        const bool fits = hi - lo < 65536u;
        if ((i & 7u) == 0u) bases[i >> 3] = fits ? lo : WIDE;
        if (fits) {
            offs[i] = make_uint4((v[0] - lo) | ((v[1] - lo) << 16), (v[2] - lo) | ((v[3] - lo) << 16),
                                 (v[4] - lo) | ((v[5] - lo) << 16), (v[6] - lo) | ((v[7] - lo) << 16));
        } else {
            wide[2u * i] = make_uint4(v[0], v[1], v[2], v[3]);
            wide[2u * i + 1u] = make_uint4(v[4], v[5], v[6], v[7]);
        }
    }
}

void unpack_piece(uint32_t* dst, const char* b, uint32_t words) {
    const uint32_t* bases = reinterpret_cast<const uint32_t*>(b);
    const uint16_t* offs = reinterpret_cast<const uint16_t*>(b + offsets_at(words));
    const uint32_t* wide = reinterpret_cast<const uint32_t*>(b + wide_at(words));
    for (uint32_t k = 0, e = 0; e < words; k++, e += kBlock) {
        const uint32_t lo = bases[k];
        const uint16_t* o = offs + e;
        uint32_t* d = dst + e;
        if (lo == WIDE) std::memcpy(d, wide + e, 4 * std::min(kBlock, words - e));
        else if (words - e >= kBlock)
            for (uint32_t j = 0; j < kBlock; j++) d[j] = lo + o[j];
        else
            for (uint32_t j = 0; j < words - e; j++) d[j] = lo + o[j];
    }
}


// Pieces whose two ends have the same alignment to 16 bytes move in 16-byte
// words but for their ends, the others word by word.
__global__ __launch_bounds__(256) void k_copy_pieces(Pieces p) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x, step = gridDim.x * blockDim.x;
    for (int k = 0; k < p.count; k++) {
        uint32_t* d = p.dst[k];
        const uint32_t* s = p.src[k];
        const uint32_t n = p.words[k];
        if (p.index[k]) {
            pack_piece(d, s, n, t, step);
            continue;
        }
        const uint32_t off = (uint32_t)(reinterpret_cast<uintptr_t>(d) >> 2) & 3u;
        uint32_t head = n, body = 0;
        if (((reinterpret_cast<uintptr_t>(d) ^ reinterpret_cast<uintptr_t>(s)) & 15u) == 0) {
            head = (4u - off) & 3u;
            head = head < n ? head : n;
            body = (n - head) / 4u;
        }
        uint4* d4 = reinterpret_cast<uint4*>(d + head);
        const uint4* s4 = reinterpret_cast<const uint4*>(s + head);
        for (uint32_t i = t; i < body; i += step) d4[i] = s4[i];
        for (uint32_t i = t; i < head; i += step) d[i] = s[i];
        for (uint32_t i = head + 4u * body + t; i < n; i += step) d[i] = s[i];
    }
}

hipError_t launch_pieces(const Pieces& p, size_t bytes, hipStream_t s) {
    const uint32_t blocks = (uint32_t)std::min<size_t>((bytes / 16 + 255) / 256, 512);
    hipLaunchKernelGGL(k_copy_pieces, dim3(std::max(blocks, 1u)), dim3(256), 0, s, p);
    return hipGetLastError();
}

struct Chunk {
    size_t first, count;  // pieces, at most Pieces::MAX
};
struct Piece {
    char* host;
    char* dev;
    size_t bytes;
    size_t off;  // in the chunk's buffer: aligned to 16 bytes, unless packed as dev is
    bool index;  // packed
};

// `out`: device to host, else host to device.
hipError_t copy_small(const std::vector<HostCopy>& v, bool out, char* stage, hipStream_t s, size_t total) {
    Pieces p{};
    size_t off = 0;
    for (const HostCopy& c : v) {
        if (!c.bytes) continue;
        if (!out) std::memcpy(stage + off, c.host, c.bytes);
        p.dst[p.count] = reinterpret_cast<uint32_t*>(out ? stage + off : (char*)c.dev);
        p.src[p.count] = reinterpret_cast<const uint32_t*>(out ? (char*)c.dev : stage + off);
        p.words[p.count++] = (uint32_t)(c.bytes / 4);
        off += (c.bytes + 15) & ~(size_t)15;
    }
    hipError_t e = launch_pieces(p, total, s);
    const hipError_t w = hipStreamSynchronize(s);  // in either case: nothing may still use the buffer
    if (e == hipSuccess) e = w;
    if (e != hipSuccess || !out) return e;
    off = 0;
    for (const HostCopy& c : v) {
        if (c.bytes) std::memcpy(c.host, stage + off, c.bytes);
        off += (c.bytes + 15) & ~(size_t)15;
    }
    return hipSuccess;
}

hipError_t copy_chunks(const std::vector<Piece>& pieces, const std::vector<Chunk>& chunks, bool out,
                       hipStream_t s, std::atomic<size_t>& next, void* b0, void* b1, int device) {
    (void)hipSetDevice(device);
    char* buf[2] = {(char*)b0, (char*)b1};
    hipEvent_t ev[2] = {nullptr, nullptr};
    hipError_t e = hipEventCreateWithFlags(&ev[0], hipEventDisableTiming);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&ev[1], hipEventDisableTiming);
    auto host_side = [&](size_t k, char* b) {
        for (size_t i = chunks[k].first; i < chunks[k].first + chunks[k].count; i++) {
            const Piece& c = pieces[i];
            if (c.index) unpack_piece(reinterpret_cast<uint32_t*>(c.host), b + c.off, (uint32_t)(c.bytes / 4));
            else if (out) std::memcpy(c.host, b + c.off, c.bytes);
            else std::memcpy(b + c.off, c.host, c.bytes);
        }
    };
    auto dma = [&](size_t k, char* b, hipEvent_t x) {
        Pieces p{};
        size_t bytes = 0;
        for (size_t i = chunks[k].first; i < chunks[k].first + chunks[k].count; i++) {
            const Piece& c = pieces[i];
            uint32_t* st = reinterpret_cast<uint32_t*>(b + c.off);
            uint32_t* dv = reinterpret_cast<uint32_t*>(c.dev);
            p.dst[p.count] = out ? st : dv;
            p.src[p.count] = out ? dv : st;
            p.index[p.count] = c.index;
            p.words[p.count++] = (uint32_t)(c.bytes / 4);
            bytes += c.bytes;
        }
        const hipError_t r = launch_pieces(p, bytes, s);
        return r != hipSuccess ? r : hipEventRecord(x, s);
    };
    const size_t none = ~(size_t)0;
    size_t have[2] = {none, none};
    for (int cur = 0; e == hipSuccess; cur ^= 1) {
        size_t k = next.fetch_add(1);
        if (k >= chunks.size()) k = none;
        if (!out && have[cur] != none) {  // the buffer's previous chunk has left it
            e = hipEventSynchronize(ev[cur]);
            have[cur] = none;
        }
        if (e == hipSuccess && k != none) {
            if (!out) host_side(k, buf[cur]);
            e = dma(k, buf[cur], ev[cur]);
            if (e == hipSuccess) have[cur] = k;
        }
        const int o = cur ^ 1;
        if (e == hipSuccess && have[o] != none && (out || k == none)) {
            e = hipEventSynchronize(ev[o]);
            if (e == hipSuccess && out) host_side(have[o], buf[o]);
            have[o] = none;
        }
        if (k == none) break;
    }
    if (e != hipSuccess) (void)hipStreamSynchronize(s);  // no copy left in flight in the buffers
    for (hipEvent_t x : ev)
        if (x) (void)hipEventDestroy(x);
    return e;
}

hipError_t copy_all(const std::vector<HostCopy>& v, bool out, hipStream_t s) {
    size_t total = 0, used = 0;
    for (const HostCopy& c : v) {
        if (c.bytes && (!c.host || !c.dev)) return hipErrorInvalidValue;  // the kernels would fault
        total += c.bytes;
        used += c.bytes != 0;
    }
    if (total == 0) return hipSuccess;
    void* buf[2 * kThreads] = {};
    buf[0] = stage_get(false);
    if (buf[0] && total <= kKernelMost && used <= (size_t)Pieces::MAX) {
        const hipError_t e = copy_small(v, out, (char*)buf[0], s, total);
        stage_put(buf[0]);
        return e;
    }
    int threads = 0;
    const int want = (int)std::min<size_t>(kThreads, std::max<size_t>(1, total / kPerThread));
    for (; threads < want; threads++) {
        void*(&b)[2] = reinterpret_cast<void*(&)[2]>(buf[2 * threads]);
        if (threads > 0) b[0] = stage_get(true);
        if (b[0]) b[1] = stage_get(threads > 0);
        if (b[0] && b[1]) continue;
        stage_put(b[0]);
        b[0] = nullptr;
        break;
    }
    if (threads == 0) {  // no pinned memory: direct copies
        hipError_t e = hipSuccess;
        for (const HostCopy& c : v) {
            if (!c.bytes || e != hipSuccess) continue;
            e = out ? hipMemcpyAsync(c.host, c.dev, c.bytes, hipMemcpyDeviceToHost, s)
                    : hipMemcpyAsync(c.dev, c.host, c.bytes, hipMemcpyHostToDevice, s);
        }
        const hipError_t w = hipStreamSynchronize(s);
        return e == hipSuccess ? w : e;
    }
    const size_t ch = std::min(kChunkMost, std::max(kChunkMin, total / (kChunks * (size_t)threads)));
    std::vector<Piece> pieces;
    std::vector<Chunk> chunks;
    size_t room = 0, at = 0;  // of the last chunk: bytes of result left, bytes of its buffer in use
    for (const HostCopy& c : v)
        for (size_t o = 0; o < c.bytes;) {
            char* dev = (char*)c.dev + o;
            if (room < 4 || chunks.back().count == (size_t)Pieces::MAX) {
                chunks.push_back({pieces.size(), 0});
                room = ch;
                at = 0;
            }
            const bool index = out && c.index;
            const size_t len = std::min(room & ~(size_t)3, c.bytes - o);
            const size_t off = ((at + 15) & ~(size_t)15) + (index ? 0 : (uintptr_t)dev & 15u);
            pieces.push_back({(char*)c.host + o, dev, len, off, index});
            chunks.back().count++;
            at = off + (index ? index_bytes((uint32_t)(len / 4)) : len);
            room -= len;
            o += len;
        }
    int device = 0;
    (void)hipGetDevice(&device);
    std::atomic<size_t> next{0};
    std::vector<hipError_t> err((size_t)threads, hipSuccess);
    std::vector<std::thread> th;
    auto part = [&](int i) {
        err[(size_t)i] = copy_chunks(pieces, chunks, out, s, next, buf[2 * i], buf[2 * i + 1], device);
    };
    for (int i = 1; i < threads; i++) {
        try {
            th.emplace_back(part, i);
        } catch (...) {  // no thread: the others take its chunks
            break;
        }
    }
    part(0);
    for (std::thread& t : th) t.join();
    for (void* b : buf) stage_put(b);
    for (hipError_t x : err)
        if (x != hipSuccess) return x;
    return hipSuccess;
}

}  // namespace

uint64_t stage_made() {
    std::lock_guard<std::mutex> lk(g_mu);
    return g_made;
}

hipError_t copy_out(const std::vector<HostCopy>& v, hipStream_t s) { return copy_all(v, true, s); }
hipError_t copy_in(const std::vector<HostCopy>& v, hipStream_t s) { return copy_all(v, false, s); }

hipError_t launch_copy_words(void* dst, const void* src, uint32_t words, hipStream_t s) {
    Pieces p{};
    p.dst[0] = static_cast<uint32_t*>(dst);
    p.src[0] = static_cast<const uint32_t*>(src);
    p.words[0] = words;
    p.count = 1;
    hipLaunchKernelGGL(k_copy_pieces, dim3(1), dim3(64), 0, s, p);
    return hipGetLastError();
}

void* host_array(size_t bytes) {
    if (bytes < kHugeMin) return malloc(std::max<size_t>(bytes, 1));
    const size_t len = (bytes + kHugePage - 1) / kHugePage * kHugePage;
    void* p = nullptr;
    if (posix_memalign(&p, kHugePage, len) != 0) return nullptr;
    (void)madvise(p, len, MADV_HUGEPAGE);  // advice only: small pages if refused
    return p;
}

// Idle streams are kept (a stream's creation and release take 55 us, a tenth
// of a small matrix's whole call); a returned one has no work left.  With the
// last one's return only what a next single call takes up is left.
hipError_t stream_get(int device, hipStream_t* s) {
    {
        std::lock_guard<std::mutex> lk(g_mu);
        for (size_t i = 0; i < g_streams.size(); i++)
            if (g_streams[i].device == device) {
                *s = g_streams[i].s;
                g_streams.erase(g_streams.begin() + (ptrdiff_t)i);
                g_live++;
                return hipSuccess;
            }
    }
    const hipError_t e = hipStreamCreate(s);
    if (e == hipSuccess) {
        std::lock_guard<std::mutex> lk(g_mu);
        g_live++;
    }
    return e;
}

void stream_put(int device, hipStream_t s) {
    if (!s) return;
    // one with an error is not handed on
    const bool idle = hipStreamSynchronize(s) == hipSuccess;
    if (!idle) (void)hipGetLastError();
    std::vector<hipStream_t> gone;
    std::vector<void*> mem;
    {
        std::lock_guard<std::mutex> lk(g_mu);
        g_live--;
        if (idle) g_streams.insert(g_streams.begin(), {device, s});
        else gone.push_back(s);
        for (; g_streams.size() > (g_live ? kStreamKeep : kStreamRest); g_streams.pop_back())
            gone.push_back(g_streams.back().s);
        for (; g_live == 0 && g_stage.size() > kStageRest; g_stage.pop_back()) mem.push_back(g_stage.back());
    }
    for (hipStream_t x : gone) (void)hipStreamDestroy(x);
    for (void* x : mem) (void)hipHostFree(x);
}

// Idle slabs: the device memory of released plans, the longest idle first.
// Never destroyed: plans may be released while the process ends.
namespace {

constexpr size_t kSlabShare = 16;        // of a device's memory, at most this part is kept idle
constexpr size_t kSlabSpare = 16u << 20;

struct Slabs {
    struct Idle {
        int device;
        void* p;
        size_t bytes;
    };
    std::mutex mu;
    std::vector<Idle> idle;
    uint64_t made = 0;
};
Slabs& slabs() {
    static Slabs* s = new Slabs();
    return *s;
}

size_t idle_bytes(const Slabs& s, int device) {
    size_t sum = 0;
    for (const Slabs::Idle& x : s.idle)
        if (x.device == device) sum += x.bytes;
    return sum;
}

}  // namespace

// Device memory of at least *bytes for the current device, which is `device`;
// *bytes becomes its size: the smallest idle slab of up to twice as much, else a
// new one.  Its contents are any.  Null when there is none.
//
// A plan's memory is mostly its workgroups' arrays (63^3 grid: 8.2 of 9.9 GB), and
// memory that has been in use once is cleared by the driver before it is given
// out again, at 42 GB/s and beside nothing else: a stream of one-shot calls that
// made and released it, 67 GB in 0.27 s of calls, ran at that rate with calls of
// up to 1.7 s among it once it had gone through the card's 288 GB.  32 such calls,
// s a round over seven rounds: 0.26 to 4.5; with slabs kept 0.25 to 0.28 (the first
// round and one other 1.1 and 0.5 where another process had left the card's memory
// in use).
void* slab_get(int device, size_t* bytes) {
    Slabs& s = slabs();
    {
        std::lock_guard<std::mutex> lk(s.mu);
        size_t best = s.idle.size();
        for (size_t i = s.idle.size(); i-- > 0;)  // of equal ones the last released
            if (s.idle[i].device == device && s.idle[i].bytes >= *bytes && s.idle[i].bytes <= 2 * *bytes + kSlabSpare &&
                (best == s.idle.size() || s.idle[i].bytes < s.idle[best].bytes))
                best = i;
        if (best < s.idle.size()) {
            void* p = s.idle[best].p;
            *bytes = s.idle[best].bytes;
            s.idle.erase(s.idle.begin() + (ptrdiff_t)best);
            return p;
        }
        s.made++;
    }
    return device_alloc(*bytes);
}

// p: of slab_get, with no work on it left.  Slabs beyond the bound go, the
// longest idle first.
void slab_put(int device, void* p, size_t bytes) {
    if (!p) return;
    size_t total = 0;
    if (hipDeviceTotalMem(&total, device) != hipSuccess) {
        (void)hipGetLastError();
        total = 0;
    }
    std::vector<void*> gone;
    Slabs& s = slabs();
    {
        std::lock_guard<std::mutex> lk(s.mu);
        s.idle.push_back({device, p, bytes});
        size_t sum = idle_bytes(s, device);
        for (size_t i = 0; i < s.idle.size() && sum > total / kSlabShare;) {
            if (s.idle[i].device != device) {
                i++;
                continue;
            }
            gone.push_back(s.idle[i].p);
            sum -= s.idle[i].bytes;
            s.idle.erase(s.idle.begin() + (ptrdiff_t)i);
        }
    }
    for (void* x : gone) (void)hipFree(x);
}

// Bytes that slabs_release would give back on `device`.
size_t slabs_idle(int device) {
    Slabs& s = slabs();
    std::lock_guard<std::mutex> lk(s.mu);
    return idle_bytes(s, device);
}

bool slabs_release() {
    std::vector<Slabs::Idle> gone;
    Slabs& s = slabs();
    {
        std::lock_guard<std::mutex> lk(s.mu);
        gone.swap(s.idle);
    }
    for (const Slabs::Idle& x : gone) (void)hipFree(x.p);
    return !gone.empty();
}

uint64_t slabs_made() {
    Slabs& s = slabs();
    std::lock_guard<std::mutex> lk(s.mu);
    return s.made;
}

// hipMalloc; what idle slabs hold is given back before it fails.
void* device_alloc(size_t bytes) {
    for (;;) {
        void* p = nullptr;
        if (hipMalloc(&p, bytes) == hipSuccess) return p;
        (void)hipGetLastError();
        if (!slabs_release()) return nullptr;
    }
}

// Idle staging buffers and streams.
void host_idle_release() {
    std::vector<IdleStream> gone;
    std::vector<void*> mem;
    {
        std::lock_guard<std::mutex> lk(g_mu);
        gone.swap(g_streams);
        mem.swap(g_stage);
    }
    for (const IdleStream& x : gone) (void)hipStreamDestroy(x.s);
    for (void* x : mem) (void)hipHostFree(x);
}

Ctrl* ctrl_get() {
    std::lock_guard<std::mutex> lk(g_mu);
    if (g_ctrl.empty()) {
        void* p = nullptr;
        if (hipHostMalloc(&p, sizeof(Ctrl) * kCtrlSlots, hipHostMallocDefault) != hipSuccess) {
            (void)hipGetLastError();
            return nullptr;
        }
        for (size_t i = 0; i < kCtrlSlots; i++) g_ctrl.push_back((Ctrl*)p + i);
    }
    Ctrl* c = g_ctrl.back();
    g_ctrl.pop_back();
    return c;
}

void ctrl_put(Ctrl* c) {
    if (!c) return;
    std::lock_guard<std::mutex> lk(g_mu);
    g_ctrl.push_back(c);
}

}  // namespace gsofa
