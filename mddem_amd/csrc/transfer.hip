// Particle columns from the device into the caller's arrays.
//
// A download was a pageable copy of each device array in its padded device
// layout (double4, int4, component-major forces) into a temporary vector, then
// a loop that picked the components: three passes over memory that is
// page-faulted twice, on one thread (4,000,000 spheres: 175 ms for 480 MB).
// Here a kernel writes the caller's layout straight into pinned host memory,
// so only the wanted bytes cross the bus, and the host copies each piece once
// to its place. The host copy with the page faults of a fresh array is the
// slower side (a few GB/s on one thread), so large downloads use several
// threads, each on its own pieces. Single-precision forces cross the bus as
// they are and become doubles on their way to the caller's array.
//
// A context's first download, unless it is large, goes without the pinned
// memory, whose allocation and release take 0.3 to 0.7 ms: a job that runs and
// takes its state once would not see them again (the state of 50,000 spheres:
// 0.70 ms without, 1.0 and 0.4 at the end with it; from 8 MiB on, the pinned
// pieces are faster even so, 200,000 spheres 1.8 ms instead of 3.4).
#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <memory>
#include <mutex>
#include <thread>

#include "transfer.hpp"

namespace mdd {

namespace {

// out[w], w < words: word w of particles first .. in the caller's layout
__global__ void k_pack(ColumnKind kind, const void* __restrict__ src, int64_t npad, int64_t first,
                       int64_t words, void* __restrict__ out) {
    const int64_t w = blockIdx.x * int64_t(blockDim.x) + threadIdx.x;
    if (w >= words) return;
    const int64_t p = first + w / 3;
    const int d = int(w % 3);
    switch (kind) {
        case ColumnKind::u32: static_cast<uint32_t*>(out)[w] = static_cast<const uint32_t*>(src)[first + w]; break;
        case ColumnKind::f64: static_cast<double*>(out)[w] = static_cast<const double*>(src)[first + w]; break;
        case ColumnKind::xyz: static_cast<double*>(out)[w] = static_cast<const double*>(src)[4 * p + d]; break;
        case ColumnKind::w: static_cast<double*>(out)[w] = static_cast<const double*>(src)[4 * (first + w) + 3]; break;
        case ColumnKind::xyzw: static_cast<double*>(out)[w] = static_cast<const double*>(src)[4 * first + w]; break;
        case ColumnKind::ixyz: static_cast<int32_t*>(out)[w] = static_cast<const int32_t*>(src)[4 * p + d]; break;
        case ColumnKind::soa32: static_cast<float*>(out)[w] = static_cast<const float*>(src)[d * npad + p]; break;
        case ColumnKind::soa64: static_cast<double*>(out)[w] = static_cast<const double*>(src)[d * npad + p]; break;
    }
}

int words_of(ColumnKind k) {
    switch (k) {
        case ColumnKind::xyz:
        case ColumnKind::ixyz:
        case ColumnKind::soa32:
        case ColumnKind::soa64: return 3;
        case ColumnKind::xyzw: return 4;
        default: return 1;
    }
}
// in pinned memory, and in the caller's array
size_t word_bytes(ColumnKind k) {
    return k == ColumnKind::u32 || k == ColumnKind::ixyz || k == ColumnKind::soa32 ? 4 : 8;
}
size_t row_bytes(ColumnKind k) { return size_t(words_of(k)) * word_bytes(k); }
size_t host_row_bytes(ColumnKind k) { return k == ColumnKind::soa32 ? 24 : row_bytes(k); }

struct Piece {
    const Column* col;
    int64_t first, count;
};

void pack(Ctx& c, const Piece& p, void* out) {
    const int64_t words = p.count * words_of(p.col->kind);
    k_pack<<<blocks_for(words, 256), 256, 0, c.stream>>>(p.col->kind, p.col->dev, c.npad, p.first,
                                                       words, out);
    MDD_HIP(hipGetLastError());
}

void place(const Piece& p, const void* from) {
    const ColumnKind k = p.col->kind;
    char* to = static_cast<char*>(p.col->host) + size_t(p.first) * host_row_bytes(k);
    if (k == ColumnKind::soa32) {
        const float* f = static_cast<const float*>(from);
        double* d = reinterpret_cast<double*>(to);
        for (int64_t w = 0; w < 3 * p.count; w++) d[w] = double(f[w]);
        return;
    }
    std::memcpy(to, from, size_t(p.count) * row_bytes(k));
}

// `raw`: the column's device array as it is
void unpack(const Column& col, const void* raw, int64_t npad, int64_t n) {
    const double* q = static_cast<const double*>(raw);
    const int32_t* q32 = static_cast<const int32_t*>(raw);
    const float* f = static_cast<const float*>(raw);
    double* out = static_cast<double*>(col.host);
    int32_t* out32 = static_cast<int32_t*>(col.host);
    switch (col.kind) {
        case ColumnKind::u32:
        case ColumnKind::f64:
        case ColumnKind::xyzw: std::memcpy(out, raw, size_t(n) * row_bytes(col.kind)); break;
        case ColumnKind::w:
            for (int64_t i = 0; i < n; i++) out[i] = q[4 * i + 3];
            break;
        case ColumnKind::xyz:
            for (int64_t i = 0; i < n; i++)
                for (int d = 0; d < 3; d++) out[3 * i + d] = q[4 * i + d];
            break;
        case ColumnKind::ixyz:
            for (int64_t i = 0; i < n; i++)
                for (int d = 0; d < 3; d++) out32[3 * i + d] = q32[4 * i + d];
            break;
        case ColumnKind::soa32:
            for (int64_t i = 0; i < n; i++)
                for (int d = 0; d < 3; d++) out[3 * i + d] = double(f[d * npad + i]);
            break;
        case ColumnKind::soa64:
            for (int64_t i = 0; i < n; i++)
                for (int d = 0; d < 3; d++) out[3 * i + d] = q[d * npad + i];
            break;
    }
}
size_t raw_bytes(ColumnKind k, int64_t npad, int64_t n) {
    switch (k) {
        case ColumnKind::u32: return 4 * size_t(n);
        case ColumnKind::f64: return 8 * size_t(n);
        case ColumnKind::ixyz: return 16 * size_t(n);
        case ColumnKind::soa32: return 12 * size_t(npad);
        case ColumnKind::soa64: return 24 * size_t(npad);
        default: return 32 * size_t(n);
    }
}

constexpr size_t kSlot = size_t(1) << 19;  // bytes of one piece
constexpr int kMaxCopiers = 8;             // host threads of one download
constexpr size_t kPlain = size_t(8) << 20; // a first download below goes without them

// pinned staging memory of at least `bytes`, kept with the context
char* staging(Ctx& c, size_t bytes) {
    if (c.stage_bytes < bytes) {
        if (c.stage) MDD_HIP(hipHostFree(c.stage));
        c.stage = nullptr;
        c.stage_bytes = 0;
        MDD_HIP(hipHostMalloc(reinterpret_cast<void**>(&c.stage), bytes, hipHostMallocDefault));
        c.stage_bytes = bytes;
    }
    return c.stage;
}

}  // namespace

void release_staging(Ctx& c) {
    for (hipEvent_t e : c.stage_ev) (void)hipEventDestroy(e);
    c.stage_ev.clear();
    if (c.stage) (void)hipHostFree(c.stage);
    c.stage = nullptr;
    c.stage_bytes = 0;
}

void download(Ctx& c, const Column* cols, int ncols, int64_t n) {
    size_t total = 0;
    for (int k = 0; k < ncols; k++) total += row_bytes(cols[k].kind) * size_t(n);
    if (total == 0) return;
    if (!c.downloaded && total < kPlain) {
        size_t most = 0;
        for (int k = 0; k < ncols; k++) most = std::max(most, raw_bytes(cols[k].kind, c.npad, n));
        const std::unique_ptr<char[]> raw(new char[most]);
        for (int k = 0; k < ncols; k++) {
            d2h(c, raw.get(), cols[k].dev, raw_bytes(cols[k].kind, c.npad, n));
            unpack(cols[k], raw.get(), c.npad, n);
        }
        c.downloaded = true;
        return;
    }
    c.downloaded = true;
    // up to 2 MiB (tens of thousands of particles): every column packed, one
    // wait, one thread. Single-precision forces are copied as they are and
    // picked here: at 20,000 atoms a force download takes 26 us, 32 with them
    // packed on the device.
    if (total <= (size_t(2) << 20)) {
        auto plain = [](const Column& col) { return col.kind == ColumnKind::soa32; };
        auto bytes = [&](const Column& col) {
            return plain(col) ? raw_bytes(col.kind, c.npad, n) : row_bytes(col.kind) * size_t(n);
        };
        size_t all = 0, at = 0;
        for (int k = 0; k < ncols; k++) all += bytes(cols[k]);
        char* s = staging(c, all);
        // (8-byte words first, so that every column is aligned)
        std::vector<std::pair<Piece, size_t>> ps;
        for (const size_t wb : {size_t(8), size_t(4)})
            for (int k = 0; k < ncols; k++) {
                if (word_bytes(cols[k].kind) != wb) continue;
                const Piece p{&cols[k], 0, n};
                if (plain(cols[k]))
                    MDD_HIP(hipMemcpyAsync(s + at, cols[k].dev, bytes(cols[k]),
                                           hipMemcpyDeviceToHost, c.stream));
                else
                    pack(c, p, s + at);
                ps.emplace_back(p, at);
                at += bytes(cols[k]);
            }
        MDD_HIP(hipStreamSynchronize(c.stream));
        for (const auto& p : ps) {
            if (plain(*p.first.col))
                unpack(*p.first.col, s + p.second, c.npad, n);
            else
                place(p.first, s + p.second);
        }
        return;
    }
    std::vector<Piece> pieces;
    for (int k = 0; k < ncols; k++) {
        const int64_t per = int64_t(kSlot / row_bytes(cols[k].kind));
        for (int64_t f = 0; f < n; f += per)
            pieces.push_back({&cols[k], f, std::min(per, n - f)});
    }
    const int np = int(pieces.size());
    const int cpus = int(std::thread::hardware_concurrency());
    const int copiers = std::max(1, std::min({kMaxCopiers, np / 2, cpus > 1 ? cpus / 2 : 1}));
    const int slots = std::min(np, 2 * copiers);
    char* s = staging(c, size_t(slots) * kSlot);
    while (int(c.stage_ev.size()) < slots) {
        hipEvent_t e;
        MDD_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
        c.stage_ev.push_back(e);
    }
    // piece q goes through slot q mod slots: packed, then placed, then the
    // slot takes piece q + slots
    auto issue = [&](int q) {
        pack(c, pieces[size_t(q)], s + size_t(q % slots) * kSlot);
        MDD_HIP(hipEventRecord(c.stage_ev[size_t(q % slots)], c.stream));
    };
    std::vector<std::thread> threads;
    threads.reserve(size_t(copiers));
    for (int q = 0; q < slots; q++) issue(q);
    std::mutex mu;  // one thread launches and records at a time
    std::exception_ptr failed;
    std::atomic<bool> stop{false};
    // copier t takes pieces t, t + copiers, ...; a slot belongs to one copier
    // (slots is a multiple of copiers, or every piece has its own slot)
    auto copier = [&](int t) {
        try {
            MDD_HIP(hipSetDevice(c.device));
            for (int q = t; q < np && !stop.load(); q += copiers) {
                MDD_HIP(hipEventSynchronize(c.stage_ev[size_t(q % slots)]));
                place(pieces[size_t(q)], s + size_t(q % slots) * kSlot);
                if (q + slots < np) {
                    std::lock_guard<std::mutex> lk(mu);
                    issue(q + slots);
                }
            }
        } catch (...) {
            std::lock_guard<std::mutex> lk(mu);
            if (!failed) failed = std::current_exception();
            stop.store(true);
        }
    };
    // a copier that gets no thread of its own has its turn on this one
    int own = copiers;
    for (int t = 1; t < own; t++) {
        try {
            threads.emplace_back(copier, t);
        } catch (...) {  // no more threads to be had
            own = t;
        }
    }
    copier(0);
    for (int t = own; t < copiers; t++) copier(t);
    for (auto& th : threads) th.join();
    if (failed) {
        (void)hipStreamSynchronize(c.stream);
        std::rethrow_exception(failed);
    }
}

}  // namespace mdd
