// k_transfer.hip -- host arrays <-> device planes (transfer.h).
#include <algorithm>
#include <atomic>
#include <cstring>
#include <thread>
#include <utility>

#include "transfer.h"

namespace vvmd {

namespace {

// A piece of a chunk: columns i0 .. i0+ni-1 of one field (or pair), or a line.
struct Piece {
    double *d0, *d1;
    int i0, ni;  // ni < 0: a line of -ni doubles
    int off;     // its place in the slot, in doubles
};
constexpr int kPieces = 40;
struct Chunk {
    int n = 0;
    int first[kPieces + 1] = {};  // first workgroup of each piece
    Piece p[kPieces];
};

// Columns a workgroup moves (half as many of a pair, whose columns are twice
// as long): their values pass through LDS, so that the host side is read or
// written as one contiguous run (PCIe wants whole lines) and the device side in
// runs of 128 bytes.
constexpr int kCols = 16, kBlock = 256;
__host__ __device__ inline int piece_cols(const Piece &p) { return p.d1 ? kCols / 2 : kCols; }

template <bool UP>
__global__ void __launch_bounds__(kBlock) k_move(Grid G, Chunk C, double *__restrict__ slot) {
    extern __shared__ double lds[];
    int q = 0;
    while (q + 1 < C.n && int(blockIdx.x) >= C.first[q + 1]) q++;
    const Piece P = C.p[q];
    double *h = slot + P.off;
    if (P.ni < 0) {
        for (int t = threadIdx.x; t < -P.ni; t += kBlock) {
            if (UP) P.d0[t] = h[t];
            else h[t] = P.d0[t];
        }
        return;
    }
    const int np = P.d1 ? 2 : 1, per = G.nz * np, ld = per | 1;  // odd LDS stride: no bank conflicts across columns
    const int c0 = (int(blockIdx.x) - C.first[q]) * piece_cols(P), nc = min(piece_cols(P), P.ni - c0);
    const int tot = nc * per;
    h += size_t(c0) * per;
    auto dev_side = [&](auto &&op) {  // (device address, LDS index), columns fastest
        for (int t = threadIdx.x; t < tot; t += kBlock) {
            const int r = t / nc, c = t - r * nc;  // r = row, or (plane, row) of a pair
            const bool second = r >= G.nz;
            const int k = second ? r - G.nz : r;
            double *d = (second ? P.d1 : P.d0) + ix(G, P.i0 + c0 + c, k);
            op(d, c * ld + k * np + (second ? 1 : 0));
        }
    };
    auto host_side = [&](auto &&op) {
        for (int t = threadIdx.x; t < tot; t += kBlock) {
            const int c = t / per;
            op(h + t, c * ld + t - c * per);
        }
    };
    if (UP) {
        host_side([&](const double *a, int l) { lds[l] = *a; });
        __syncthreads();
        dev_side([&](double *d, int l) { *d = lds[l]; });
    } else {
        dev_side([&](const double *d, int l) { lds[l] = *d; });
        __syncthreads();
        host_side([&](double *a, int l) { *a = lds[l]; });
    }
}

}  // namespace

void HostLink::release() {
    for (int s = 0; s < kSlots; s++) {
        if (slot[s]) (void)hipHostFree(slot[s]);
        if (ev[s]) (void)hipEventDestroy(ev[s]);
        slot[s] = slot_dev[s] = nullptr;
        ev[s] = nullptr;
    }
    slot_doubles = 0;
    nslots = 0;
}

int HostLink::reserve(int n, size_t doubles) {
    if (n <= nslots && doubles <= slot_doubles) return VVM_OK;
    n = std::max(n, nslots);
    doubles = std::max(doubles, slot_doubles);
    release();
    for (int s = 0; s < n; s++) {
        if (hipHostMalloc(reinterpret_cast<void **>(&slot[s]), doubles * sizeof(double),
                          hipHostMallocMapped | hipHostMallocCoherent) != hipSuccess) {
            slot[s] = nullptr;
            release();
            return VVM_ERR_NOMEM;
        }
        if (hipHostGetDevicePointer(reinterpret_cast<void **>(&slot_dev[s]), slot[s], 0) != hipSuccess ||
            hipEventCreateWithFlags(&ev[s], hipEventDisableTiming) != hipSuccess) {
            release();
            return VVM_ERR_HIP;
        }
    }
    nslots = n;
    slot_doubles = doubles;
    return VVM_OK;
}

bool HostLink::host_arrays_overlap(const Grid &G) const {
    std::vector<std::pair<const double *, const double *>> r;
    for (const Item &it : items)
        r.emplace_back(it.host, it.host + (it.n > 0 ? size_t(it.n) : size_t(G.nx) * G.nz * (it.dev2 ? 2 : 1)));
    std::sort(r.begin(), r.end());
    for (size_t q = 1; q < r.size(); q++)
        if (r[q].first < r[q - 1].second) return true;
    return false;
}

// Chunks of at most a slot; small states go as one, by this thread alone.
// Otherwise up to kThreads threads each keep two slots going: while the GPU
// moves one, the thread copies the other (one thread copies at 10 to 18 GB/s,
// PCIe moves 50).  Every launch goes to the caller's stream.
int HostLink::move(bool up, const Grid &G, int device, hipStream_t st) {
    size_t total = 0;
    const size_t col = size_t(G.nz);
    for (const Item &it : items) total += it.n > 0 ? size_t(it.n) : col * G.nx * (it.dev2 ? 2 : 1);
    if (total == 0) return VVM_OK;
    const size_t cap = std::min(total, kSlotBytes / sizeof(double));
    std::vector<Chunk> chunks(1);
    std::vector<std::vector<double *>> host(1);  // the caller's side of each piece
    size_t used = 0;
    auto put = [&](double *h, const Piece &p0, size_t doubles) {
        if (chunks.back().n == kPieces) {
            chunks.emplace_back();
            host.emplace_back();
            used = 0;
        }
        Chunk &c = chunks.back();
        Piece p = p0;
        p.off = int(used);
        const int blocks = p.ni < 0 ? 1 : (p.ni + piece_cols(p) - 1) / piece_cols(p);
        c.first[c.n + 1] = c.first[c.n] + blocks;
        c.p[c.n++] = p;
        host.back().push_back(h);
        used += doubles;
    };
    auto room = [&](size_t least) {  // doubles left in the last chunk, a new one if fewer than least
        if (cap - used < least && used > 0) {
            chunks.emplace_back();
            host.emplace_back();
            used = 0;
        }
        return cap - used;
    };
    for (const Item &it : items) {
        double *h = const_cast<double *>(it.host);
        if (it.n > 0) {
            for (int t = 0; t < it.n;) {
                const int n = int(std::min<size_t>(room(1), size_t(it.n - t)));
                put(h + t, {it.dev + t, nullptr, 0, -n, 0}, n);
                t += n;
            }
            continue;
        }
        const size_t per = col * (it.dev2 ? 2 : 1);  // at most 960 doubles a column: far less than a slot
        for (int i = 0; i < G.nx;) {
            const int n = int(std::min<size_t>(room(per) / per, size_t(G.nx - i)));
            put(h + size_t(i) * per, {it.dev, it.dev2, i, n, 0}, per * n);
            i += n;
        }
    }
    // arrays of a download that share memory: one thread, whose copies follow the
    // list, so that the array listed last is the one that stays
    const bool shared = !up && host_arrays_overlap(G);
    const int nc = int(chunks.size()), nt = shared ? 1 : std::min(kThreads, (nc + 1) / 2), per_thread = std::min(2, nc);
    if (const int rc = reserve(nt * per_thread, cap)) return rc;
    const size_t lds = size_t(kCols) * (G.nz + 1) * sizeof(double);
    auto copy = [&](int c, double *s) {
        for (int q = 0; q < chunks[c].n; q++) {
            const Piece &p = chunks[c].p[q];
            const size_t n = p.ni < 0 ? size_t(-p.ni) : col * (p.d1 ? 2 : 1) * p.ni;
            if (up) std::memcpy(s + p.off, host[c][q], n * sizeof(double));
            else std::memcpy(host[c][q], s + p.off, n * sizeof(double));
        }
    };
    auto launch = [&](int c, int s) {
        const dim3 g(chunks[c].first[chunks[c].n]);
        if (up) hipLaunchKernelGGL(k_move<true>, g, dim3(kBlock), lds, st, G, chunks[c], slot_dev[s]);
        else hipLaunchKernelGGL(k_move<false>, g, dim3(kBlock), lds, st, G, chunks[c], slot_dev[s]);
        return hipGetLastError() == hipSuccess && hipEventRecord(ev[s], st) == hipSuccess;
    };
    std::atomic<bool> ok{true};
    std::atomic<int> next{0};
    auto worker = [&](int t) {
        if (hipSetDevice(device) != hipSuccess) ok = false;
        int in_slot[2] = {-1, -1};  // the chunk each of this thread's slots holds
        const int s0 = t * per_thread;
        int turn = 0;
        auto settle = [&](int b) {  // the slot's chunk is through the GPU
            if (in_slot[b] < 0) return;
            if (hipEventSynchronize(ev[s0 + b]) != hipSuccess) ok = false;
            if (!up && ok) copy(in_slot[b], slot[s0 + b]);
            in_slot[b] = -1;
        };
        for (int c = next++; c < nc && ok; c = next++, turn ^= (per_thread - 1)) {
            settle(turn);
            if (up) copy(c, slot[s0 + turn]);
            if (!launch(c, s0 + turn)) ok = false;
            in_slot[turn] = c;
        }
        for (int b = 0; b < per_thread; b++) settle(turn ^ (b * (per_thread - 1)));
    };
    std::vector<std::thread> pool;
    try {
        for (int t = 1; t < nt; t++) pool.emplace_back(worker, t);
    } catch (...) {
        // no more threads to be had: those there are take all chunks
    }
    worker(0);
    for (std::thread &t : pool) t.join();
    return ok ? VVM_OK : VVM_ERR_HIP;
}

}  // namespace vvmd
