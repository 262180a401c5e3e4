// transfer.h -- the model state between host arrays ([i][k], k fastest) and
// device planes ([k][i], padded pitch).
#pragma once

#include <vector>

#include "vvm_internal.h"

namespace vvmd {

// A list of arrays, moved in one go: a kernel transposes them between the
// device planes and pieces of pinned, mapped host memory, and the host copies
// those from or to the caller's arrays meanwhile.  The pinned memory (at most
// kSlots of kSlotBytes) stays with the link for the next transfer.
class HostLink {
   public:
    ~HostLink() { release(); }
    void release();
    void clear() { items.clear(); }
    void field(const double *host, double *dev) { items.push_back({host, dev, nullptr, 0}); }
    // an AB2 history: host [i][k][2], two planes
    void pair(const double *host, double *dev0, double *dev1) { items.push_back({host, dev0, dev1, 0}); }
    void line(const double *host, double *dev, int n) { items.push_back({host, dev, nullptr, n}); }
    // VVM_OK once the move is complete (host arrays written, or device planes).
    int upload(const Grid &G, int device, hipStream_t st) { return move(true, G, device, st); }
    int download(const Grid &G, int device, hipStream_t st) { return move(false, G, device, st); }

   private:
    struct Item {
        const double *host;
        double *dev, *dev2;
        int n;  // > 0: a line of n doubles
    };
    std::vector<Item> items;
    static constexpr int kThreads = 4, kSlots = 2 * kThreads;
    static constexpr size_t kSlotBytes = size_t(1) << 20;
    double *slot[kSlots] = {}, *slot_dev[kSlots] = {};
    hipEvent_t ev[kSlots] = {};
    size_t slot_doubles = 0;
    int nslots = 0;
    int reserve(int n, size_t doubles);
    bool host_arrays_overlap(const Grid &G) const;
    int move(bool up, const Grid &G, int device, hipStream_t st);
};

}  // namespace vvmd
