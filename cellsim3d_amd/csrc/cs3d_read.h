// cs3d_read.h - how a list of device segments is cut into gather launches and pinned
// slots (host code; the reads of cs3d_api.hip and a host test use it).
#pragma once
#include <stddef.h>
#include <stdint.h>

#include <algorithm>
#include <atomic>
#include <exception>
#include <memory>
#include <vector>

namespace cs3d {

// Pieces of device memory that one launch copies into a buffer (k_gather).
constexpr int kMaxGather = 16;
struct GatherList {
    const uint32_t* src[kMaxGather];
    uint32_t dst[kMaxGather];    // first word in the buffer, a multiple of 4
    uint32_t words[kMaxGather];
    int32_t n;
};

struct ReadSeg {
    const void* dev;
    void* host;
    size_t bytes;  // whole words
};
struct ReadPiece {
    char* host;
    size_t off, bytes;  // offset in the slot
};
struct ReadPlan {
    std::vector<GatherList> lists;               // one for each slot
    std::vector<std::vector<ReadPiece>> pieces;  // what the host copies out of it
    std::unique_ptr<std::atomic<int>[]> done;    // readers that have copied it
    size_t total = 0;
};

// Cuts the segments into slots of slot_bytes, each piece 16-byte aligned in its slot.
// Returns false where the host's memory does not suffice for the plan.
inline bool plan_reads(const ReadSeg* segs, int n_segs, size_t slot_bytes, ReadPlan& plan) noexcept {
    try {
        size_t used = slot_bytes;
        for (int i = 0; i < n_segs; ++i) {
            plan.total += segs[i].bytes;
            for (size_t at = 0; at < segs[i].bytes;) {
                if (used + 16 > slot_bytes || plan.lists.back().n == kMaxGather) {
                    plan.lists.emplace_back();
                    plan.lists.back().n = 0;
                    plan.pieces.emplace_back();
                    used = 0;
                }
                const size_t len = std::min(segs[i].bytes - at, slot_bytes - used);
                GatherList& g = plan.lists.back();
                g.src[g.n] = reinterpret_cast<const uint32_t*>(static_cast<const char*>(segs[i].dev) + at);
                g.dst[g.n] = (uint32_t)(used / 4);
                g.words[g.n++] = (uint32_t)(len / 4);
                plan.pieces.back().push_back(ReadPiece{static_cast<char*>(segs[i].host) + at, used, len});
                used += (len + 15) / 16 * 16;
                at += len;
            }
        }
        plan.done.reset(new std::atomic<int>[plan.lists.size()]);
        for (size_t k = 0; k < plan.lists.size(); ++k) plan.done[k].store(0, std::memory_order_relaxed);
        return true;
    } catch (const std::exception&) {
        return false;
    }
}

}  // namespace cs3d
