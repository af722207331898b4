// Which of a table's device words a call uses to find its longest row, so that no two calls that can be under
// way at once use the same ones.  Host code, free of HIP (table_slot() of common.hpp asks the stream).
#pragma once

#include <map>
#include <mutex>
#include <utility>

namespace dnatok {

class StreamSlots {
public:
    static constexpr int kStreams = 64, kCaptures = 64, kSlots = kStreams + kCaptures;

    // A call made on `stream`: calls on one stream are ordered, so they share a slot.  A call that is being captured
    // (capture != 0: the id of its capture) runs on whatever streams the graph is replayed on, beside any other
    // call, so it shares a slot only with the calls it is ordered with in its own graph: those of the same stream in
    // the same capture.  -1: no slot is left.
    int of(void *stream, unsigned long long capture)
    {
        std::lock_guard<std::mutex> hold(lock_);
        const auto key = std::make_pair(stream, capture);
        const auto it = slot_of_.find(key);
        if (it != slot_of_.end()) return it->second;
        int &used = capture ? captures_ : streams_;
        if (used == (capture ? kCaptures : kStreams)) return -1;
        const int slot = (capture ? kStreams : 0) + used;
        slot_of_.emplace(key, slot);
        ++used;
        return slot;
    }

private:
    std::mutex lock_;
    std::map<std::pair<void *, unsigned long long>, int> slot_of_;
    int streams_ = 0, captures_ = 0;
};

}  // namespace dnatok
