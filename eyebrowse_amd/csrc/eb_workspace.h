// A device's grow-only workspace: which buffer it is, when it grows, and which outgrown buffers
// graphs still use. The memory calls are a template argument (Mem), so that the rules are tested
// on the host:
//   eb_status alloc(size_t floats, float **p)   EB_OUT_OF_MEMORY, with nothing changed, without room
//   eb_status drain()                            waits for the stream that uses the buffer
//   eb_status free(float *p)
#pragma once

#include <algorithm>
#include <cstddef>
#include <unordered_map>
#include <vector>

#include "eyebrowse_hip.h"

namespace eb {

// After memory was refused, this many calls that would like as much do without before one asks
// again: a refusal costs an allocation call, and its reason may pass at any time.
constexpr int kRefusedCalls = 63;

class Workspace {
  public:
    float *ptr() const { return ptr_; }
    size_t floats() const { return floats_; }

    // Grows to hold want floats, or at least least (<= want) where there is no memory for want.
    // A buffer that holds least is given up only once a larger one is there.
    template <class Mem>
    eb_status grow(Mem &mem, size_t want, size_t least) {
        if (want <= floats_) return EB_OK;
        if (least < want && !(refused_ > 0 && want >= refused_ && left_ > 0)) {
            float *p = nullptr;
            const eb_status st = mem.alloc(want, &p);
            if (st == EB_OK) {
                const eb_status dropped = drop(mem);
                if (dropped != EB_OK) {
                    (void)mem.free(p);
                    return dropped;
                }
                if (want >= refused_) refused_ = 0;
                ptr_ = p;
                floats_ = want;
                return EB_OK;
            }
            if (st != EB_OUT_OF_MEMORY) return st;
            refused_ = want;
            left_ = kRefusedCalls;
        } else if (least < want) {
            --left_;
        }
        if (least <= floats_) return EB_OK;
        // No room for both: the old buffer goes first.
        const eb_status st = drop(mem);
        if (st != EB_OK) return st;
        float *p = nullptr;
        const eb_status got = mem.alloc(least, &p);
        if (got != EB_OK) return got;
        ptr_ = p;
        floats_ = least;
        return EB_OK;
    }

    // A graph whose kernels have the current buffer in their arguments keeps it.
    float *ref() {
        if (ptr_) ++refs_[ptr_];
        return ptr_;
    }
    // Drops such a reference (the caller has drained the stream, so no replay still runs). A buffer
    // the workspace has outgrown is freed with its last graph.
    template <class Mem>
    void unref(Mem &mem, float *p) {
        const auto it = refs_.find(p);
        if (it == refs_.end() || --it->second > 0) return;
        refs_.erase(it);
        const auto r = std::find(retired_.begin(), retired_.end(), p);
        if (r == retired_.end()) return;
        retired_.erase(r);
        (void)mem.free(p);
    }

    // At the device's end, its stream drained.
    template <class Mem>
    void free_all(Mem &mem) {
        if (ptr_) (void)mem.free(ptr_);
        for (float *p : retired_) (void)mem.free(p);
        ptr_ = nullptr;
        floats_ = 0;
        retired_.clear();
    }

  private:
    // Stream ordered: the buffer is freed only after the stream drains, and not at all while a
    // graph has it (it is then retired).
    template <class Mem>
    eb_status drop(Mem &mem) {
        if (!ptr_) return EB_OK;
        if (refs_.count(ptr_)) {
            retired_.push_back(ptr_);
        } else {
            eb_status st = mem.drain();
            if (st == EB_OK) st = mem.free(ptr_);
            if (st != EB_OK) return st;
        }
        ptr_ = nullptr;
        floats_ = 0;
        return EB_OK;
    }

    float *ptr_ = nullptr;
    size_t floats_ = 0;
    std::unordered_map<float *, int> refs_;  // live graph references per buffer
    std::vector<float *> retired_;           // outgrown buffers that a graph still references
    size_t refused_ = 0;                     // the size that memory was last refused for
    int left_ = 0;                           // calls that do without before one asks again
};

}  // namespace eb
