// pin_pool.hpp -- blocks of pinned host memory that a call borrows for as long
// as it runs.  Any thread may take and give; a given block serves the next
// taker, whichever object it belongs to, so an object's first call makes one
// only while every other block is out.  At most `keep` blocks lie free.
//
// Alloc: static uint8_t* make() (nullptr when it fails), static void drop(uint8_t*).
#pragma once
#include <cstddef>
#include <cstdint>
#include <mutex>
#include <vector>

namespace memvanta {
namespace hip {

template <typename Alloc>
class PinPool {
public:
    explicit PinPool(std::size_t keep) { free_.reserve(keep_ = keep); }
    uint8_t* take() {
        {
            std::lock_guard<std::mutex> lock(mu_);
            if (!free_.empty()) {
                uint8_t* const p = free_.back();
                free_.pop_back();
                return p;
            }
        }
        return Alloc::make();
    }
    // whether the block was kept (nothing may still use it then); the caller
    // keeps it otherwise
    bool give(uint8_t* p) {
        std::lock_guard<std::mutex> lock(mu_);
        if (free_.size() >= keep_) return false;
        free_.push_back(p);
        return true;
    }
    // free blocks beyond n go back to the system
    void trim(std::size_t n) {
        std::vector<uint8_t*> drop;
        {
            std::lock_guard<std::mutex> lock(mu_);
            for (; free_.size() > n; free_.pop_back()) drop.push_back(free_.back());
        }
        for (uint8_t* p : drop) Alloc::drop(p);
    }

private:
    std::mutex mu_;
    std::vector<uint8_t*> free_;
    std::size_t keep_;
};

}  // namespace hip
}  // namespace memvanta
