// Calls of one rank that wait for the other ranks', first in first out.
//
// Mostly one call waits at a time: the vector keeps its memory and a call is moved in and out of it without an allocation.  A
// rank may also run far ahead.  What has been taken is dropped from the front only when it is at least half of what the vector
// holds, so each call is moved at most once more on average, however many wait; a vector that grew is given back once empty.
#pragma once
#include <cstddef>
#include <utility>
#include <vector>

namespace ops_hccl {

template <class Call>
class CallQueue {
public:
    static constexpr size_t kKeep = 64;   // calls whose memory an empty queue keeps

    size_t size() const { return calls_.size() - head_; }
    bool empty() const { return head_ == calls_.size(); }
    size_t capacity() const { return calls_.capacity(); }

    void Push(Call &&c) { calls_.push_back(std::move(c)); }

    // The call at the head; the queue is not empty.
    Call Take()
    {
        Call c = std::move(calls_[head_++]);
        if (head_ == calls_.size()) {
            if (calls_.capacity() > kKeep) {
                std::vector<Call>().swap(calls_);
            } else {
                calls_.clear();
            }
            head_ = 0;
        } else if (head_ >= kKeep && 2 * head_ >= calls_.size()) {
            calls_.erase(calls_.begin(), calls_.begin() + static_cast<std::ptrdiff_t>(head_));
            head_ = 0;
        }
        return c;
    }

private:
    std::vector<Call> calls_;
    size_t head_ = 0;   // calls_[0 .. head_) have been taken
};

}  // namespace ops_hccl
