// Device memory of closed flow handles, kept for the next flow: the policy,
// apart from the runtime's calls (Api: alloc(bytes), null if refused; release(p)).
//
// A program that follows a data set replaces its flow over and over (the next
// handle made, then the old one closed), and freeing and allocating the
// 2 x 44 MB of a 96-frame field cost 330 us of a 550 us set-up.  So a closed
// flow's arrays wait here for the next one, while the device has another flow:
// the last handle to close gives everything back.  What is held also goes back
// where an allocation fails, and when the program asks for it.  Other allocators
// cannot have it otherwise, so it is little: at most kMostBytes a device, a
// thousandth of its memory, which two 96-frame fields fill; a larger flow's
// memory is freed as it closes.
// One instance per device; callers lock.
#pragma once

#include <cstddef>
#include <initializer_list>
#include <vector>

namespace nbx {

template <class Api>
class FlowBlocks {
   public:
    struct Block {
        void* p;
        size_t bytes;
    };
    static constexpr size_t kMostBytes = size_t(256) << 20;

    // a gridded flow more
    void open() { ++flows_; }

    // a held block of at least `bytes` and at most an eighth more, or a new one
    Block take(size_t bytes) {
        for (size_t i = 0; i < held_.size(); ++i) {
            const Block b = held_[i];
            if (b.bytes < bytes || b.bytes > bytes + bytes / 8) continue;
            held_.erase(held_.begin() + static_cast<std::ptrdiff_t>(i));
            bytes_ -= b.bytes;
            return b;
        }
        void* p = Api::alloc(bytes);
        if (p == nullptr && give_back()) p = Api::alloc(bytes);
        return Block{p, bytes};
    }

    // the arrays of a closing flow (null entries allowed); idle: nothing on the
    // device uses them any more
    void close(std::initializer_list<Block> blocks, bool idle) {
        --flows_;
        for (const Block& b : blocks) {
            if (b.p == nullptr) continue;
            if (idle && flows_ > 0 && bytes_ + b.bytes <= kMostBytes) {
                held_.push_back(b);
                bytes_ += b.bytes;
            } else {
                Api::release(b.p);
            }
        }
        if (flows_ <= 0) give_back();
    }

    // whether anything was held
    bool give_back() {
        const bool any = !held_.empty();
        for (const Block& b : held_) Api::release(b.p);
        held_.clear();
        bytes_ = 0;
        return any;
    }

   private:
    std::vector<Block> held_;
    size_t bytes_ = 0;
    int flows_ = 0;  // live gridded flows
};

}  // namespace nbx
