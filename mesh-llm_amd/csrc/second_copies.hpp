// Second copies of a stage's weights, in a layout that some calls read faster.  Nothing needs them: where there is no room the
// stage does without, and whatever the process allocates on the GPU through device_alloc takes their room when it finds no other.
#pragma once

#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <functional>
#include <mutex>
#include <shared_mutex>
#include <vector>

namespace mesh {

// hipMalloc on the current device.  Where that finds no room the copies of the stages on this device are given back, one stage
// after the other, until it does.  A failure leaves no error behind for the next launch's check.  Not for a thread that holds
// SecondCopies::in_use().
hipError_t device_alloc(void **p, size_t bytes);

// bytes on `device` that device_alloc would give back
size_t second_copies_bytes(int device);

class SecondCopies {
  public:
    struct Item {
        void **slot;                            // where the address of the copy goes; null while there is none
        size_t bytes;
        std::function<int(void *)> fill;        // writes it (null stream)
    };
    SecondCopies() = default;
    SecondCopies(const SecondCopies &) = delete;
    SecondCopies &operator=(const SecondCopies &) = delete;
    ~SecondCopies();

    // Makes all of the copies on the current device, or none: they may take at most an eighth of the memory that is free without
    // them, which is asked before they are allocated and again after, when other processes may have taken theirs.  No room is no
    // error; one of a fill is.
    int make(const std::vector<Item> &items);

    // Held by a call from before it reads a slot until its last launch is on its stream.
    std::shared_lock<std::shared_mutex> in_use() {
        std::lock_guard<std::mutex> turn(turn_);
        return std::shared_lock<std::shared_mutex>(use_);
    }
    bool present() const { return !memory_.empty(); }       // (under in_use)

  private:
    friend hipError_t device_alloc(void **p, size_t bytes);
    friend size_t second_copies_bytes(int device);
    bool give_back();
    void release();
    std::mutex turn_;               // held while waiting for the calls under way, so that new ones queue up behind
    std::shared_mutex use_;
    std::vector<void *> memory_;
    std::vector<void **> slots_;
    size_t bytes_ = 0;
    int device_ = 0;
};

}  // namespace mesh
