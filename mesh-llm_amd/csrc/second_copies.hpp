// Second copies of a stage's weights, in a layout that some calls read faster.  Nothing needs them: where there is no room the
// stage does without.
#pragma once

#include <cstddef>
#include <functional>
#include <vector>

namespace mesh {

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

  private:
    void release();
    std::vector<void *> memory_;
};

}  // namespace mesh
