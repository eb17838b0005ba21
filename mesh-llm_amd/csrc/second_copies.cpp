#include "second_copies.hpp"

#include "mesh_common.hpp"

namespace mesh {

// an eighth: the rest belongs to the caller's sessions
static bool copies_fit(size_t bytes, size_t held) {
    size_t free_bytes = 0, total = 0;
    if (hipMemGetInfo(&free_bytes, &total) != hipSuccess) { (void)hipGetLastError(); return false; }
    return bytes <= (free_bytes + held) / 8;
}

int SecondCopies::make(const std::vector<Item> &items) {
    size_t bytes = 0;
    for (const Item &i : items) bytes += i.bytes;
    if (!bytes || !copies_fit(bytes, 0)) return MESH_OK;
    for (const Item &i : items) {
        void *p = nullptr;
        const hipError_t e = hipMalloc(&p, i.bytes);
        if (e != hipSuccess) {
            (void)hipGetLastError();                    // (the next launch's check must not meet it)
            release();
            if (e == hipErrorOutOfMemory) return MESH_OK;
            return fail(MESH_ERR_DEVICE, "hipMalloc(%zu) failed: %s", i.bytes, hipGetErrorString(e));
        }
        memory_.push_back(p);
    }
    if (!copies_fit(bytes, bytes)) { release(); return MESH_OK; }
    int rc = MESH_OK;
    for (size_t i = 0; i < items.size() && rc == MESH_OK; ++i) rc = items[i].fill(memory_[i]);
    const hipError_t e = hipDeviceSynchronize();
    if (rc == MESH_OK && e != hipSuccess) rc = fail(MESH_ERR_DEVICE, "second copies of the weights: %s", hipGetErrorString(e));
    if (rc != MESH_OK) { release(); return rc; }
    for (size_t i = 0; i < items.size(); ++i) *items[i].slot = memory_[i];
    return MESH_OK;
}

void SecondCopies::release() {
    for (void *p : memory_) (void)hipFree(p);
    memory_.clear();
}

SecondCopies::~SecondCopies() { release(); }

}  // namespace mesh
