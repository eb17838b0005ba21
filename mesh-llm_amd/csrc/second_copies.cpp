#include "second_copies.hpp"

#include <algorithm>

#include "mesh_common.hpp"

namespace mesh {

namespace {
// the stages that hold copies (never destroyed: stages may outlive the library's static objects)
struct Holders {
    std::mutex mu;
    std::vector<SecondCopies *> all;
};
Holders &holders() {
    static Holders *h = new Holders();
    return *h;
}
// an eighth: the rest belongs to the caller's sessions
bool copies_fit(size_t bytes, size_t held) {
    size_t free_bytes = 0, total = 0;
    if (hipMemGetInfo(&free_bytes, &total) != hipSuccess) { (void)hipGetLastError(); return false; }
    return bytes <= (free_bytes + held) / 8;
}
}  // namespace

hipError_t device_alloc(void **p, size_t bytes) {
    hipError_t e = hipMalloc(p, bytes);
    if (e == hipSuccess) return e;
    (void)hipGetLastError();
    int device = 0;
    if (e != hipErrorOutOfMemory || hipGetDevice(&device) != hipSuccess) return e;
    Holders &h = holders();
    std::lock_guard<std::mutex> lk(h.mu);
    for (;;) {
        e = hipMalloc(p, bytes);            // (first of all: another thread may have given back what it takes)
        if (e == hipSuccess) return e;
        (void)hipGetLastError();
        auto it = std::find_if(h.all.rbegin(), h.all.rend(), [&](const SecondCopies *c) { return c->device_ == device; });
        if (e != hipErrorOutOfMemory || it == h.all.rend() || !(*it)->give_back()) return e;
        h.all.erase(std::next(it).base());
    }
}

size_t second_copies_bytes(int device) {
    Holders &h = holders();
    std::lock_guard<std::mutex> lk(h.mu);
    size_t n = 0;
    for (const SecondCopies *c : h.all)
        if (c->device_ == device) n += c->bytes_;
    return n;
}

int SecondCopies::make(const std::vector<Item> &items) {
    size_t bytes = 0;
    for (const Item &i : items) bytes += i.bytes;
    if (!bytes || !copies_fit(bytes, 0)) return MESH_OK;
    MESH_HIP_TRY(hipGetDevice(&device_));
    for (const Item &i : items) {
        void *p = nullptr;
        const hipError_t e = hipMalloc(&p, i.bytes);    // (not device_alloc: copies do not take the room of copies)
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
    for (size_t i = 0; i < items.size(); ++i) {
        *items[i].slot = memory_[i];
        slots_.push_back(items[i].slot);
    }
    bytes_ = bytes;
    Holders &h = holders();
    std::lock_guard<std::mutex> lk(h.mu);
    h.all.push_back(this);
    return MESH_OK;
}

// Waits for the calls that may have read a slot, then for their launches; the device is current.
bool SecondCopies::give_back() {
    std::lock_guard<std::mutex> turn(turn_);
    std::unique_lock<std::shared_mutex> use(use_);
    if (hipDeviceSynchronize() != hipSuccess) { (void)hipGetLastError(); return false; }
    for (void **s : slots_) *s = nullptr;
    release();
    return true;
}

void SecondCopies::release() {
    for (void *p : memory_) (void)hipFree(p);
    memory_.clear();
    slots_.clear();
    bytes_ = 0;
}

SecondCopies::~SecondCopies() {
    Holders &h = holders();
    std::lock_guard<std::mutex> lk(h.mu);
    h.all.erase(std::remove(h.all.begin(), h.all.end(), this), h.all.end());
    release();
}

}  // namespace mesh
