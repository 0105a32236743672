// The caching device allocator.
#include "ddj_internal.h"

#include <algorithm>

namespace ddj {

// Size classes: powers of two up to 1 MiB, then multiples of 2 MiB.  Every
// block also has 64 spare bytes so kernels may touch whole 16-byte vectors
// past a logical end.
size_t Allocator::round_size(size_t bytes) {
    bytes += 64;
    if (bytes <= (1u << 20)) {
        size_t s = 256;
        while (s < bytes) s <<= 1;
        return s;
    }
    const size_t g = 2u << 20;
    return (bytes + g - 1) / g * g;
}

void* Allocator::take_locked(size_t s) {
    void* p = nullptr;
    auto it = free_.find(s);
    if (it != free_.end() && !it->second.empty()) {
        p = it->second.back();
        it->second.pop_back();
    } else if (hipMalloc(&p, s) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    live_[p] = s;
    in_use_ += s;
    return p;
}

void* Allocator::alloc(size_t bytes) {
    const size_t s = round_size(bytes);
    {
        std::lock_guard<std::mutex> lk(mu_);
        void* p = take_locked(s);
        if (!p) {  // give the cached blocks back and retry
            trim_locked();
            p = take_locked(s);
        }
        if (p) return p;
    }
    if (group_) {
        // the blocks that the others keep, with everyone stopped, so that none of
        // them caches more meanwhile (nobody waits for the group holding a lock)
        std::lock_guard<std::mutex> gl(group_->mu);
        std::vector<std::unique_lock<std::mutex>> locks;
        for (Allocator* m : group_->members) locks.emplace_back(m->mu_);
        for (Allocator* m : group_->members) m->trim_locked();
        if (void* p = take_locked(s)) return p;
    }
    fail(DDJ_ENOMEM, "device allocation of " + std::to_string(s) + " bytes failed");
}

void Allocator::share(Allocator& other) {
    if (!other.group_) {
        other.group_ = std::make_shared<Group>();
        other.group_->members.push_back(&other);
    }
    std::lock_guard<std::mutex> gl(other.group_->mu);
    other.group_->members.push_back(this);
    group_ = other.group_;
}

void Allocator::free(void* p) {
    if (!p) return;
    std::lock_guard<std::mutex> lk(mu_);
    auto it = live_.find(p);
    if (it == live_.end()) return;
    free_[it->second].push_back(p);
    in_use_ -= it->second;
    live_.erase(it);
}

bool Allocator::detach(void* p, size_t* cls) {
    std::lock_guard<std::mutex> lk(mu_);
    auto it = live_.find(p);
    if (it == live_.end()) return false;
    if (cls) *cls = it->second;
    in_use_ -= it->second;
    live_.erase(it);
    return true;
}

void Allocator::adopt(void* p, size_t cls) {
    std::lock_guard<std::mutex> lk(mu_);
    live_[p] = cls;
    in_use_ += cls;
}

void Allocator::trim() {
    std::lock_guard<std::mutex> lk(mu_);
    trim_locked();
}

void Allocator::trim_locked() {
    (void)hipDeviceSynchronize();
    for (auto& kv : free_)
        for (void* p : kv.second) (void)hipFree(p);
    free_.clear();
}

Allocator::~Allocator() {
    if (group_) {
        std::lock_guard<std::mutex> gl(group_->mu);
        auto& m = group_->members;
        m.erase(std::find(m.begin(), m.end(), this));
    }
    trim_locked();
    for (auto& kv : live_) (void)hipFree(kv.first);
}

}  // namespace ddj
