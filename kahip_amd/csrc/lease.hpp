// Objects kept per device between calls (the entry points' engines), lent to one call at a time.
#pragma once

#include <exception>
#include <map>
#include <memory>
#include <mutex>
#include <utility>

#include "devbuf.hpp"

namespace kahip {

// The current device's kept T for the life of the lease, created at first use. A call that finds it
// lent to another thread gets a T of its own; a lease that ends by an exception drops the kept T.
// The kept objects are never destroyed at exit (their memory goes with the process).
template <class T>
class Lease {
public:
    Lease() : unwinding_(std::uncaught_exceptions()) {
        int dev = 0;
        KH_CHECK(hipGetDevice(&dev));
        Slot* c;
        {
            std::lock_guard<std::mutex> g(mutex());
            Slot*& slot = slots()[dev];
            if (!slot) slot = new Slot();
            c = slot;
        }
        std::unique_lock<std::mutex> lk(c->mu, std::try_to_lock);
        if (lk.owns_lock()) {
            used_before_ = c->obj != nullptr;
            if (!c->obj) c->obj.reset(new T());
            kept_ = c;
            obj_ = c->obj.get();
            lk_ = std::move(lk);
        } else {
            own_.reset(new T());
            obj_ = own_.get();
        }
    }
    ~Lease() {
        if (kept_ && std::uncaught_exceptions() > unwinding_) {
            kept_->obj.reset();
            dropped() |= used_before_;
        }
    }
    Lease(const Lease&) = delete;
    Lease& operator=(const Lease&) = delete;
    T& operator*() { return *obj_; }
    T* operator->() { return obj_; }

    // Frees the kept objects that are not lent; whether there was one.
    static bool release_idle() {
        bool any = false;
        std::lock_guard<std::mutex> g(mutex());
        for (auto& kv : slots()) {
            std::unique_lock<std::mutex> lk(kv.second->mu, std::try_to_lock);
            if (!lk.owns_lock()) continue;
            any |= kv.second->obj != nullptr;
            kv.second->obj.reset();
        }
        return any;
    }
    // Whether a lease of this thread has dropped an object that earlier calls had used.
    static bool& dropped() {
        thread_local bool d = false;
        return d;
    }

private:
    struct Slot {
        std::mutex mu;
        std::unique_ptr<T> obj;
    };
    static std::mutex& mutex() {
        static auto* m = new std::mutex();
        return *m;
    }
    static std::map<int, Slot*>& slots() {
        static auto* s = new std::map<int, Slot*>();
        return *s;
    }
    int unwinding_;
    bool used_before_ = false;
    Slot* kept_ = nullptr;
    T* obj_ = nullptr;
    std::unique_ptr<T> own_;
    std::unique_lock<std::mutex> lk_;
};

// Runs f. If device memory runs out while kept objects hold some (the buffers of earlier calls, and
// the margins of those that grew), gives that back and runs f once more, so that a call is not
// refused for what the calls before it left behind. f has no effect before its last allocation.
template <class T, class F>
void run_giving_back(F&& f) {
    Lease<T>::dropped() = false;
    try {
        f();
        return;
    } catch (const OutOfMemory&) {
        const bool idle = Lease<T>::release_idle();
        if (!idle && !Lease<T>::dropped()) throw;
    }
    f();
}

}  // namespace kahip
