// Host values that depend on a key alone (matrices of an order), made once and
// shared between handles and threads.
#pragma once

#include <cstddef>
#include <cstdint>
#include <map>
#include <memory>
#include <mutex>

namespace sphstk {

// Vectors by key, at most `bound` bytes of them: beyond that the least recently
// used ones are given back (whoever holds one keeps it).  A value is made outside
// the lock, so that threads making different ones do not wait for each other; a
// second thread that wants the one being made waits for it.  What make() throws
// passes through, and the next caller makes the value anew.
template <typename Key, typename Vec>
class Pool {
    struct Slot {
        std::once_flag once;
        std::shared_ptr<const Vec> v;
        size_t bytes = 0;
        uint64_t used = 0;
    };
    std::mutex mu_;
    std::map<Key, std::shared_ptr<Slot>> slots_;
    const size_t bound_;
    size_t total_ = 0;
    uint64_t clock_ = 0;

    void trim(const Slot *keep) {
        while (total_ > bound_) {
            auto oldest = slots_.end();
            for (auto it = slots_.begin(); it != slots_.end(); ++it)
                if (it->second->v && it->second.get() != keep &&
                    (oldest == slots_.end() || it->second->used < oldest->second->used))
                    oldest = it;
            if (oldest == slots_.end()) return;
            total_ -= oldest->second->bytes;
            slots_.erase(oldest);
        }
    }

  public:
    explicit Pool(size_t bound) : bound_(bound) {}
    template <typename F>
    std::shared_ptr<const Vec> get(const Key &key, F make) {
        std::shared_ptr<Slot> s;
        {
            std::lock_guard<std::mutex> lock(mu_);
            auto &e = slots_[key];
            if (!e) e = std::make_shared<Slot>();
            s = e;
            s->used = ++clock_;
        }
        std::call_once(s->once, [&] {
            auto v = std::make_shared<const Vec>(make());
            std::lock_guard<std::mutex> lock(mu_);
            s->bytes = v->size() * sizeof(typename Vec::value_type);
            s->v = std::move(v);
            total_ += s->bytes;
            trim(s.get());
        });
        return s->v;
    }
    size_t bytes() {
        std::lock_guard<std::mutex> lock(mu_);
        return total_;
    }
};

// The same without a bound, for the tables themselves: references stay valid.
template <typename Key, typename T>
class Tables {
    struct Slot {
        std::once_flag once;
        std::unique_ptr<T> v;
    };
    std::mutex mu_;
    std::map<Key, Slot> slots_;

  public:
    template <typename F>
    const T &get(const Key &key, F make) {
        Slot *s;
        {
            std::lock_guard<std::mutex> lock(mu_);
            s = &slots_[key];
        }
        std::call_once(s->once, [&] { s->v = make(); });
        return *s->v;
    }
};

} // namespace sphstk
