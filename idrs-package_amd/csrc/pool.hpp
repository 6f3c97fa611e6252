// A bounded pool of idle buffers: plain host code over an allocate/free pair,
// so that its rules can be run without a GPU.  The device pools are in
// pool.hip.
#pragma once

#include <cstddef>
#include <list>
#include <map>
#include <mutex>
#include <vector>

namespace idrs {

// Buffers given back are kept for requests of the same size.  At most 'cap'
// bytes are kept: past that the buffers longest idle are freed, so a program
// that moves on to other sizes keeps those, and a request that the device
// cannot serve frees every idle buffer and is tried once more.  Any thread may
// call any member.
class BufferPool {
public:
    struct Memory {
        void *(*alloc)(size_t bytes);   // null: out of memory
        void (*free)(void *p);
    };
    BufferPool(Memory m, size_t cap) : mem(m), cap_(cap) {}
    BufferPool(const BufferPool &) = delete;
    BufferPool &operator=(const BufferPool &) = delete;

    // a buffer of exactly 'bytes', an idle one (the longest idle of that size)
    // or a new one; null: out of memory
    void *take(size_t bytes) {
        {
            std::lock_guard<std::mutex> g(mu);
            auto it = by_size.find(bytes);
            if (it != by_size.end()) {
                std::list<Idle>::iterator e = it->second.front();
                it->second.pop_front();
                if (it->second.empty()) by_size.erase(it);
                void *p = e->p;
                kept_ -= bytes;
                idle.erase(e);
                return p;
            }
        }
        return allocate(bytes);
    }
    void give(void *p, size_t bytes) {
        std::vector<void *> drop;
        if (bytes > cap_) {
            drop.push_back(p);
        } else {
            std::lock_guard<std::mutex> g(mu);
            evict(cap_ - bytes, drop);
            idle.push_back({p, bytes});
            by_size[bytes].push_back(std::prev(idle.end()));
            kept_ += bytes;
        }
        for (void *q : drop) mem.free(q);
    }
    // memory that is not kept for reuse: the idle buffers make room when the
    // device has none left
    void *allocate(size_t bytes) {
        void *p = mem.alloc(bytes);
        if (!p && trim() > 0) p = mem.alloc(bytes);
        return p;
    }
    // frees every idle buffer; the bytes freed
    size_t trim() {
        std::vector<void *> drop;
        size_t freed;
        {
            std::lock_guard<std::mutex> g(mu);
            freed = kept_;
            evict(0, drop);
        }
        for (void *q : drop) mem.free(q);
        return freed;
    }

private:
    struct Idle {
        void *p;
        size_t bytes;
    };
    // takes the buffers longest idle off the list until at most 'most' bytes remain
    void evict(size_t most, std::vector<void *> &drop) {
        while (kept_ > most) {
            const Idle e = idle.front();
            auto it = by_size.find(e.bytes);
            it->second.pop_front();
            if (it->second.empty()) by_size.erase(it);
            idle.pop_front();
            kept_ -= e.bytes;
            drop.push_back(e.p);
        }
    }
    const Memory mem;
    const size_t cap_;
    std::mutex mu;
    std::list<Idle> idle;   // longest idle first
    std::map<size_t, std::list<std::list<Idle>::iterator>> by_size;   // in the same order
    size_t kept_ = 0;
};

}  // namespace idrs
