// Buffers that a library keeps per (device, stream) for calls made of several launches.  Launches on one stream run in the order in
// which they were queued, so the calls of a stream can share a buffer as long as no call's launches stand between another's: two
// host threads may use one stream, so a call holds its buffer's lock until its last launch is queued.
#pragma once
#include <cstddef>
#include <mutex>

template <int COUNT>
class KeptBuffers {
public:
    // queue(ptr) with the buffer of (dev, stream), made by make(bytes) on the first call and never given back: a captured graph may
    // hold its address.  Returns false, and queues nothing, where there is none: `need` beyond its size, the COUNT buffers taken, or
    // make() returned null (the next call tries again).
    template <class Make, class Queue>
    bool with(int dev, const void* stream, size_t need, size_t bytes, Make make, Queue queue) {
        Buffer* b = find(dev, stream, need, bytes, make);
        if (!b) return false;
        std::lock_guard<std::mutex> lock(b->queueing);
        queue(b->ptr);
        return true;
    }

private:
    struct Buffer {
        int dev;
        const void* stream;
        void* ptr;
        size_t bytes;
        std::mutex queueing;
    };
    template <class Make>
    Buffer* find(int dev, const void* stream, size_t need, size_t bytes, Make make) {
        std::lock_guard<std::mutex> lock(list_);
        for (int i = 0; i < n_; ++i)
            if (buf_[i].dev == dev && buf_[i].stream == stream) return need <= buf_[i].bytes ? &buf_[i] : nullptr;
        if (n_ == COUNT || need > bytes) return nullptr;
        void* ptr = make(bytes);
        if (!ptr) return nullptr;
        Buffer& b = buf_[n_++];
        b.dev = dev;
        b.stream = stream;
        b.ptr = ptr;
        b.bytes = bytes;
        return &b;
    }
    std::mutex list_;
    Buffer buf_[COUNT];
    int n_ = 0;
};
