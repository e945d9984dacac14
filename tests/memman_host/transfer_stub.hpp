#pragma once
#include <stddef.h>

#include <atomic>
#include <functional>

extern std::atomic<bool> g_frame;       // a frame is queued on the stream
extern std::atomic<size_t> g_copied;    // bytes copied by hipMemcpyAsync
extern std::atomic<size_t> g_pinned;    // pinned bytes allocated
extern std::function<void()> g_on_wait; // runs where the frame is waited for
