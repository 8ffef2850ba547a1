// The log object behind nce_log_handle_t, shared by the host-side translation units.
#pragma once

#include <atomic>
#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <mutex>
#include <string>

struct nce_log_s {
    std::mutex mu;
    std::string text;
    int level = 1;
    std::atomic<uint64_t> lines{0};  // lines ever added (tells a caller whether something it called had anything to say)

    void add(int lvl, const char* fmt, ...) {
        if (lvl > level) return;
        char buf[1024];
        va_list ap;
        va_start(ap, fmt);
        vsnprintf(buf, sizeof(buf), fmt, ap);
        va_end(ap);
        lines.fetch_add(1, std::memory_order_relaxed);
        std::lock_guard<std::mutex> lk(mu);
        if (text.size() > (1u << 20)) text.clear();  // bounded
        text += buf;
        text += '\n';
    }
};
