// Device memory to pageable host memory through a ring of pinned slots.
#pragma once

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstdint>
#include <cstring>
#include <memory>
#include <string>
#include <thread>
#include <vector>

#include "error.hpp"

namespace qne {

// Polls `ready` until it is true, spinning at first, and like the reference's device poll
// (kernels/src/lib.rs:399-405) ends in an error after timeout_s instead of blocking forever.
template <class Ready>
void poll_device(Ready ready, double timeout_s) {
    using clk = std::chrono::steady_clock;
    const auto start = clk::now();
    int spins = 0;
    while (!ready()) {
        if (++spins > 2000) std::this_thread::sleep_for(std::chrono::microseconds(50));
        if (std::chrono::duration<double>(clk::now() - start).count() > timeout_s)
            throw Error(QNE_EDEVICE, "GPU wait failed: timed out after " + std::to_string((long long)timeout_s) + " s");
    }
}

// `bytes` to dst in pieces of slot_bytes. dev.send(slot, offset, len) starts the transfer of a piece into
// a slot of `ring`, dev.landed(slot) says whether the last one sent there has arrived. The calling thread
// alone talks to the device; up to `threads` others, which live for this call, copy the pieces out. A
// device error, or timeout_s gone by, stops them and is thrown once they have ended. Without any (threads
// 0, or the system grants none) the calling thread copies too.
template <class Device>
void read_through_ring(Device& dev, size_t bytes, uint8_t* dst, const uint8_t* ring, size_t slot_bytes, size_t slots,
                       int threads, double timeout_s) {
    using clk = std::chrono::steady_clock;
    const auto start = clk::now();
    const size_t pieces = (bytes + slot_bytes - 1) / slot_bytes, n = std::min(slots, pieces);
    std::unique_ptr<std::atomic<size_t>[]> emptied(new std::atomic<size_t>[n]);  // 1 + the last piece copied out of a slot
    for (size_t i = 0; i < n; i++) emptied[i] = 0;
    std::atomic<size_t> next{0}, arrived{0};  // the next piece to copy; pieces that are in their slots
    std::atomic<bool> stop{false};
    auto len = [&](size_t i) { return std::min(slot_bytes, bytes - i * slot_bytes); };
    auto copy = [&](size_t i) {
        std::memcpy(dst + i * slot_bytes, ring + (i % n) * slot_bytes, len(i));
        emptied[i % n] = i + 1;
    };
    auto work = [&] {
        for (size_t i; (i = next.fetch_add(1)) < pieces;) {
            while (arrived <= i && !stop) std::this_thread::yield();
            if (stop) return;
            copy(i);
        }
    };
    size_t sent = 0;
    auto send = [&] {
        dev.send(sent % n, sent * slot_bytes, len(sent));
        sent++;
    };
    std::vector<std::thread> others;
    auto join = [&] {
        for (std::thread& t : others) t.join();
    };
    others.reserve(std::max(0, threads));
    try {
        while (sent < n) send();
        try {
            for (size_t t = 0; t < std::min((size_t)std::max(0, threads), n); t++) others.emplace_back(work);
        } catch (...) {  // no thread for it
        }
        while (arrived < pieces) {
            poll_device([&] {
                bool moved = sent < pieces && emptied[sent % n] == sent - n + 1;
                if (moved) send();
                if (arrived < sent && dev.landed(arrived % n)) {
                    arrived++;
                    moved = true;
                    if (others.empty()) copy(next++);
                }
                return moved;
            }, timeout_s - std::chrono::duration<double>(clk::now() - start).count());
        }
    } catch (...) {
        stop = true;
        join();
        throw;
    }
    work();  // what is left
    join();
}

}  // namespace qne
