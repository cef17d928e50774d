"""read_through_ring (qwen-native-engine_amd/csrc/host_read.hpp), which brings a batch's logits to pageable
host memory, and poll_device, the wait with a deadline that it and every stream wait use (CPU). Both are
compiled with g++ into a small driver whose device is host memory: a transfer lands some polls after it is
sent, never, or with an error."""
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
CSRC = ROOT / "qwen-native-engine_amd" / "csrc"

DRIVER = r"""
#include <cstdio>
#include <cstdlib>
#include "host_read.hpp"
// driver bytes slot_bytes slots threads fails_at(-1: never) stuck_at(-1: never) timeout
struct Device {
    std::vector<uint8_t>& mem;
    std::vector<uint8_t>& ring;
    size_t slot_bytes;
    long fails_at, stuck_at, sent = 0;
    std::vector<size_t> offset, len, polls;
    std::vector<long> piece;
    void send(size_t slot, size_t off, size_t n) {
        if (sent >= (long)piece.size() && polls[slot] != 0) std::abort();  // sent again before it landed
        if (n > slot_bytes || off + n > mem.size()) std::abort();
        offset[slot] = off, len[slot] = n, polls[slot] = 3 + off % 5, piece[slot] = sent++;
        std::fill_n(ring.begin() + slot * slot_bytes, slot_bytes, 0xEE);
    }
    bool landed(size_t slot) {
        if (piece[slot] == fails_at) throw qne::Error(QNE_EFORMAT, "transfer error");
        if (piece[slot] == stuck_at || (polls[slot] && --polls[slot])) return false;
        std::memcpy(ring.data() + slot * slot_bytes, mem.data() + offset[slot], len[slot]);
        return true;
    }
};
int main(int, char** v) {
    const size_t bytes = atol(v[1]), slot = atol(v[2]), slots = atol(v[3]);
    std::vector<uint8_t> mem(bytes), ring(slot * slots), out(bytes + 1, 0x55);
    for (size_t i = 0; i < bytes; i++) mem[i] = (uint8_t)(i * 2654435761u >> 13);
    Device d{mem, ring, slot, atol(v[5]), atol(v[6])};
    d.offset.resize(slots), d.len.resize(slots), d.polls.resize(slots), d.piece.resize(slots);
    try {
        qne::read_through_ring(d, bytes, out.data(), ring.data(), slot, slots, atoi(v[4]), atof(v[7]));
    } catch (const qne::Error& e) {
        std::printf("error %d", (int)e.code);
        return 0;
    }
    std::printf("%s", std::equal(mem.begin(), mem.end(), out.begin()) && out[bytes] == 0x55 ? "same" : "differ");
}
"""


@pytest.fixture(scope="module")
def read(tmp_path_factory):
    d = tmp_path_factory.mktemp("read")
    (d / "main.cpp").write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", f"-I{CSRC}", str(d / "main.cpp"), "-o", str(d / "read")], check=True)

    def f(nbytes, slot, slots, threads, fails_at=-1, stuck_at=-1, timeout=30.0):
        cmd = [str(d / "read"), *map(str, (nbytes, slot, slots, threads, fails_at, stuck_at, timeout))]
        return subprocess.run(cmd, capture_output=True, text=True, check=True, timeout=60).stdout

    return f


@pytest.mark.parametrize("threads", [0, 1, 4, 16])
@pytest.mark.parametrize("nbytes", [1, 4096, 4097, 8 * 4096, 8 * 4096 + 1, 37 * 4096 - 5])
def test_every_byte_arrives(read, nbytes, threads):
    assert read(nbytes, 4096, 8, threads) == "same"
    assert read(nbytes, 4096, 1, threads) == "same"


@pytest.mark.parametrize("threads", [0, 4])
@pytest.mark.parametrize("at", [0, 7, 20])
def test_a_device_error_ends_the_threads_and_is_thrown(read, threads, at):
    assert read(21 * 4096, 4096, 8, threads, fails_at=at) == "error -5"


@pytest.mark.parametrize("threads", [0, 4])
@pytest.mark.parametrize("at", [0, 20])
def test_a_transfer_that_never_lands_is_a_device_error(read, threads, at):
    assert read(21 * 4096, 4096, 8, threads, stuck_at=at, timeout=0.2) == "error -4"
