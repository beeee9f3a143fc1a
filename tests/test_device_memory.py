"""Device allocation and the slabs (mb_memory.h) against a small fake card,
compiled for the host: an allocation that does not fit beside the idle slabs
frees them and succeeds, a call whose dataset left slabs of other sizes frees
its own unused ones, memory in use stays, what cannot fit fails cleanly, and
no exception leaves them where the host has no memory. The scores of the fits
alive together pin a bounded part of the host's memory."""
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]

FAKE = r"""
#pragma once
#include <cstddef>
#include <cstdlib>
#include <map>
enum hipError_t { hipSuccess, hipErrorOutOfMemory };
// a card of `total` bytes (addresses only), counting what is allocated
struct Card {
    size_t total = 0, used = 0, next = 4096, syncs = 0;
    std::map<void *, size_t> live;
    hipError_t last = hipSuccess;
};
inline Card card;
inline hipError_t hipMalloc(void **p, size_t n) {
    if (card.used + n > card.total) return card.last = hipErrorOutOfMemory;
    *p = (void *)card.next;
    card.next += n;
    card.live[*p] = n;
    card.used += n;
    return hipSuccess;
}
inline hipError_t hipFree(void *p) {
    if (!card.live.count(p)) std::abort();
    card.used -= card.live[p];
    card.live.erase(p);
    return hipSuccess;
}
enum { hipHostMallocDefault };
inline size_t pinned = 0, refuse_pinned = 0;
inline std::map<void *, size_t> pinned_live;
inline hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    if (refuse_pinned) return card.last = hipErrorOutOfMemory;
    pinned += n;
    pinned_live[*p = std::malloc(n)] = n;
    return hipSuccess;
}
inline hipError_t hipHostFree(void *p) {
    if (!pinned_live.count(p)) std::abort();
    pinned -= pinned_live[p];
    pinned_live.erase(p);
    std::free(p);
    return hipSuccess;
}
inline hipError_t hipDeviceSynchronize() { return ++card.syncs, hipSuccess; }
inline hipError_t hipGetLastError() {
    const hipError_t e = card.last;
    card.last = hipSuccess;
    return e;
}
"""

PROGRAM = r"""
#include <cstdio>
#include "mb_memory.h"
using namespace mb;
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); std::exit(1); } } while (0)
constexpr size_t M = 1 << 20;

void *place(Arena &a, size_t bytes) {
    void *p = nullptr;
    return a.place(bytes, &p) == hipSuccess ? p : nullptr;
}

int main() {
    card.total = 1000 * M;
    int a = 0, b = 0;  // two datasets
    {
        Arena run(&a);
        CHECK(place(run, 300 * M) && place(run, 10 * M) && place(run, 10 * M));
    }
    {
        Arena run(&b);
        CHECK(place(run, 200 * M));
    }
    CHECK(card.used == (300 + 32 + 200) * M);  // idle
    void *p = nullptr;
    // beside the idle slabs there is no room: a dataset, a prediction, binning
    CHECK(device_malloc(&p, 900 * M) == hipSuccess && card.used == 900 * M && card.last == hipSuccess);
    CHECK(hipFree(p) == hipSuccess);

    // a call's memory is not idle
    {
        Arena run(&a);
        CHECK(place(run, 600 * M));
        CHECK(device_malloc(&p, 500 * M) != hipSuccess && card.last == hipSuccess);
        CHECK(device_malloc(&p, 390 * M) == hipSuccess);
        CHECK(hipFree(p) == hipSuccess);
        // a slab of the usual size does not fit, the buffer does
        CHECK(device_malloc(&p, 390 * M) == hipSuccess);
        CHECK(place(run, 8 * M) && card.used == 998 * M);
        CHECK(!place(run, 8 * M));
        CHECK(hipFree(p) == hipSuccess);
    }
    CHECK(card.used == 608 * M);

    // the dataset's next call needs one larger buffer than its slabs are
    {
        Arena run(&a);
        void *small = place(run, M);
        CHECK(small && place(run, 700 * M) == nullptr);  // the 600 MB slab holds `small`
        CHECK(place(run, 390 * M));
    }
    card.total = 1400 * M;
    {
        Arena run(&a);
        CHECK(place(run, 1300 * M));  // every slab left is unused, and freed
        CHECK(card.used == 1300 * M);
    }
    slab_pool().drop(&a);
    CHECK(card.used == 0 && card.live.empty());

    // a call on no dataset takes what it places, and leaves nothing
    {
        Arena run(nullptr);
        CHECK(place(run, 1000) && place(run, 1000) && card.used == 2048);
    }
    CHECK(card.used == 0);
    return 0;
}
"""


NO_HOST_MEMORY = r"""
#include <cstdio>
#include <cstdlib>
#include <new>
static bool no_memory = false;
void *operator new(std::size_t n) {
    if (no_memory) throw std::bad_alloc();
    return std::malloc(n ? n : 1);
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, std::size_t) noexcept { std::free(p); }
#include "mb_memory.h"
using namespace mb;
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); std::exit(1); } } while (0)
int main() {
    card.total = (size_t)1 << 30;
    int owner = 0;
    void *p = nullptr;
    {
        Arena run(&owner);
        CHECK(run.place(100, &p) == hipSuccess);
        no_memory = true;  // while the call ends
    }
    CHECK(card.used == 0);
    {
        Arena run(&owner);
        CHECK(run.place(100, &p) == hipErrorOutOfMemory && card.used == 0);
        no_memory = false;
        CHECK(run.place(100, &p) == hipSuccess);
    }
    CHECK(card.used == (size_t)32 << 20);
    no_memory = true;  // while the call begins: the slab stays idle
    {
        Arena run(&owner);
        no_memory = false;
        CHECK(run.place(100, &p) == hipSuccess && card.used == (size_t)64 << 20);
    }
    CHECK(slab_pool().drop(&owner) == (size_t)64 << 20 && card.used == 0);
    return 0;
}
"""


PINNED = r"""
#include <cstdio>
#include <memory>
#include "mb_memory.h"
using namespace mb;
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); std::exit(1); } } while (0)
int main() {
    const size_t count = (size_t)12 << 20;  // 96 MB a fit
    {
        std::vector<std::unique_ptr<HostScores>> fits;
        for (int i = 0; i < 30; ++i) {
            fits.emplace_back(new HostScores());
            fits.back()->reserve(count);
            fits.back()->p[count - 1] = i;
            CHECK(pinned <= (size_t)1 << 30 && fits.back()->n == count);
        }
        CHECK(pinned == 10 * 8 * count);  // the first ten
        fits.erase(fits.begin(), fits.begin() + 3);
        CHECK(pinned == 7 * 8 * count);
        fits.emplace_back(new HostScores());
        fits.back()->reserve(count);
        CHECK(pinned == 8 * 8 * count);  // room again
        fits.back()->reserve(100);
        CHECK(pinned == 7 * 8 * count && fits.back()->n == 100);  // small ones are not pinned
        fits.back()->reserve(0);
        refuse_pinned = 1;
        fits.back()->reserve(count);
        CHECK(pinned == 7 * 8 * count && fits.back()->p && card.last == hipSuccess);
        refuse_pinned = 0;
    }
    CHECK(pinned == 0);
    HostScores a, b;
    a.reserve(((size_t)1 << 30) / 8);  // all of it
    CHECK(pinned == (size_t)1 << 30);
    b.reserve((size_t)1 << 18);
    CHECK(pinned == (size_t)1 << 30);
    return 0;
}
"""


@pytest.fixture(scope="module")
def build(tmp_path_factory):
    at = tmp_path_factory.mktemp("memory")
    (at / "hip").mkdir()
    (at / "hip" / "hip_runtime.h").write_text(FAKE)

    def run(text):
        (at / "p.cpp").write_text(text)
        subprocess.run(["g++", "-g", "-O1", "-std=c++17", f"-I{at}", f"-I{ROOT / 'mojoboost_amd' / 'csrc'}",
                        str(at / "p.cpp"), "-o", str(at / "p"), "-lpthread"], check=True)
        return subprocess.run([str(at / "p")], capture_output=True, text=True)

    return run


def test_allocation_frees_idle_slabs(build):
    out = build(PROGRAM)
    assert out.returncode == 0, out.stdout + out.stderr


def test_no_exception_without_host_memory(build):
    out = build(NO_HOST_MEMORY)
    assert out.returncode == 0, out.stdout + out.stderr


def test_fits_alive_pin_a_bounded_total(build):
    out = build(PINNED)
    assert out.returncode == 0, out.stdout + out.stderr


def test_every_allocation_is_made_there():
    """No file of the library but mb_memory.h calls hipMalloc."""
    for f in sorted((ROOT / "mojoboost_amd" / "csrc").iterdir()):
        if f.suffix in (".hip", ".h", ".cpp") and f.name != "mb_memory.h":
            assert "hipMalloc(" not in f.read_text(), f.name
