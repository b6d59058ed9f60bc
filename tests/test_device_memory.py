"""The host-side owners of device memory against a small device of their own: the HIP calls they make are replaced by ones
that hand out host memory up to a limit (compiled for the host only; no GPU and no HIP runtime)."""
import subprocess

import pytest

from raytracergpu_mastersproject_amd import build as B

FAKE = r"""
#include <cstdio>
#include <cstdlib>
#include <map>
#include "rt_internal.hpp"
using namespace rtgpu;

static size_t limit = 1u << 30, used = 0;
static int mallocs = 0, live_events = 0;
static std::map<void *, size_t> blocks;
static std::atomic<int> news_left{1 << 30};  // operator new fails when it has run out
void *operator new(size_t n) {
    if (news_left-- <= 0) throw std::bad_alloc();
    return std::malloc(n ? n : 1);
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }
extern "C" {
hipError_t hipMalloc(void **p, size_t n) {
    ++mallocs;
    if (used + n > limit) return hipErrorOutOfMemory;
    *p = std::malloc(1);
    blocks[*p] = n;
    used += n;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    auto it = blocks.find(p);
    if (it == blocks.end()) std::abort();
    used -= it->second;
    blocks.erase(it);
    std::free(p);
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { ++live_events; *e = reinterpret_cast<hipEvent_t>(1); return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { ++live_events; *e = reinterpret_cast<hipEvent_t>(1); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { --live_events; return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { *p = std::malloc(n); return hipSuccess; }
hipError_t hipHostFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) { std::memcpy(d, s, n); return hipSuccess; }
}
#define CHECK(c) do { if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); return 1; } } while (0)
int main() {
    constexpr size_t MB = 1u << 20;
@BODY@
    return 0;
}
"""


def _run(tmp_path, body):
    src = tmp_path / "fake.hip"
    src.write_text(FAKE.replace("@BODY@", body))
    flags = [f for f in B.COMMON if not f.startswith("--offload-arch")]
    subprocess.run([B.HIPCC, "--offload-host-only", *flags, "-c", str(src), "-o", str(tmp_path / "fake.o")], check=True)
    subprocess.run(["g++", str(tmp_path / "fake.o"), "-o", str(tmp_path / "fake"), "-pthread"], check=True)
    r = subprocess.run([str(tmp_path / "fake")], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


MAKES_ROOM = {
    "another scene": "DevBuf b(600 * MB, &pool); CHECK(b.p);",
    "an arena": "DevBuf b; b.alloc_own(600 * MB, pool); CHECK(b.p && b.bytes == 600 * MB);",
    "path storage": "ScratchCache c(pool); { ScratchLease l(c, 600 * MB, nullptr); CHECK(l.ptr()); }",
}


@pytest.mark.parametrize("what", MAKES_ROOM)
def test_kept_memory_makes_room(tmp_path, what):
    """700 MB kept of a released scene, 324 MB left: 600 MB for something else of the same context."""
    _run(tmp_path, """
    {
        DevPool pool;
        { DevBuf a(350 * MB, &pool), b(340 * MB, &pool); }
        CHECK(used > 690 * MB);  // kept
        %s
        try { DevBuf b; b.alloc_own(2000 * MB, pool); CHECK(false); } catch (const Error &e) { CHECK(e.status == RT_ERR_NO_MEMORY); }
    }
    CHECK(used == 0 && live_events == 0);
""" % MAKES_ROOM[what])


def test_scene_size_is_what_it_takes_of_the_device(tmp_path):
    """Pooled blocks are rounded up to 4..7 times a power of two."""
    _run(tmp_path, """
    DevPool pool;
    Scene s;
    s.wide.alloc(33 * MB, &pool);
    s.records.alloc(4097, &pool);
    s.tris.alloc(100 * MB, &pool);
    CHECK(s.device_bytes() == used);
    s.spheres = DevBuf(5 * MB, &pool);  // moved, as the build does
    s.qwide.alloc(9 * MB, &pool);
    CHECK(s.device_bytes() == used);
    s.qwide.release();
    CHECK(s.device_bytes() < used);  // kept, but not the scene's
""")


def test_events_of_a_refused_build_are_destroyed(tmp_path):
    _run(tmp_path, """
    try {
        Event a, b;
        CHECK(live_events == 2);
        throw Error(RT_ERR_INVALID, "triangle 3: materialIndex out of range");
    } catch (const Error &) {
    }
    CHECK(live_events == 0);
""")


def test_staged_copy_goes_on_without_the_threads_it_cannot_start(tmp_path):
    _run(tmp_path, """
    HostStage stage;
    const size_t n = 9 * MB + 5;
    char *from = static_cast<char *>(std::malloc(n)), *to = static_cast<char *>(std::malloc(n));
    for (int k = 0; k < 12; ++k) {  // memory for the first k allocations only
        for (size_t i = 0; i < n; ++i) from[i] = (char)(i * 7 + i / 256 + k);
        std::memset(to, 0, n);
        news_left = k;
        stage.copy(0, to, from, n);
        news_left = 1 << 30;
        CHECK(std::memcmp(from, to, n) == 0);
    }
""")
