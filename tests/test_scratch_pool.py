"""The kept scratch of the stateless gradient (csrc/nrc_scratch.hpp) against a stand-in HIP runtime of two
GPUs, which records for every allocation, event and wait the GPU and stream that it belongs to.  A C++
program with the header and the stand-in is built and run on the CPU."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

RUNTIME = r"""
#include "nrc_scratch.hpp"
#include <cstdio>
#include <cstdlib>
#include <map>
#define CHECK(c) do { if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); std::exit(1); } } while (0)

struct ihipStream_t { int device; bool capturing; };
struct ihipEvent_t { int device; hipStream_t on; bool over; };

static int g_device = 0;
static size_t g_free[2] = {1000, 1000};       // bytes that each GPU has left
struct Alloc { int device; size_t bytes; bool ordered; };
static std::map<void *, Alloc> g_live;
static hipError_t g_last = hipSuccess;

static int device_of(hipStream_t s) {
	CHECK(s != hipStreamLegacy);
	return s && s != hipStreamPerThread ? s->device : g_device;
}
static hipError_t ret(hipError_t e) { if (e != hipSuccess) g_last = e; return e; }
static hipError_t alloc(void **p, size_t n, int device, bool ordered) {
	if (n > g_free[device]) return ret(hipErrorOutOfMemory);
	g_free[device] -= n;
	*p = std::malloc(1);
	g_live[*p] = Alloc{device, n, ordered};
	return hipSuccess;
}
static hipError_t release(void *p, int device, bool ordered) {
	CHECK(g_live.count(p) && g_live[p].device == device && g_live[p].ordered == ordered);
	g_free[device] += g_live[p].bytes;
	g_live.erase(p);
	std::free(p);
	return hipSuccess;
}
extern "C" {
hipError_t hipGetDevice(int *d) { *d = g_device; return hipSuccess; }
hipError_t hipStreamGetDevice(hipStream_t s, hipDevice_t *d) {
	CHECK(s != hipStreamLegacy && s != hipStreamPerThread); // HIP's reads through these handles
	*d = device_of(s);
	return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *c) {
	CHECK(s != hipStreamLegacy);
	*c = s && s != hipStreamPerThread && s->capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
	return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode *) { return hipSuccess; }
hipError_t hipGetLastError(void) { hipError_t e = g_last; g_last = hipSuccess; return e; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = new ihipEvent_t{g_device, nullptr, true}; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t e) { return e->over ? hipSuccess : hipErrorNotReady; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
	if (e->device != device_of(s)) return ret(hipErrorInvalidHandle);
	e->on = s;
	e->over = false;
	return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t, unsigned) { (void)device_of(s); return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) { return alloc(p, n, g_device, false); }
hipError_t hipFree(void *p) { return release(p, g_live[p].device, false); }
hipError_t hipMallocAsync(void **p, size_t n, hipStream_t s) {
	CHECK(g_last == hipSuccess); // nothing that the pool tried may be reported by the launches after it
	return alloc(p, n, device_of(s), true);
}
hipError_t hipFreeAsync(void *p, hipStream_t s) { return release(p, device_of(s), true); }
}
static nrc::ScratchPool pool(100);
"""


def run(tmp_path, body):
    src, exe = tmp_path / "scratch.cpp", tmp_path / "scratch"
    src.write_text(RUNTIME + "int main() {\n" + body + "\n}\n")
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-isystem", "/opt/rocm/include",
                    "-I", os.path.join(ROOT, "vknrc_amd", "csrc"), str(src), "-o", str(exe), "-pthread"], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=30)
    assert r.returncode == 0, r.stdout


# a stream gets memory of its own GPU, whichever is current, and no event of another; each GPU's own
# streams share its kept blocks, and a capturing stream takes none
@pytest.mark.parametrize("current", [0, 1])
def test_scratch_is_on_the_streams_gpu(tmp_path, current):
    run(tmp_path, f"""
	g_device = {current};
	ihipStream_t here{{{current}, false}}, there{{{1 - current}, false}}, graph{{{current}, true}};
	nrc::ScratchPool::Lease a, b, c, d;
	CHECK(pool.take(a, 50, &there) == hipSuccess);
	CHECK(g_live.at(a.p).device == {1 - current} && g_live.at(a.p).ordered);
	CHECK(pool.take(b, 50, &here) == hipSuccess);
	CHECK(g_live.at(b.p).device == {current} && !g_live.at(b.p).ordered);
	CHECK(pool.give(a, &there) == hipSuccess && pool.give(b, &here) == hipSuccess);
	void *kept = b.p;
	CHECK(pool.take(c, 50, nullptr) == hipSuccess); // the null stream is the current GPU's; b's use is not over
	CHECK(c.p != kept && !g_live.at(c.p).ordered && g_live.at(c.p).device == {current});
	nrc::ScratchPool::Lease again;
	CHECK(pool.take(again, 50, &here) == hipSuccess && again.p == kept);
	CHECK(pool.take(d, 50, &graph) == hipSuccess && g_live.at(d.p).ordered);
	CHECK(pool.give(c, nullptr) == hipSuccess && pool.give(again, &here) == hipSuccess && pool.give(d, &graph) == hipSuccess);
	CHECK(g_last == hipSuccess && g_live.size() == 2);
	return 0;""")


# the handles of the default streams, which not every runtime call takes
@pytest.mark.parametrize("handle", ["nullptr", "hipStreamLegacy", "hipStreamPerThread"])
def test_scratch_of_the_default_streams(tmp_path, handle):
    run(tmp_path, f"""
	g_device = 1;
	nrc::ScratchPool::Lease a, b, big;
	CHECK(pool.take(a, 50, {handle}) == hipSuccess && pool.give(a, {handle}) == hipSuccess);
	CHECK(pool.take(b, 50, {handle}) == hipSuccess && b.p == a.p && g_live.at(b.p).device == 1);
	CHECK(pool.take(big, 200, {handle}) == hipSuccess && g_live.at(big.p).ordered);
	CHECK(pool.give(b, {handle}) == hipSuccess && pool.give(big, {handle}) == hipSuccess);
	CHECK(g_last == hipSuccess && g_live.size() == 1);
	return 0;""")


# idle blocks go before an allocation of the library or a stream-ordered one is refused, and when they are
# asked for; a block in a call's hands stays, and so does an error that trimming cannot help
def test_scratch_is_given_back(tmp_path):
    run(tmp_path, """
	g_free[0] = 250;
	ihipStream_t s{0, false}, t{0, false};
	nrc::ScratchPool::Lease a, b, big;
	CHECK(pool.take(a, 50, &s) == hipSuccess && pool.take(b, 50, &t) == hipSuccess && g_free[0] == 50);
	CHECK(pool.give(a, &s) == hipSuccess);
	void *p = nullptr, *q = nullptr;
	CHECK(pool.malloc(&p, 120) == hipSuccess && g_free[0] == 30); // a's block went, b's is held
	CHECK(pool.malloc(&q, 120) == hipErrorOutOfMemory);
	CHECK(pool.give(b, &t) == hipSuccess && pool.malloc(&q, 120) == hipSuccess && g_free[0] == 10);
	CHECK(hipFree(p) == hipSuccess && hipFree(q) == hipSuccess && g_live.empty());

	g_last = hipSuccess;
	CHECK(pool.take(a, 50, &s) == hipSuccess && pool.give(a, &s) == hipSuccess && g_free[0] == 150);
	CHECK(pool.take(big, 240, &s) == hipSuccess && g_live.at(big.p).ordered && g_free[0] == 10);
	CHECK(g_last == hipSuccess && pool.give(big, &s) == hipSuccess);
	CHECK(pool.take(a, 50, &s) == hipSuccess && pool.give(a, &s) == hipSuccess);
	pool.trim();
	CHECK(g_live.empty() && g_free[0] == 250);
	return 0;""")


# the library's own allocations all go through the pool, so none is refused while idle scratch is kept
def test_library_allocations_go_through_the_pool():
    src = open(os.path.join(ROOT, "vknrc_amd", "csrc", "nrc_api.cpp")).read()
    assert "g_scratch.malloc(" in src and "hipMalloc(" not in src and "hipExtMalloc" not in src
