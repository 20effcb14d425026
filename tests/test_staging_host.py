"""The pinned ring of the large host copies (csrc/staging.hip) on the CPU, over a stand-in for the HIP runtime whose
transfers take their time: bytes in both directions, an error half way, and what the copying threads cost
while they wait for the transfers."""
import os
import subprocess

from axion_grav_amd import build

# Transfers are queued and done, in order, when their event (or the stream) is waited for, each taking
# `pace` ms.  Page-locked memory is what hipHostMalloc gave.
PROGRAM = """
#include "axg_internal.h"
#include <string.h>
#include <sys/resource.h>
#include <chrono>
#include <deque>
#include <set>
#include <thread>

struct Op { void* d; const void* s; size_t n; hipEvent_t after; };
static std::deque<Op> g_ops;
static std::set<void*> g_pinned;
static int g_pace = 0, g_fail = -1, g_copies = 0;
static void run_to(hipEvent_t e)
{
    while (!g_ops.empty()) {
        const Op o = g_ops.front();
        g_ops.pop_front();
        if (o.d) {
            std::this_thread::sleep_for(std::chrono::milliseconds(g_pace));
            memcpy(o.d, o.s, o.n);
        } else if (o.after == e) {
            return;
        }
    }
}
extern "C" {
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = malloc(n); g_pinned.insert(*p); return hipSuccess; }
hipError_t hipHostFree(void* p) { g_pinned.erase(p); free(p); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = (hipEvent_t)malloc(1); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { free(e); return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void*) { a->type = hipMemoryTypeUnregistered; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t)
{
    if (g_copies++ == g_fail) return hipErrorUnknown;
    g_ops.push_back({d, s, n, nullptr});
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { g_ops.push_back({nullptr, nullptr, 0, e}); return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) { run_to(e); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { run_to((hipEvent_t)-1); return hipSuccess; }
}

static double cpu()
{
    rusage r;
    getrusage(RUSAGE_SELF, &r);
    return r.ru_utime.tv_sec + r.ru_stime.tv_sec + 1e-6 * (r.ru_utime.tv_usec + r.ru_stime.tv_usec);
}
static double now() { return std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count(); }
#define CHECK(c) do { if (!(c)) { fprintf(stderr, "line %d: %s\\n", __LINE__, #c); return 1; } } while (0)

int main(int argc, char** argv)
{
    const size_t MIB = 1 << 20;
    const bool wait = argc > 1;
    axg::staging_retain(0);
    // chunks of 4 MiB and a remainder, fewer and more than the ring has slots
    for (size_t bytes : {16 * MIB, 17 * MIB + 12345, 61 * MIB + 7, 16 * MIB - 1}) {
        std::vector<char> src(bytes), dst(bytes, 0);
        for (size_t i = 0; i < bytes; i++) src[i] = (char)(i * 2654435761u >> 13);
        axg::copy_to_host(0, nullptr, dst.data(), src.data(), bytes);
        CHECK(dst == src);
        dst.assign(bytes, 0);
        axg::copy_to_device(0, nullptr, dst.data(), src.data(), bytes);
        CHECK(hipStreamSynchronize(nullptr) == hipSuccess && dst == src);
    }
    // a transfer that fails: the call reports it, and the next copy is whole
    for (int at : {0, 3, 11}) {
        for (int out = 0; out < 2; out++) {
            std::vector<char> src(60 * MIB, 5), dst(60 * MIB, 0);
            g_copies = 0;
            g_fail = at;
            bool thrown = false;
            try {
                if (out) axg::copy_to_host(0, nullptr, dst.data(), src.data(), src.size());
                else axg::copy_to_device(0, nullptr, dst.data(), src.data(), src.size());
            } catch (const axg::Error&) {
                thrown = true;
            }
            g_fail = -1;
            CHECK(thrown && g_ops.empty());
            axg::copy_to_host(0, nullptr, dst.data(), src.data(), src.size());
            CHECK(dst == src);
        }
    }
    // the host's share of a slow copy: moving 80 MiB twice, 0.05 s or so of 0.8 s each way
    if (wait) {
        std::vector<char> src(80 * MIB, 3), dst(80 * MIB, 0);
        g_pace = 40;
        for (int out = 0; out < 2; out++) {
            const double c0 = cpu(), t0 = now();
            if (out) axg::copy_to_host(0, nullptr, dst.data(), src.data(), src.size());
            else axg::copy_to_device(0, nullptr, dst.data(), src.data(), src.size());
            const double c = cpu() - c0, t = now() - t0;
            printf("out %d: %.3f s of processors in %.3f s\\n", out, c, t);
            CHECK(t > 0.7 && c < 0.5 * t);
        }
        CHECK(dst == src);
    }
    axg::staging_release(0);
    CHECK(g_pinned.empty());
    return 0;
}
"""


def program(tmp_path):
    (tmp_path / "p.hip").write_text(PROGRAM)
    objs = []
    for src in (str(tmp_path / "p.hip"), os.path.join(build.CSRC, "staging.hip")):
        objs.append(str(tmp_path / (os.path.basename(src) + ".o")))
        subprocess.run([build.HIPCC, *build.FLAGS, "--offload-host-only", "-I", build.CSRC, "-c", src, "-o", objs[-1]], check=True)
    exe = str(tmp_path / "p")
    subprocess.run(["g++", "-pthread", *objs, "-o", exe], check=True)
    return exe


def test_ring_copies_and_waits(tmp_path):
    exe = program(tmp_path)
    r = subprocess.run([exe], timeout=60, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe, "wait"], timeout=60, capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
