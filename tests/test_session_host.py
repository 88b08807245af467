"""The session's host side with the device played by deferred calls: a launch runs when the stream is waited for."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qwen3.ink.cpp_amd", "csrc")

DEVICE = r"""
#include <cstdlib>
#include <functional>
#include "decoder_session.h"
static std::vector<std::function<void()>> waiting;
static void run_all() { for (auto& f : waiting) f(); waiting.clear(); }
extern "C" {
hipError_t hipMalloc(void** p, size_t n) { *p = malloc(n); return hipSuccess; }
hipError_t hipFree(void* p) { run_all(); free(p); return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = malloc(n); return hipSuccess; }
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipMemset(void* p, int v, size_t n) { memset(p, v, n); return hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { run_all(); memcpy(d, s, n); return hipSuccess; }
hipError_t hipStreamCreate(hipStream_t* s) { *s = nullptr; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { run_all(); return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorUnknown; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t*) { return hipErrorUnknown; }
hipError_t hipGraphInstantiate(hipGraphExec_t*, hipGraph_t, hipGraphNode_t*, char*, size_t) { return hipErrorUnknown; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorUnknown; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = nullptr; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 0; return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
}
namespace a81w41 {
hipError_t launch_take_tokens(const int* h, int n, int* d, const int* hw, int nw, int* dw, hipStream_t) {
    waiting.push_back([=] { std::copy_n(h, n, d); std::copy_n(hw, nw, dw); });
    return hipSuccess;
}
hipError_t launch_give_floats(const float* x, float* h, size_t n, hipStream_t) {
    waiting.push_back([=] { std::copy_n(x, n, h); });
    return hipSuccess;
}
hipError_t launch_zero_words(void* p, size_t words, hipStream_t) {
    waiting.push_back([=] { memset(p, 0, 4 * words); });
    return hipSuccess;
}
hipError_t launch_argmax_token(const float*, int, int*, int*, int, int*, hipStream_t) { return hipSuccess; }
}  // namespace a81w41

// A pass appends its ids to `seen`; the first one fails after half its launches when asked to.
struct Model : a81w41::DecoderSession {
    std::vector<int> seen;
    bool fails = false;
    int start(int max_rows) { return init_session(64, 8, max_rows); }
    int ready() const override { return 0; }
    int enqueue_pass(int m, const int*, int, hipStream_t) override {
        waiting.push_back([=] { seen.insert(seen.end(), ids, ids + m); });
        return fails ? a81w41::failf(A81W41_ERR_HIP, "a launch failed") : 0;
    }
    size_t weight_bytes() const override { return 0; }
};
int main() {
    const int first[4] = {11, 12, 13, 14}, second[4] = {21, 22, 23, 24}, want[1] = {3};
    float logits[8];
    int out[2];
    for (bool generates : {false, true}) {  // a pass that fails on its way, then another one
        Model m;
        if (m.start(4)) return 2;
        auto call = [&](const int* ids) { return generates ? m.generate_greedy(ids, 4, 1, out, nullptr, nullptr) : m.forward(ids, 4, want, 1, logits); };
        m.fails = true;
        if (!call(first)) return 3;
        m.fails = false;
        if (m.reset() || call(second)) return 4;
        if (m.seen != std::vector<int>{11, 12, 13, 14, 21, 22, 23, 24}) return 5;  // what was handed in, each pass its own
    }
    Model m;  // portions
    if (m.start(2) || m.generate_greedy(first, 4, 1, out, nullptr, nullptr) || m.forward(second, 4, want, 1, logits)) return 6;
    return m.seen == std::vector<int>{11, 12, 13, 14, 21, 22, 23, 24} ? 0 : 7;
}
"""


@pytest.mark.skipif(not shutil.which("g++"), reason="no host compiler")
def test_ids_of_a_pass_are_not_overwritten_while_they_wait(tmp_path):
    source, exe = tmp_path / "device.cpp", tmp_path / "device"
    source.write_text("#include <algorithm>\n#include <cstring>\n" + DEVICE)
    built = subprocess.run(["g++", "-std=c++17", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I", CSRC, str(source),
                            os.path.join(CSRC, "decoder_session.cpp"), os.path.join(CSRC, "status.cpp"), "-o", str(exe)],
                           capture_output=True, text=True)
    assert built.returncode == 0, built.stderr[-2000:]
    assert subprocess.run([str(exe)], timeout=60).returncode == 0
