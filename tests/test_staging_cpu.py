"""Small host transfers (staging.cpp) against a runtime whose asynchronous copies
read and write the host's memory only when the stream is synchronised: the
caller's memory is its own again when ctx_put returns, with page-locked memory
and without, and ctx_fetch fills every destination."""
import os
import subprocess

import pytest

from conftest import PKG, ROOT

HIP = "/opt/rocm/include"

_DRIVER = r"""
#include <cstdlib>
#include <cstring>
#include <functional>
#include <vector>
#include "bem_internal.h"
static std::vector<std::function<void()>> queue;
static bool pinned = true;
extern "C" {
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    queue.push_back([=] { std::memcpy(d, s, n); });
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
    for (auto& f : queue) f();
    queue.clear();
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    *p = pinned ? std::malloc(n) : nullptr;
    return pinned ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return ""; }
}
int bem_fail(bem_ctx*, int code, const std::string&) { return code; }
int main(int argc, char** argv) {
    pinned = std::atoi(argv[1]);
    const size_t bytes = std::strtoull(argv[2], nullptr, 10);
    bem_ctx c;
    std::vector<char> src(bytes), want, back;
    std::vector<std::vector<char>> dev(5, std::vector<char>(bytes));
    for (int k = 0; k < 5; k++) {  // the source is used again after every call
        for (size_t i = 0; i < bytes; i++) src[i] = (char)(31 * i + 7 * k + 1);
        want.insert(want.end(), src.begin(), src.end());
        if (ctx_put(&c, dev[k].data(), src.data(), bytes)) return 2;
        std::memset(src.data(), 0, bytes);
    }
    back.resize(want.size());
    char* b = back.data();
    if (ctx_fetch(&c, {{b, dev[0].data(), bytes}, {b + bytes, dev[1].data(), bytes}, {b + 2 * bytes, dev[2].data(), bytes},
                       {b + 3 * bytes, dev[3].data(), bytes}, {b + 4 * bytes, dev[4].data(), bytes}}))
        return 3;
    return back == want ? 0 : 1;
}
"""


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    if not os.path.isdir(HIP):
        pytest.skip("no HIP headers")
    d = tmp_path_factory.mktemp("staging")
    (d / "driver.cpp").write_text(_DRIVER)
    csrc = os.path.join(PKG, "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-I" + HIP, "-I" + csrc,
                    "-I" + os.path.join(ROOT, "include"), "-o", str(d / "driver"), str(d / "driver.cpp"),
                    os.path.join(csrc, "staging.cpp")], check=True)
    return str(d / "driver")


@pytest.mark.parametrize("nbytes", [1, 64, 4097, 300000, 1 << 19, (1 << 19) + 8, 3 << 20])
@pytest.mark.parametrize("pinned", [1, 0])
def test_small_transfers(driver, pinned, nbytes):
    assert subprocess.run([driver, str(pinned), str(nbytes)]).returncode == 0
