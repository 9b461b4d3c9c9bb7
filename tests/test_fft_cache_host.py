"""A plan's rocFFT cache is made once, also when several threads meet at its
first stage call (plans whose operators run the fused passes have none until
then).  Host only: pf_fft.cpp compiled against stand-ins of the rocFFT entry
points, with an allocator slow enough that every thread is past an unguarded
check before the first cache exists."""

import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pyfourier_amd", "csrc")

PROGRAM = r"""
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <new>
#include <thread>
#include <vector>
#include "pf_fft.cpp"

static std::atomic<int> caches{0}, plans{0};
void* operator new(std::size_t n, const std::nothrow_t&) noexcept {
    if (n == sizeof(pf_fft_cache)) {
        ++caches;
        std::this_thread::sleep_for(std::chrono::milliseconds(200));
    }
    return std::malloc(n);
}
int pf_fail(int code, const std::string&) { return code; }
extern "C" {
rocfft_status rocfft_setup() { return rocfft_status_success; }
rocfft_status rocfft_plan_description_create(rocfft_plan_description*) { return rocfft_status_success; }
rocfft_status rocfft_plan_description_destroy(rocfft_plan_description) { return rocfft_status_success; }
rocfft_status rocfft_plan_description_set_data_layout(rocfft_plan_description, rocfft_array_type, rocfft_array_type,
                                                      const size_t*, const size_t*, size_t, const size_t*, size_t, size_t,
                                                      const size_t*, size_t) { return rocfft_status_success; }
rocfft_status rocfft_plan_create(rocfft_plan*, rocfft_result_placement, rocfft_transform_type, rocfft_precision, size_t,
                                 const size_t*, size_t, const rocfft_plan_description) {
    ++plans;
    return rocfft_status_success;
}
rocfft_status rocfft_plan_destroy(rocfft_plan) { return rocfft_status_success; }
rocfft_status rocfft_plan_get_work_buffer_size(const rocfft_plan, size_t* n) { *n = 0; return rocfft_status_success; }
rocfft_status rocfft_execution_info_create(rocfft_execution_info*) { return rocfft_status_success; }
rocfft_status rocfft_execution_info_destroy(const rocfft_execution_info) { return rocfft_status_success; }
rocfft_status rocfft_execution_info_set_work_buffer(rocfft_execution_info, void*, size_t) { return rocfft_status_success; }
rocfft_status rocfft_execution_info_set_stream(rocfft_execution_info, void*) { return rocfft_status_success; }
rocfft_status rocfft_execute(const rocfft_plan, void**, void**, rocfft_execution_info) { return rocfft_status_success; }
hipError_t hipMalloc(void**, size_t) { return hipErrorOutOfMemory; }
hipError_t hipFree(void*) { return hipSuccess; }
}

int main() {
    pf_plan p;
    for (int a = 0; a < 3; ++a) p.os[a] = 11;
    p.ndim = 3;
    pf_batch b{};
    b.C = b.Cv = b.Cb = b.R = b.L = b.K = b.nfg = b.nimg = 1;
    std::vector<std::thread> t;
    std::atomic<int> bad{0};
    for (int i = 0; i < 8; ++i) t.emplace_back([&] { bad += pf_fft_exec(&p, b, nullptr, 0, nullptr) != PF_OK; });
    for (auto& x : t) x.join();
    std::printf("%d %d %d\n", caches.load(), plans.load(), bad.load());
}
"""


def test_concurrent_first_calls_share_one_cache(tmp_path):
    src, out = tmp_path / "race.cpp", tmp_path / "race"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-w", "-D__HIP_PLATFORM_AMD__", "-I", CSRC,
                    "-I/opt/rocm/include", str(src), "-o", str(out)], check=True)
    run = subprocess.run([str(out)], check=True, capture_output=True, text=True, timeout=60)
    assert run.stdout.split() == ["1", "1", "0"]  # one cache, one plan, no failed call
