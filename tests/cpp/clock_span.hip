// The device clock of a persistent kernel (bar_begin, bar_end): one block's
// last wave waits `wait` ticks before the end; prints the span the clock shows.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "sg_device.hpp"

using namespace sg;

__global__ void k_span(GridBarrier gb, long long wait)
{
    bar_begin(gb, xcc_id());
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x >= blockDim.x - kWave) {
        const long long t0 = wall_clock64();
        while (wall_clock64() - t0 < wait) __builtin_amdgcn_s_sleep(8);
    }
    bar_end(gb);
}

int main(int argc, char **argv)
{
    if (argc != 4) {
        std::fprintf(stderr, "usage: clock_span <blocks> <threads> <ticks>\n");
        return 2;
    }
    const int blocks = std::atoi(argv[1]), threads = std::atoi(argv[2]);
    const long long wait = std::atoll(argv[3]);
    if (blocks < 1 || blocks > 256 || threads < 1 || threads > 1024 || threads % kWave || wait < 0 || wait > 1000000) return 2;
    const size_t bytes = kBarWords * 4 + (1 + blocks) * 8;
    GridBarrier gb{};
    if (hipMalloc((void **)&gb.words, bytes) != hipSuccess || hipMemset(gb.words, 0, bytes) != hipSuccess) return 1;
    gb.clock = (uint64_t *)(gb.words + kBarWords);
    hipLaunchKernelGGL(k_span, dim3(blocks), dim3(threads), 0, 0, gb, wait);
    std::vector<uint64_t> t(1 + blocks);
    if (hipGetLastError() != hipSuccess || hipDeviceSynchronize() != hipSuccess ||
        hipMemcpy(t.data(), gb.clock, t.size() * 8, hipMemcpyDeviceToHost) != hipSuccess)
        return 1;
    std::printf("%llu\n", (unsigned long long)(*std::max_element(t.begin() + 1, t.end()) - t[0]));
    return hipFree(gb.words) == hipSuccess ? 0 : 1;
}
