// The launchers of device.hip over a recording stand-in for the HIP runtime -- test code.
//
// Linked with device.hip compiled for the host only.  Nothing is run: every launch is checked against
// the limits of one (fewer than 2^32 threads along a grid dimension, at most 65535 workgroups along y
// and z) and the pieces of a work list have to follow each other and cover it.
#include <cstdio>
#include <cstring>
#include <vector>

#include "device.hpp"

using namespace mq;

namespace {

struct Launch {
    dim3 grid, block;
    const char* list;  // the kernel argument that walks through the work list
};
std::vector<Launch> launches;
int list_arg = 0;
dim3 next_grid, next_block;

const char* base() { return reinterpret_cast<const char*>(uintptr_t(1) << 20); }
template <class T> const T* list() { return reinterpret_cast<const T*>(base()); }

int bad = 0;
template <class F>
void check(const char* what, int64_t n, size_t elem, int arg, F launch) {
    launches.clear();
    list_arg = arg;
    const hipError_t e = launch();
    int64_t at = 0;
    bool ok = e == hipSuccess && !launches.empty();
    for (Launch const& l : launches) {
        ok = ok && l.grid.x > 0 && uint64_t(l.grid.x) * l.block.x < (uint64_t(1) << 32) && l.grid.y <= 65535 &&
             l.grid.z <= 65535 && l.list == base() + at * int64_t(elem);
        at += l.grid.x;
    }
    ok = ok && at == n;
    printf("%s, %lld workgroups: %zu launches, %s\n", what, (long long)n, launches.size(), ok ? "ok" : "WRONG");
    bad += !ok;
}

}  // namespace

extern "C" {
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t, hipStream_t) {
    next_grid = grid;
    next_block = block;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, hipStream_t* stream) {
    *grid = next_grid;
    *block = next_block;
    *shared = 0;
    *stream = nullptr;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void*, dim3 grid, dim3 block, void** args, size_t, hipStream_t) {
    Launch l{grid, block, nullptr};
    memcpy(&l.list, args[list_arg], sizeof(l.list));
    launches.push_back(l);
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipGetSymbolAddress(void**, const void*) { return hipSuccess; }
void** __hipRegisterFatBinary(const void*) { return nullptr; }
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, dim3*, dim3*, int*) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void**) {}
}

int main() {
    // one launch, and around the largest one of 256 and of 512 threads a workgroup, and several
    for (int64_t n : {int64_t(1), int64_t(1) << 20, (int64_t(1) << 23) - 1, int64_t(1) << 23, (int64_t(1) << 24) - 1,
                      int64_t(1) << 24, (int64_t(1) << 26) + 3}) {
        for (GemmPrec p : {GEMM_F64, GEMM_F32, GEMM_F32_OUT_F64, GEMM_BF3, GEMM_BF3_OUT_F64})
            check("gemm items", n, sizeof(GemmItem), 2, [&] {
                return launch_gemm(p, nullptr, nullptr, list<GemmItem>(), n, nullptr, 0, 0, nullptr, Bases{}, nullptr);
            });
        check("gemm split sums", n, sizeof(GemmReduce), 1, [&] {
            return launch_gemm(GEMM_F64, nullptr, nullptr, nullptr, 0, list<GemmReduce>(), n, 128 * 128, nullptr, Bases{}, nullptr);
        });
        check("term-sum blocks, FP64", n, sizeof(SWork), 1, [&] {
            return launch_sblocks<double>(nullptr, list<SWork>(), n, nullptr, SWorkCounts(), nullptr, nullptr, nullptr,
                                          nullptr, nullptr, nullptr, nullptr, false, nullptr);
        });
        check("term-sum blocks, FP32", n, sizeof(SWork), 1, [&] {
            return launch_sblocks<float>(nullptr, list<SWork>(), n, nullptr, SWorkCounts(), nullptr, nullptr, nullptr,
                                         nullptr, nullptr, nullptr, nullptr, true, nullptr);
        });
        check("small lines", n, sizeof(SSmallWork), 0, [&] {
            return launch_small_lines<double>(list<SSmallWork>(), n, nullptr, nullptr, nullptr, nullptr, nullptr);
        });
        check("lines", n, sizeof(SLine), 0,
              [&] { return launch_slines(list<SLine>(), n, nullptr, nullptr, nullptr, nullptr); });
        check("term gradient", n, sizeof(TermGradWork), 0, [&] {
            return launch_term_grad(list<TermGradWork>(), n, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr);
        });
    }
    return bad != 0;
}
