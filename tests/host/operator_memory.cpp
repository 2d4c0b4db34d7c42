// The operator's build (spmm.hip, host side) on a card with little memory: the HIP calls it makes and the
// kernels it launches are stand-ins that count bytes.  The build by tiles needs a table; where that does
// not fit, the general path has to be taken, whose scratch is smaller, with nothing left allocated and
// no error left for a launch to find.
#include <cstdio>
#include <cstdlib>
#include <map>
#include <string>

#include <hip/hip_runtime.h>

#include "engine.h"

namespace {

size_t g_limit = ~size_t(0), g_used = 0, g_peak = 0;
std::map<void*, size_t> g_blocks;
hipError_t g_last = hipSuccess;
bool g_unsorted = false;
int g_tiles = 0, g_sorts = 0;
std::string g_message;

hipError_t take(void** p, size_t n) {
    if (n > g_limit - g_used) return g_last = hipErrorOutOfMemory;
    *p = std::calloc(1, 64);  // never read as what it stands for
    g_blocks[*p] = n;
    g_used += n;
    g_peak = std::max(g_peak, g_used);
    return hipSuccess;
}
hipError_t give(void* p) {
    if (!p) return hipSuccess;
    g_used -= g_blocks.at(p);
    g_blocks.erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t launched() {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
void require(bool ok, const char* what) {
    if (!ok) {
        std::printf("FAILED: %s (limit %zu, used %zu, %s)\n", what, g_limit, g_used, g_message.c_str());
        std::exit(1);
    }
}

}  // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t n) { return take(p, n); }
hipError_t hipMallocAsync(void** p, size_t n, hipStream_t) { return take(p, n); }
hipError_t hipFree(void* p) { return give(p); }
hipError_t hipFreeAsync(void* p, hipStream_t) { return give(p); }
hipError_t hipGetLastError() { return launched(); }
const char* hipGetErrorString(hipError_t e) { return e == hipSuccess ? "no error" : "out of memory"; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipMemcpy(void*, const void*, size_t, hipMemcpyKind) { return hipSuccess; }
hipError_t hipMemcpyAsync(void* to, const void*, size_t n, hipMemcpyKind k, hipStream_t) {
    if (k == hipMemcpyDeviceToHost && n == sizeof(uint32_t)) *(uint32_t*)to = g_unsorted;
    return hipSuccess;
}
}

namespace fdi {
void set_error(const std::string& m) { g_message = m; }
uint32_t csc_tile_cols(uint64_t, uint64_t C, bool narrow) { return narrow && C < 400000 ? 512 : 2048; }
uint64_t csc_tiles(uint64_t C, uint32_t cols) { return (C + cols - 1) / cols; }
uint64_t csc_tile_groups(uint64_t C, uint32_t cols) { return (csc_tiles(C, cols) + 15) / 16; }
hipError_t launch_fill_u32(uint32_t*, uint64_t, uint32_t, hipStream_t) { return launched(); }
hipError_t launch_fill_u64(uint64_t*, uint64_t, uint64_t, hipStream_t) { return launched(); }
hipError_t launch_scan_u32(const uint32_t*, uint64_t, uint64_t*, uint64_t*, uint64_t*, hipStream_t) {
    return launched();
}
hipError_t launch_global_rows(int, const uint64_t*, const uint64_t*, const uint64_t*, const uint64_t*, uint64_t,
                              uint64_t, uint64_t*, hipStream_t) {
    return launched();
}
hipError_t launch_pack_rows(uint64_t, const uint64_t*, const float*, int, float*, uint16_t*, hipStream_t) {
    return launched();
}
hipError_t launch_row_tiles(uint64_t, const uint64_t*, const uint64_t*, const float*, uint64_t, uint32_t, uint32_t*,
                            float*, uint32_t*, hipStream_t) {
    return launched();
}
hipError_t launch_tile_totals(uint64_t, uint64_t, uint32_t, const uint32_t*, uint32_t*, hipStream_t) {
    return launched();
}
hipError_t launch_place_tiles(int, uint64_t, uint64_t, uint32_t, const uint32_t*, const uint64_t*, const uint64_t*, const float*,
                              const float*, const uint64_t*, uint32_t*, uint64_t*, uint32_t*, void*, hipStream_t) {
    g_tiles++;
    return launched();
}
hipError_t launch_col_count(uint64_t, const uint64_t*, uint32_t*, hipStream_t) { return launched(); }
hipError_t launch_col_scatter(uint64_t, const uint64_t*, const uint64_t*, const void*, int, const uint64_t*, uint32_t*,
                              uint32_t*, void*, hipStream_t) {
    return launched();
}
hipError_t launch_col_sort(uint64_t, const uint64_t*, uint32_t*, void*, int, hipStream_t) {
    g_sorts++;
    return launched();
}
hipError_t launch_spmm(int, uint64_t, const uint64_t*, const uint32_t*, const void*, const float*, const float*, int,
                       uint64_t, uint64_t, float*, hipStream_t) {
    return launched();
}
}  // namespace fdi

namespace {

// The least memory with which the operator of a matrix is built, and the peak with plenty.
struct Needs {
    size_t least, plenty;
    bool tiles;
};
int build(const fd_dosemat& m, int type, size_t limit) {
    g_limit = limit;
    g_used = g_peak = 0;
    g_tiles = g_sorts = 0;
    fd_spmm* p = nullptr;
    const int r = fd_spmm_create(&m, type, &p, nullptr);
    require((r == FD_OK) == (p != nullptr), "an operator or an error");
    require(r == FD_OK || g_message.find("out of memory") != std::string::npos, "the error says what it is");
    require(r != FD_OK || g_tiles + g_sorts == 1, "built once");
    require(g_last == hipSuccess, "no error left behind");
    fd_spmm_destroy(p);
    require(g_used == 0 && g_blocks.empty(), "nothing left allocated");
    return r;
}
Needs needs(const fd_dosemat& m, int type) {
    Needs n{};
    require(build(m, type, size_t(1) << 50) == FD_OK, "built with plenty of memory");
    n.plenty = g_peak;
    n.tiles = g_tiles == 1;
    size_t lo = 0, hi = n.plenty;  // fails with lo, builds with hi
    require(build(m, type, lo) != FD_OK, "not built without memory");
    while (hi - lo > 1) {
        const size_t mid = lo + (hi - lo) / 2;
        (build(m, type, mid) == FD_OK ? hi : lo) = mid;
    }
    n.least = hi;
    return n;
}

}  // namespace

int main() {
    const struct {
        uint64_t rows, cols, nnz;
    } cases[] = {{4000, 262144, 2000000}, {2700, 6400000, 50000000}, {100, 2048, 5000}, {24000, 6400000, 460000000}};
    for (const auto& c : cases)
        for (int type : {FD_VAL_F32, FD_VAL_BF16}) {
            fd_dosemat m{};
            m.n_cols = c.cols;
            m.rows = {c.rows};
            m.nnz = {c.nnz};
            m.off_off = {0};
            m.nnz_off = {0};
            m.used_nnz = c.nnz;
            m.used_off = c.rows + 1;
            g_unsorted = true;  // the general path alone
            const Needs general = needs(m, type);
            require(!general.tiles, "unsorted rows take the general path");
            g_unsorted = false;
            const Needs both = needs(m, type);
            std::printf("rows %llu cols %llu type %d: tiles %zu, general path from %zu\n", (unsigned long long)c.rows,
                        (unsigned long long)c.cols, type, both.plenty, both.least);
            require(both.tiles, "sorted rows take the tiles");
            // what the general path needs without having tried the tiles first
            const uint64_t vb = type == FD_VAL_F32 ? 4 : 2;
            const size_t own = (c.cols + 1) * 8 + c.nnz * 4 + c.nnz * vb + (vb == 2 ? c.rows * 4 : 0) + (c.rows + 1) * 8;
            const size_t scratch = c.cols * 4 + (vb == 2 ? c.nnz * 2 : 0) + fdi::scan_scratch_size(c.cols) * 8;
            require(both.least <= std::max(own + scratch, both.plenty) && both.least <= own + scratch,
                    "built wherever the general path fits");
        }
    std::printf("operator memory: ok\n");
    return 0;
}
