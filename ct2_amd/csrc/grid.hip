// grid.hip -- ct2's cell binning of the container (particle_to_grid,
// particle.cpp:59-114, 349-362) and its cell accessors (particle.cpp:290-300).
//
// ct2 partitions the active range [rung_begin, n) recursively in place into
// Ncell^3 cells and keeps, per cell, its range of the (now cell-ordered)
// arrays.  Here the range is sorted stably by cell index
// ((ix Ncell) + iy) Ncell + iz, ix = floor(x Ncell / 2^32) (cellsort.h); the
// sorted records carry the positions, and velocities and rungs, set aside as one
// 16-byte record per particle, follow by index.  Inside a cell the particles keep
// their previous relative order, so the result does not depend on scheduling.
#include "cellsort.h"
#include "internal.h"

namespace ct2 {
namespace {

struct GridState {
    uint4* sorted = nullptr;   // [m] (x, y, z, position in the range) in cell order
    uint4* other = nullptr;    // [m] the sort's second buffer
    float4* motion = nullptr;  // [m] (vx, vy, vz, rung) in the old order
    size_t cap = 0;
    void* tmp = nullptr;
    size_t tmp_bytes = 0;
    unsigned long long* starts = nullptr;  // [ncell^3 + 1], absolute container indices
    size_t starts_cap = 0;
    int ncell = 0;
    size_t r0 = 0, r1 = 0;  // the range the starts describe
} g_grid;

struct CellKey {
    uint32_t nc;
    __device__ __forceinline__ uint32_t at(uint32_t x) const { return (uint32_t)(((uint64_t)x * nc) >> 32); }
    __device__ __forceinline__ uint32_t operator()(const uint4& p) const { return (at(p.x) * nc + at(p.y)) * nc + at(p.z); }
};

struct PutStart {
    unsigned long long* starts;
    long r0;
    __device__ __forceinline__ void operator()(long q, long e) const { starts[q] = (unsigned long long)(r0 + e); }
};

__global__ __launch_bounds__(256) void grid_pack(const float* __restrict__ VX, const float* __restrict__ VY,
                                                 const float* __restrict__ VZ, const int8_t* __restrict__ R, long r0,
                                                 long m, float4* __restrict__ motion) {
    const long e = (long)blockIdx.x * 256 + threadIdx.x;
    if (e < m) motion[e] = make_float4(VX[r0 + e], VY[r0 + e], VZ[r0 + e], __int_as_float(R[r0 + e]));
}

// The container's range in the new order, from copies of all it held.
__global__ __launch_bounds__(256) void grid_unpack(const uint4* __restrict__ sorted, const float4* __restrict__ motion,
                                                   long r0, long m, uint32_t* __restrict__ X, uint32_t* __restrict__ Y,
                                                   uint32_t* __restrict__ Z, float* __restrict__ VX,
                                                   float* __restrict__ VY, float* __restrict__ VZ,
                                                   int8_t* __restrict__ R) {
    const long e = (long)blockIdx.x * 256 + threadIdx.x;
    if (e >= m) return;
    const uint4 p = sorted[e];
    const float4 v = motion[p.w];
    X[r0 + e] = p.x;
    Y[r0 + e] = p.y;
    Z[r0 + e] = p.z;
    VX[r0 + e] = v.x;
    VY[r0 + e] = v.y;
    VZ[r0 + e] = v.z;
    R[r0 + e] = (int8_t)__float_as_int(v.w);
}

void free_arrays() {
    dev_free(g_grid.sorted);
    dev_free(g_grid.other);
    dev_free(g_grid.motion);
    g_grid.sorted = g_grid.other = nullptr;
    g_grid.motion = nullptr;
    g_grid.cap = 0;
}

int ensure_arrays(size_t m) {
    if (m <= g_grid.cap) return CT2_OK;
    free_arrays();
    CT2_TRY(dev_alloc((void**)&g_grid.sorted, m * sizeof(uint4), "grid sorted records"));
    CT2_TRY(dev_alloc((void**)&g_grid.other, m * sizeof(uint4), "grid records"));
    CT2_TRY(dev_alloc((void**)&g_grid.motion, m * sizeof(float4), "grid velocities"));
    g_grid.cap = m;
    return CT2_OK;
}

}  // namespace

void release_grid() {
    free_arrays();
    dev_free(g_grid.tmp);
    g_grid.tmp = nullptr;
    g_grid.tmp_bytes = 0;
    dev_free(g_grid.starts);
    g_grid.starts = nullptr;
    g_grid.starts_cap = 0;
    g_grid.ncell = 0;
}

}  // namespace ct2

using namespace ct2;

extern "C" int ct2_particles_to_grid(int ncell, uint64_t* starts) {
    CT2_TRY(require_particles());
    if (ncell < 1 || ncell > CT2_GRID_MAX_NCELL)
        return set_error(CT2_ERR_INVALID, "ncell %d out of [1, %d]", ncell, CT2_GRID_MAX_NCELL);
    Context& c = ctx();
    const long r0 = (long)c.rung_begin, m = (long)c.n - r0;
    const long ncells = (long)ncell * ncell * ncell;
    hipStream_t st = c.stream;
    if (g_grid.starts_cap < (size_t)ncells + 1) {
        dev_free(g_grid.starts);
        g_grid.starts = nullptr;
        g_grid.starts_cap = 0;
        CT2_TRY(dev_alloc((void**)&g_grid.starts, ((size_t)ncells + 1) * 8, "cell starts"));
        g_grid.starts_cap = (size_t)ncells + 1;
    }
    const CellKey key{(uint32_t)ncell};
    if (m > 0) {
        CT2_TRY(ensure_arrays((size_t)m));
        int bits = 1;
        while ((1L << bits) < ncells) ++bits;
        CT2_TRY(cell_sort(c.x + r0, c.y + r0, c.z + r0, (int)m, key, bits, g_grid.sorted, g_grid.other, &g_grid.tmp,
                          &g_grid.tmp_bytes, st));
        const unsigned pb = (unsigned)((m + 255) / 256);
        grid_pack<<<pb, 256, 0, st>>>(c.vx, c.vy, c.vz, c.rung, r0, m, g_grid.motion);
        CT2_LAUNCH_CHECK();
        grid_unpack<<<pb, 256, 0, st>>>(g_grid.sorted, g_grid.motion, r0, m, c.x, c.y, c.z, c.vx, c.vy, c.vz, c.rung);
        CT2_LAUNCH_CHECK();
    }
    CT2_TRY(cell_starts(g_grid.sorted, key, (int)(m > 0 ? m : 0), ncells, PutStart{g_grid.starts, r0}, st));
    if (starts)
        CT2_HIP(hipMemcpyAsync(starts, g_grid.starts, ((size_t)ncells + 1) * 8, hipMemcpyDeviceToHost, st));
    CT2_HIP(hipStreamSynchronize(st));
    g_grid.ncell = ncell;
    g_grid.r0 = (size_t)r0;
    g_grid.r1 = c.n;
    c.forces_valid = false;  // the stored forces no longer match the order
    return CT2_OK;
}
