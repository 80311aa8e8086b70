// Device helpers shared by the conjugate-gradient kernels: block decomposition
// and deterministic, atomic-free sums (wave, block, and the totals of block
// partials).
#pragma once

#include "common.hpp"

// Multiply-adds fuse only within one source expression (s += a * b is one
// FMA everywhere), so that an inline function gives the same bits in every
// kernel that holds it.
#pragma clang fp contract(on)

namespace ins {

constexpr int VB = 512;       // threads per block of the vector kernels
constexpr int SB = 256;       // threads per block of the SpMV kernels
constexpr int MAXG = 2048;    // max blocks of a partial-producing kernel
// partial slots
constexpr int P_PQ = 0, P_RR = 1, P_RZ = 2, P_TT = 3, P_BB = 4, NSLOT = 5;

// v of the lane that the DPP control CTRL names, both halves of a double
template <int CTRL, typename T>
__device__ inline T dpp_mov(T v)
{
    if constexpr (sizeof(T) == 4) {
        return __builtin_bit_cast(T, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xf,
                                                              0xf, true));
    } else {
        const uint64_t a = __builtin_bit_cast(uint64_t, v);
        const uint32_t lo = __builtin_amdgcn_mov_dpp((int)(uint32_t)a, CTRL, 0xf, 0xf, true);
        const uint32_t hi = __builtin_amdgcn_mov_dpp((int)(uint32_t)(a >> 32), CTRL, 0xf, 0xf, true);
        return __builtin_bit_cast(T, ((uint64_t)hi << 32) | lo);
    }
}

// Sum over groups of G = 2 .. 16 neighbouring lanes, in every lane: the
// butterfly over xor 1, 2, 4, 8.  Once the groups of 4 (8) agree, the mirror
// of 8 (16) lanes brings the other group's value, so every stage is a DPP
// move (a shuffle through the LDS costs ten times its latency).
template <int G, typename T>
__device__ inline T group_sum(T v)
{
    v += dpp_mov<0xB1>(v);                        // quad_perm 1 0 3 2
    if constexpr (G >= 4) v += dpp_mov<0x4E>(v);  // quad_perm 2 3 0 1
    if constexpr (G >= 8) v += dpp_mov<0x141>(v); // row_half_mirror
    if constexpr (G >= 16) v += dpp_mov<0x140>(v);// row_mirror
    if constexpr (G >= 32) v += __shfl_xor(v, 16, 64);
    return v;
}

__device__ inline double lane_value(double v, int lane)
{
    const uint64_t a = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = __builtin_amdgcn_readlane((int)(uint32_t)a, lane);
    const uint32_t hi = __builtin_amdgcn_readlane((int)(uint32_t)(a >> 32), lane);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// sum over the wave, in every lane: rows of 16 lanes by DPP, then the four
// rows through scalar registers
__device__ inline double wave_sum(double v)
{
    v = group_sum<16>(v);
    return (lane_value(v, 0) + lane_value(v, 16)) + (lane_value(v, 32) + lane_value(v, 48));
}

// sum of v over the block, returned to every thread (fixed order)
template <int NV>
__device__ inline void block_allsum(double (&v)[NV])
{
    __shared__ double sh[NV][16];
#pragma unroll
    for (int k = 0; k < NV; k++) v[k] = wave_sum(v[k]);
    const int nw = blockDim.x >> 6;
    __syncthreads();
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int k = 0; k < NV; k++) sh[k][threadIdx.x >> 6] = v[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NV; k++) {
        double s = 0.;
        for (int w = 0; w < nw; w++) s += sh[k][w];
        v[k] = s;
    }
}

// A block's place in the decomposition of one solve: its index and the
// number of blocks.  A plain launch uses blockIdx/gridDim; a batched launch
// (several solves in one grid) gives every solve the decomposition it has
// alone, so its sums, and hence its iterates, do not depend on the batch.
struct Blk {
    int id, n;
};
__device__ inline Blk grid_blk() { return Blk{(int)blockIdx.x, (int)gridDim.x}; }

// one partial per block
template <int NV>
__device__ inline void block_partials(double (&v)[NV], double* part, const int (&slot)[NV],
                                      Blk b = grid_blk())
{
    block_allsum<NV>(v);
    if (threadIdx.x == 0)
#pragma unroll
        for (int k = 0; k < NV; k++) part[slot[k] * MAXG + b.id] = v[k];
}

// every block: the same total of cnt partials of the given slots
template <int NV>
__device__ inline void totals(const double* part, int cnt, const int (&slot)[NV], double (&t)[NV])
{
#pragma unroll
    for (int k = 0; k < NV; k++) t[k] = 0.;
    for (int i = threadIdx.x; i < cnt; i += blockDim.x)
#pragma unroll
        for (int k = 0; k < NV; k++) t[k] += part[slot[k] * MAXG + i];
    block_allsum<NV>(t);
}

__device__ inline bool leader(Blk b = grid_blk()) { return b.id == 0 && threadIdx.x == 0; }

// this thread's share of totals<NV> (the loads only; block_allsum finishes
// it), so that a kernel can issue them together with its other loads
template <int NV>
__device__ inline void totals_share(const double* part, int cnt, const int (&slot)[NV],
                                    double (&t)[NV])
{
#pragma unroll
    for (int k = 0; k < NV; k++) t[k] = 0.;
    for (int i = threadIdx.x; i < cnt; i += blockDim.x)
#pragma unroll
        for (int k = 0; k < NV; k++) t[k] += part[slot[k] * MAXG + i];
}

// index of the calling wavefront within its block, as a wave-uniform value:
// slice indices derived from it stay in scalar registers, so the per-slice
// offset, pattern and column-offset reads go through the scalar cache rather
// than through one vector load per lane
__device__ inline int wave_in_block() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }

// Workgroups are placed on the 8 XCDs round-robin by block id.
constexpr int NXCD = 8;

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x2 __attribute__((ext_vector_type(2)));

template <typename TV>
__device__ inline void load4(const TV* p, TV (&o)[4])
{
    if constexpr (sizeof(TV) == 4) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(p);
        o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w;
    } else {
        const f64x2 a = *reinterpret_cast<const f64x2*>(p);
        const f64x2 b = *reinterpret_cast<const f64x2*>(p + 2);
        o[0] = a.x; o[1] = a.y; o[2] = b.x; o[3] = b.y;
    }
}

struct SellView {
    const int32_t* perm;   // slice row -> matrix row (null: identity)
    const int64_t* sptr;   // value offset of every slice
    const int32_t* spat;   // column-offset list (pattern) of every slice
    const int32_t* pptr;
    const int32_t* plen;
    const int32_t* pdel;
};

}  // namespace ins
