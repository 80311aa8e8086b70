// Resident conjugate gradients: one launch holds a solve on the chip for many
// iterations.  The rows are cut into segments of R slices (64 rows each), one
// segment per block, at most one block per compute unit.  A block keeps the
// part of p that its rows read (its window) in LDS; what the blocks exchange
// in an iteration are two sums and z = D^-1 r.
//
// The same segments, with the same sums, exist as three plain kernels per
// iteration (seg_*), for callers that cannot run the resident kernel; both
// give the same bits.
#pragma once

#include "cg_device.hpp"

namespace ins {

constexpr int RT = 1024;          // threads of a segment block
constexpr int RW = RT / 64;       // its waves
constexpr int RBMAX = 256;        // most segments of a solve
constexpr int LDS_MAX = 160 * 1024;

// Decomposition of one solve into segments (B = 0: none)
struct Seg {
    int B = 0;   // blocks
    int R = 0;   // slices of 64 rows per block
};

// Segment of a block: workgroups go to the XCDs round-robin, so that with B a
// multiple of 8 every XCD gets one contiguous eighth of the rows
__device__ inline int seg_of_block(int id, int B)
{
    return (B % NXCD) ? id : (id % NXCD) * (B / NXCD) + id / NXCD;
}

// ---------------------------------------------------------------------------
// CSR rows: LPR lanes per row, 4 entries per lane in flight (the order of
// csr_row); p(k) gives the vector value of entry k
template <int LPR, typename TV, typename TX, class P>
__device__ inline TX csr_seg_row(int32_t k0, int32_t e, const TV* __restrict__ val, P p)
{
    TX s = (TX)0;
    for (; k0 < e; k0 += 4 * LPR) {
        TV vv[4];
        TX xx[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int32_t k = k0 + j * LPR;
            vv[j] = (k < e) ? val[k] : (TV)0;
            xx[j] = (k < e) ? p(k) : (TX)0;
        }
#pragma unroll
        for (int j = 0; j < 4; j++) s += (TX)vv[j] * xx[j];
    }
    return group_sum<LPR>(s);
}

// f(i) for every item of this thread in segment seg of `sl` slices: the items
// of the resident kernel in its order (component c of item a at c * n + a)
template <int D, class F>
__device__ inline void seg_items(int seg, int sl, int64_t n, F f)
{
    const int lane = threadIdx.x & 63;
    for (int k = wave_in_block(); k < sl; k += RW) {
        const int64_t a = ((int64_t)seg * sl + k) * 64 + lane;
        if (a < n)
#pragma unroll
            for (int c = 0; c < D; c++) f(c * n + a);
    }
}

// launchers (resident.hip)
int resident_blocks(int n_cu);
Seg csr_segments(int64_t n, int lpr, int n_cu);
int csr_windows(Ctx* c, const Seg& g, int vec_bytes);
template <typename T>
int resident_csr(Ctx* c, const Seg& g, int lpr, const T* val, T* x, T* r, T* p, T* z,
                 const T* dinv, int iters, int limit);

}  // namespace ins
