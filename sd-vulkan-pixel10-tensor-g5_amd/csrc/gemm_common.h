// Device helpers shared by the MFMA kernels (k_gemm.hip, k_conv.hip, k_dense.hip).
#pragma once

#include "sdu_internal.h"

namespace sdu {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// s_waitcnt vmcnt(N) lgkmcnt(0): at most N vector-memory ops (the DMA of later
// tiles) outstanding, and every LDS read of this wave complete, so that after the
// following barrier no wave still reads the ring stage the next DMA overwrites.
template <int N>
__device__ __forceinline__ void wait_vmcnt_lgkm0() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 0xF) | (0x7 << 4) | (0x0 << 8) | ((N >> 4) << 14));
}

// lgkmcnt(0) alone
__device__ __forceinline__ void wait_lgkm0() { __builtin_amdgcn_s_waitcnt(0xF | (0x7 << 4) | (0x0 << 8) | (0x3 << 14)); }

// Sum the per-thread column statistics of a block over the threads that own the same
// 8 columns (thread t owns chunk t % CPR; chunk c covers columns col0 + 8c ..) through
// LDS and add them to the per-(image, channel) fp64 statistics of images b0 and (nslot 2)
// b0 + 1, one atomic per value, the sums spread over all threads (each one's NTH / CPR LDS
// reads issued together).  red must hold NTH * 32 floats and be free (the caller's last LDS
// use is complete after the first barrier here).  Value v of thread t sits at v * NTH +
// (t ^ v): the stores (one v, consecutive t) and the loads (consecutive v, one t) both fall
// on distinct banks (a thread-major layout, 32 floats per thread, put every lane of a
// store on one bank).
template <int NTH, int CPR>
__device__ __forceinline__ void stats_flush(const GemmArgs& a, const float (&st)[2][2][8], int b0, int nslot,
                                            int col0, float* red) {
    static_assert(NTH % 32 == 0, "swizzle stays within a row");
    const int tid = threadIdx.x;
    __syncthreads();
#pragma unroll
    for (int sl = 0; sl < 2; ++sl)
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int v = sl * 16 + q * 8 + e;
                red[v * NTH + (tid ^ v)] = st[sl][q][e];
            }
    __syncthreads();
    // value v of chunk c: slot v / 16, sum (0) or sum of squares (1) = (v / 8) % 2, column v % 8
    // (thread t owns chunk t % CPR; threads past the last whole group of CPR kept zeros)
#pragma unroll
    for (int q = tid; q < CPR * 32; q += NTH) {
        const int c = q >> 5, v = q & 31;
        const int col = col0 + c * 8 + (v & 7);
        if ((v >> 4) >= nslot || col >= a.N) continue;
        float t = 0.f;
#pragma unroll
        for (int j = 0; j < NTH / CPR; ++j) t += red[v * NTH + ((c + j * CPR) ^ v)];
        atomicAdd(&a.stats[((int64_t)(b0 + (v >> 4)) * a.N + col) * 2 + ((v >> 3) & 1)], (double)t);
    }
}

// 8 consecutive fp32 values from 16-byte-aligned LDS
__device__ __forceinline__ void ld8(const float* p, float (&v)[8]) {
    const float4 x = *(const float4*)p, y = *(const float4*)(p + 4);
    v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w; v[4] = y.x; v[5] = y.y; v[6] = y.z; v[7] = y.w;
}

// Logical block id of this workgroup: hardware ids go round-robin over the 8 XCDs; each XCD
// gets a contiguous range of the nblk logical tiles (XCD x: nblk / 8 tiles, one more for the
// first nblk % 8 XCDs), so that neighbouring tiles share that XCD's L2.
// (vb: the hardware id, or a persistent block's id plus a multiple of its grid.)
__device__ __forceinline__ int xcd_block(int nblk, int vb) {
    const int xcd = vb & 7, per = nblk >> 3, extra = nblk & 7;
    return xcd * per + min(xcd, extra) + (vb >> 3);
}

}  // namespace sdu
