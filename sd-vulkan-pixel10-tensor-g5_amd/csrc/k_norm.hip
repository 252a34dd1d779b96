// GroupNorm(+SiLU) and LayerNorm for NHWC fp16 activations (memory-bound).
//
// GroupNorm replaces groupnorm_f32.comp / groupnorm_silu.comp (vk_engine.cpp:548-549):
// statistics per (image, group), eps inside the rsqrt, affine, optional SiLU.
// The reference reduces one group per 256-thread workgroup; here the image is
// split into pixel chunks so the whole chip streams the tensor:
//   pass 1 (stats): each block reads a stretch of pixels x all channels with 16-byte
//     loads, reduces per-group sum and sum of squares in fp64 and stores them as mean and
//     squared deviations.
//   pass 2 (apply): adds the partials up; mean = S1/N, var = S2/N - mean^2 in fp64; then
//     y = x * a_c + b_c (a_c = rstd_g gamma_c, b_c = beta_c - mean_g a_c),
//     optional SiLU, 16-byte loads and stores.
// Both passes accept a second source concatenated along channels (the up-path
// skip concat, vk_engine.cpp:678-688), so the concat is never materialised.
// When one (image, group) slab is small (HW * C/G <= 32K elements: the 32x32 and
// smaller levels of the 64x64 UNet) and fits the registers of a 512-thread block,
// a single kernel does it all: the slab is loaded once into registers, the sums and
// sums of squares of x minus the group's first value are reduced in one pass (the
// shift keeps the one-pass variance free of cancellation when the mean dwarfs the
// spread), and the normalised values are stored -- one launch, one read and one
// write of the tensor.
//
// LayerNorm replaces layernorm_f32.comp (vk_engine.cpp:652): one wave per token,
// exact two-pass mean / variance in registers.
#include "sdu_internal.h"

#include <algorithm>
#include <cstdio>

namespace sdu {

static constexpr int GN_THREADS = 512;
static constexpr int GN_MAXG = 32;
static constexpr int GN_MAXC = 2560;

// Blocks of GN_THREADS threads over one image: thread t takes channel octet t % V and pixels
// t / V + k R of its block's P (V = C / 8 octets, R = GN_THREADS / V pixel phases; the
// threads past R V idle), so a block's loads and stores are one linear stretch and a thread's
// channels never change.
struct GnGeom {
    int P, nblk;  // pixels per block, blocks per image
};

static GnGeom gn_geom(int B, int HW, int C, int blocks) {
    const int R = GN_THREADS / (C / 8), want = std::min(HW, std::max(1, blocks / B));
    GnGeom g;
    g.P = ((HW + want - 1) / want + R - 1) / R * R;
    g.nblk = (HW + g.P - 1) / g.P;
    return g;
}

// One statistics block per CU, so that the apply blocks have few partials to add up.
static constexpr int GN_STATS_BLOCKS = 256;
size_t groupnorm_acc_bytes(int B, int G) { return (size_t)std::max(B, GN_STATS_BLOCKS) * G * sizeof(float2); }

// A thread's channel octet of the two-source input: pixel p of image b at src + (b HW + p) ld.
struct GnSrc {
    const f16* p;
    int ld;
};
__device__ __forceinline__ GnSrc gn_src(const f16* x, const f16* x2, int C1, int C2, int ch) {
    return ch < C1 ? GnSrc{x + ch, C1} : GnSrc{x2 + (ch - C1), C2};
}

// Per-group (mean, sum of squared deviations from it) of a block's pixels, stored as
// part[b][block][g]: no atomics and nothing to clear.  The sums are fp64: fp32 ones lose the variance
// of groups whose mean dwarfs their spread, and fp32 ones less a value of the group that of groups
// where that value is an outlier (relative error 1e-3 at 300 spreads); the conversions are no more
// instructions than the shift was.  8 pixels per thread and round, all in flight.  Bound by latency
// at the networks' sizes: 2 x 4096 x 960 with its apply 17.0 us (17.3 to 17.6 with shifted fp32 sums,
// whose shift was one more dependent load; 37.1 with fp64 atomics per 8192 elements and their clear).
__global__ __launch_bounds__(GN_THREADS) void gn_stats_kernel(const f16* x, const f16* x2, int C1, int C2, int HW,
                                                              int P, int G, float2* part) {
    constexpr int U = 8;
    const int C = C1 + C2, V = C / 8, cpg = C / G, R = GN_THREADS / V;
    const int b = blockIdx.y, tid = threadIdx.x;
    const int ph = tid / V, o = tid - ph * V;
    const int p0 = blockIdx.x * P, pe = min(HW, p0 + P);
    // [R][C], rows of C + 2: a group's reads of consecutive rows fall on other banks
    const int S = C + 2;
    __shared__ __attribute__((aligned(16))) double s1[GN_THREADS * 10], s2[GN_THREADS * 10];
    if (ph < R) {
        const GnSrc src = gn_src(x, x2, C1, C2, o * 8);
        const f16* base = src.p + (int64_t)b * HW * src.ld;
        double a[8], q[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) { a[e] = 0.0; q[e] = 0.0; }
        for (int p = p0 + ph; p < pe; p += U * R) {
            uint4 raw[U];
#pragma unroll
            for (int u = 0; u < U; ++u) raw[u] = *(const uint4*)(base + (int64_t)min(p + u * R, pe - 1) * src.ld);
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (p + u * R >= pe) raw[u] = make_uint4(0, 0, 0, 0);
#pragma unroll
            for (int e = 0; e < 8; ++e)
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const double f = (float)((const f16*)&raw[u])[e];
                    a[e] += f;
                    q[e] = fma(f, f, q[e]);
                }
        }
        double2* w1 = (double2*)(s1 + ph * S + o * 8);
        double2* w2 = (double2*)(s2 + ph * S + o * 8);
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
            w1[e / 2] = make_double2(a[e], a[e + 1]);
            w2[e / 2] = make_double2(q[e], q[e + 1]);
        }
    }
    __syncthreads();
    // TPG threads (at most a wave) per group, its R cpg sums dealt over them: with 16 threads that
    // each walked the R rows of their channels, few channels left most of them idle in front of up
    // to 512 dependent adds (2 x 112 x 32 18.7 us with the apply, 2 x 13 x 8 in 8 groups 48.7; 8.7
    // and 8.0 so)
    const int TPG = G > 16 ? 16 : G > 8 ? 32 : 64;
    const int g = tid / TPG, sub = tid % TPG;
    if (g >= G) return;
    double ga = 0.0, gq = 0.0;
    const int dr = TPG / cpg, di = TPG - dr * cpg;
    int r = sub / cpg, i = sub - r * cpg;
#pragma unroll 4
    for (int k = sub; k < R * cpg; k += TPG) {
        const int at = r * S + g * cpg + i;
        ga += s1[at];
        gq += s2[at];
        r += dr;
        i += di;
        if (i >= cpg) { i -= cpg; ++r; }
    }
    for (int off = 1; off < TPG; off <<= 1) {
        ga += __shfl_xor(ga, off);
        gq += __shfl_xor(gq, off);
    }
    const double mean = ga / ((double)(pe - p0) * cpg);
    if (sub == 0) part[((int64_t)b * gridDim.x + blockIdx.x) * G + g] = make_float2((float)mean, (float)(gq - ga * mean));
}

// (v_rcp_f32 is within 1 ulp: an error of 2^-24 in front of the fp16 rounding)
__device__ __forceinline__ float silu_f(float x) { return x * __builtin_amdgcn_rcpf(1.0f + __expf(-x)); }

// Apply y = act((x - mean_g) * rstd_g * gamma + beta): block (i, b) does the pixels of GnGeom's
// block i of image b, GNA_U pixels per thread and round, the next round's loads in flight
// during this one's arithmetic and the first round's during the statistics.
// CST = false: the groups' statistics from gn_stats_kernel's partials, part[b][npart][G] of npart
// blocks of SP pixels (the last one the rest), put together as sums in fp64.  (y may be x: a block
// reads no pixels but its own.)
// CST = true: from per-channel sums st1 [B][C1][2] and st2 [B][C2][2] kept by the GEMM epilogues
// that produced x and x2.
static constexpr int GNA_U = 4;

template <bool CST>
__global__ __launch_bounds__(GN_THREADS) void gn_apply_kernel(const f16* x, const f16* x2, int C1, int C2,
                                                              const f16* gamma, const f16* beta, f16* y, int HW,
                                                              int P, int G, float eps, int silu, const float2* part,
                                                              int npart, int SP, const double* st1, const double* st2) {
    const int C = C1 + C2, V = C / 8, cpg = C / G, R = GN_THREADS / V;
    const int b = blockIdx.y, tid = threadIdx.x;
    const int ph = tid / V, o = tid - ph * V;
    const int p0 = blockIdx.x * P, pe = min(HW, p0 + P);
    const GnSrc src = gn_src(x, x2, C1, C2, o * 8);
    const f16* base = src.p + (int64_t)b * HW * src.ld;
    uint4 raw[GNA_U];
    auto load = [&](uint4 (&v)[GNA_U], int p) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < GNA_U; ++u) v[u] = *(const uint4*)(base + (int64_t)min(p + u * R, pe - 1) * src.ld);
    };
    load(raw, p0 + ph);
    const uint4 gv = *(const uint4*)(gamma + o * 8), bv = *(const uint4*)(beta + o * 8);
    __shared__ float s_mean[GN_MAXG], s_rstd[GN_MAXG];
    __shared__ double2 red[CST ? 1 : GN_THREADS];
    // 16 threads add up each group
    const int g = tid / 16, sub = tid % 16;
    double ga = 0.0, gq = 0.0;
    if constexpr (CST) {
        if (g < G) {
            // 2 channels per round, loads issued together (clamped, weighted 0 / 1)
            for (int i0 = sub; i0 < cpg; i0 += 32) {
                double2 qv[2];
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const int c = g * cpg + min(i0 + 16 * u, cpg - 1);
                    qv[u] = *(const double2*)(c < C1 ? st1 + ((int64_t)b * C1 + c) * 2 : st2 + ((int64_t)b * C2 + (c - C1)) * 2);
                }
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const bool use = i0 + 16 * u < cpg;
                    ga += use ? qv[u].x : 0.0;
                    gq += use ? qv[u].y : 0.0;
                }
            }
        }
    } else {
        // partials dealt over the block in memory order, then the lanes of a group
        const int NP = GN_THREADS / G, pi = tid / G, pg = tid - pi * G;
        const float2* pp = part + (int64_t)b * npart * G + pg;
        if (pi < NP) {
            for (int i0 = pi; i0 < npart; i0 += 4 * NP) {
                float2 v[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) v[u] = pp[(int64_t)min(i0 + u * NP, npart - 1) * G];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int i = i0 + u * NP;
                    const double s = (double)(min(SP, HW - i * SP) * cpg) * (double)v[u].x;
                    ga += i < npart ? s : 0.0;
                    gq += i < npart ? fma(s, (double)v[u].x, (double)v[u].y) : 0.0;
                }
            }
        }
        red[tid] = make_double2(ga, gq);
        __syncthreads();
        ga = 0.0;
        gq = 0.0;
        if (g < G)
            for (int i = sub; i < NP; i += 16) {
                ga += red[i * G + g].x;
                gq += red[i * G + g].y;
            }
    }
#pragma unroll
    for (int off = 1; off < 16; off <<= 1) {
        ga += __shfl_xor(ga, off);
        gq += __shfl_xor(gq, off);
    }
    if (g < G && sub == 0) {
        const double n = (double)HW * cpg;
        const double mean = ga / n;
        const double var = fmax(gq / n - mean * mean, 0.0);
        s_mean[g] = (float)mean;
        s_rstd[g] = (float)(1.0 / sqrt(var + (double)eps));
    }
    __syncthreads();
    if (ph >= R) return;
    float sc[8], sh[8];
    {
        const f16* hg = (const f16*)&gv;
        const f16* hb = (const f16*)&bv;
        int cg = o * 8 / cpg, nb = (cg + 1) * cpg;  // group of channel o * 8, its end
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            if (o * 8 + e >= nb) { ++cg; nb += cpg; }  // channels step by one: one group at a time
            sc[e] = s_rstd[cg] * (float)hg[e];
            sh[e] = (float)hb[e] - s_mean[cg] * sc[e];
        }
    }
    f16* dst = y + (int64_t)b * HW * C + o * 8;
    for (int p = p0 + ph; p < pe; p += GNA_U * R) {
        uint4 nxt[GNA_U];
        load(nxt, p + GNA_U * R);  // (past the end: the last pixel again)
#pragma unroll
        for (int u = 0; u < GNA_U; ++u) {
            const f16* hv = (const f16*)&raw[u];
            uint4 outv;
            f16* ov = (f16*)&outv;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                float z = (float)hv[e] * sc[e] + sh[e];
                if (silu) z = silu_f(z);
                ov[e] = (f16)z;
            }
            if (p + u * R < pe) *(uint4*)(dst + (int64_t)(p + u * R) * C) = outv;
        }
#pragma unroll
        for (int u = 0; u < GNA_U; ++u) raw[u] = nxt[u];
    }
}

// Two apply blocks per CU: each forms the statistics of its image first, a chain of about 3 us
// that more blocks pay again (2 x 4096 x 960: 10.7 us with 512 blocks, 13.1 with 1024, 20.4
// with 2048; 11.8 in a form with 960 blocks, channel tables in LDS and an IEEE division per
// SiLU).  Images from 256 x 256 x 256 on stream at 5.2 TB/s, the rate of a copy; the decoder's 30
// applies 423 us against 499, the batch-16 UNet's 314 against 369.
static constexpr int GNA_BLOCKS = 512;

__global__ void zero_kernel(uint4* p, int64_t n16) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n16) p[i] = make_uint4(0, 0, 0, 0);
}

// ----------------------------------------------------------------- single-pass GroupNorm

// 512 threads: the 8x8 - 32x32 slabs (2.5K - 20K elements) leave most of a 1024-thread
// block idle through its block reductions; per forward the GroupNorms took 418 against
// 434 us at B=2 64x64 and 898 against 976 us at B=16 (256 threads: 467 / 921 us).
static constexpr int GNF_THREADS = 512;

// Sums over the block of two floats per thread, in fp64 across waves; every thread
// gets the results.
__device__ __forceinline__ double2 gnf_block_sum2(float v, float u, double2* red) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        v += __shfl_xor(v, off);
        u += __shfl_xor(u, off);
    }
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (lane == 0) red[wave] = make_double2((double)v, (double)u);
    __syncthreads();
    double2 t = make_double2(0.0, 0.0);
#pragma unroll
    for (int w = 0; w < GNF_THREADS / 64; ++w) {
        t.x += red[w].x;
        t.y += red[w].y;
    }
    return t;
}

// One block per (group, image), grid G * B.  Thread t owns VW consecutive channels (vector
// t % (cpg/VW) of the group) and pixels t / (cpg/VW) + k*P (P = pixels per sweep of the
// block), k < EP: each load / store is one VW*2-byte vector at a fixed stride, and
// vectors never straddle the concat split (C1 and C/G are multiples of VW).
template <int VW>
struct GnfVec;
template <>
struct GnfVec<2> {
    typedef uint32_t T;
    static __device__ T load(__amdgpu_buffer_rsrc_t rs, int off) { return __builtin_amdgcn_raw_buffer_load_b32(rs, off, 0, 0); }
};
template <>
struct GnfVec<4> {
    typedef uint2 T;
    static __device__ T load(__amdgpu_buffer_rsrc_t rs, int off) {
        return __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(rs, off, 0, 0));
    }
};
template <>
struct GnfVec<8> {
    typedef uint4 T;
    static __device__ T load(__amdgpu_buffer_rsrc_t rs, int off) {
        return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0));
    }
};

template <int EP, int VW>
__global__ __launch_bounds__(GNF_THREADS) void gn_fused_kernel(const f16* x, const f16* x2, int C1, int C2,
                                                               const f16* gamma, const f16* beta, f16* y,
                                                               int B, int HW, int G, float eps, int silu) {
    typedef typename GnfVec<VW>::T V;
    __shared__ double2 red[GNF_THREADS / 64];
    const int C = C1 + C2, cpg = C / G, vpg = cpg / VW;
    // Workgroups are dealt round-robin over the 8 XCDs, each with its own L2.  The
    // groups of one image share the 128-byte lines of every pixel row, so each XCD is
    // given whole images (consecutive groups): a line then crosses the fabric once.
    const int nblk = gridDim.x;
    const int q = (nblk & 7) ? (int)blockIdx.x : (int)(blockIdx.x & 7) * (nblk >> 3) + (int)(blockIdx.x >> 3);
    const int g = q % G, b = q / G, tid = threadIdx.x;
    const int P = GNF_THREADS / vpg;
    const int cv = tid % vpg, pp0 = tid / vpg;
    const bool act = pp0 < P;
    const int pp = act ? pp0 : P - 1;
    const int c = g * cpg + VW * cv;
    // All loads are issued before any is used, with 32-bit byte offsets into the
    // source; pixels past HW reload pixel HW-1 and are not accumulated.
    V raw[EP];
    {
        const bool first = c < C1;
        const int Cs = first ? C1 : C2;
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
            (void*)(first ? x : x2), (short)0, B * HW * Cs * 2, 0x00020000);
        const int vo = ((int)b * HW * Cs + (first ? c : c - C1)) * 2;
#pragma unroll
        for (int k = 0; k < EP; ++k) raw[k] = GnfVec<VW>::load(rs, vo + min(pp + k * P, HW - 1) * Cs * 2);
    }
    // One pass over the values shifted by the group's first value (the same element
    // for every thread): the sum and sum of squares of x - shift do not cancel for a
    // group whose mean is large against its spread.  (x - shift is exact in fp32.)
    const int c0 = g * cpg;
    const float shift = (float)(c0 < C1 ? x[(int64_t)b * HW * C1 + c0] : x2[(int64_t)b * HW * C2 + (c0 - C1)]);
    float s = 0.f, ss = 0.f;
#pragma unroll
    for (int k = 0; k < EP; ++k) {
        if (act && pp + k * P < HW) {
            const f16* h = (const f16*)&raw[k];
#pragma unroll
            for (int e = 0; e < VW; ++e) {
                const float dv = (float)h[e] - shift;
                s += dv;
                ss += dv * dv;
            }
        }
    }
    const double n = (double)HW * cpg;
    const double2 t = gnf_block_sum2(s, ss, red);
    const double m1 = t.x / n;
    const double mean = shift + m1;
    const double var = fmax(t.y / n - m1 * m1, 0.0);
    const float mf = (float)mean;
    const float rstd = (float)(1.0 / sqrt(var + (double)eps));
    float sc[VW], sh[VW];
#pragma unroll
    for (int e = 0; e < VW; ++e) {
        sc[e] = rstd * (float)gamma[c + e];
        sh[e] = (float)beta[c + e] - mf * sc[e];
    }
    f16* dst = y + c;
#pragma unroll
    for (int k = 0; k < EP; ++k) {
        const int p = pp + k * P;
        if (!act || p >= HW) continue;
        const f16* h = (const f16*)&raw[k];
        V o;
        f16* oh = (f16*)&o;
#pragma unroll
        for (int e = 0; e < VW; ++e) {
            float z = (float)h[e] * sc[e] + sh[e];
            if (silu) z = silu_f(z);
            oh[e] = (f16)z;
        }
        *(V*)(dst + ((int64_t)b * HW + p) * C) = o;
    }
}

hipError_t zero_launch(void* p, size_t bytes, hipStream_t s) {
    const int64_t n16 = (int64_t)((bytes + 15) / 16);
    if (n16 == 0) return hipSuccess;
    launch_timed("zero_kernel", 0.0, 16.0 * n16, [&] {
        SDU_LAUNCH(zero_kernel, dim3((unsigned)((n16 + 255) / 256)), dim3(256), 0, s, (uint4*)p, n16);
    });
    return hipGetLastError();
}

hipError_t groupnorm_launch(const f16* x, const f16* x2, int C1, int C2, const f16* gamma,
                            const f16* beta, f16* y, int B, int HW, int G, float eps, int silu,
                            void* acc, hipStream_t s) {
    const int C = C1 + C2;
    if (G > GN_MAXG || C > GN_MAXC || C % G || C % 8 || C1 % 8 || (C2 && !x2) || (int64_t)HW * C >= 0x7fffffff)
        return hipErrorInvalidValue;
    const double xbytes = 2.0 * B * HW * C;
    const int cpg = C / G;
    // channels per thread: the widest vector that divides the group and the concat split
    const int vw = (cpg % 8 == 0 && C1 % 8 == 0) ? 8 : (cpg % 4 == 0 && C1 % 4 == 0) ? 4 : 2;
    const int sweep = cpg % 2 == 0 ? GNF_THREADS / (cpg / vw) : 0;  // pixels per block sweep
    const int nsweep = sweep ? (HW + sweep - 1) / sweep : 1 << 30;
    // one block per (image, group) wins while the slab is small (up to 64K elements: the
    // 32x32 concat GroupNorms of B=2, 1920 channels 17.8 against 20.7 us for statistics +
    // apply, 1280 channels 13.9 against 17.8); larger slabs stream faster through the
    // chunked two-kernel path, which spreads them over the chip
    if (cpg % 2 == 0 && C1 % 2 == 0 && cpg / vw <= GNF_THREADS && nsweep <= 32 &&
        (int64_t)HW * cpg <= 65536 && 2 * (int64_t)B * HW * C < 0x7fffffff) {
        const int ep = nsweep <= 4 ? 4 : nsweep <= 8 ? 8 : nsweep <= 16 ? 16 : 32;
        char name[40];
        snprintf(name, sizeof name, "gn_fused_kernel<%d,%d>", ep, vw);
        const dim3 grid(G * B);
        launch_timed(name, 0.0, 2.0 * xbytes, [&] {
#define GNF_LAUNCH(EPV, VWV)                                                                                 \
    SDU_LAUNCH((gn_fused_kernel<EPV, VWV>), grid, dim3(GNF_THREADS), 0, s, x, x2, C1, C2, gamma, beta, y, \
                       B, HW, G, eps, silu)
#define GNF_VW(EPV)                      \
    if (vw == 8) GNF_LAUNCH(EPV, 8);     \
    else if (vw == 4) GNF_LAUNCH(EPV, 4); \
    else GNF_LAUNCH(EPV, 2)
            if (ep == 4) { GNF_VW(4); }
            else if (ep == 8) { GNF_VW(8); }
            else if (ep == 16) { GNF_VW(16); }
            else { GNF_VW(32); }
#undef GNF_VW
#undef GNF_LAUNCH
        });
        return hipGetLastError();
    }
    const GnGeom gs = gn_geom(B, HW, C, GN_STATS_BLOCKS), ga = gn_geom(B, HW, C, GNA_BLOCKS);
    float2* part = (float2*)acc;
    launch_timed("gn_stats_kernel", 0.0, xbytes, [&] {
        SDU_LAUNCH(gn_stats_kernel, dim3(gs.nblk, B), dim3(GN_THREADS), 0, s, x, x2, C1, C2, HW, gs.P, G, part);
    });
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    launch_timed("gn_apply_kernel<0>", 0.0, 2.0 * xbytes, [&] {
        SDU_LAUNCH(gn_apply_kernel<false>, dim3(ga.nblk, B), dim3(GN_THREADS), 0, s, x, x2, C1, C2, gamma, beta, y,
                   HW, ga.P, G, eps, silu, (const float2*)part, gs.nblk, gs.P, (const double*)nullptr, (const double*)nullptr);
    });
    return hipGetLastError();
}

hipError_t groupnorm_apply_stats_launch(const f16* x, const f16* x2, int C1, int C2, const double* st1,
                                        const double* st2, const f16* gamma, const f16* beta, f16* y,
                                        int B, int HW, int G, float eps, int silu, hipStream_t s) {
    const int C = C1 + C2;
    if (G > GN_MAXG || C > GN_MAXC || C % G || C % 8 || C1 % 8 || (C2 && (!x2 || !st2)) || !st1 ||
        (int64_t)HW * C >= 0x7fffffff)
        return hipErrorInvalidValue;
    const double xbytes = 2.0 * B * HW * C;
    const GnGeom ga = gn_geom(B, HW, C, GNA_BLOCKS);
    launch_timed("gn_apply_kernel<1>", 0.0, 2.0 * xbytes, [&] {
        SDU_LAUNCH(gn_apply_kernel<true>, dim3(ga.nblk, B), dim3(GN_THREADS), 0, s, x, x2, C1, C2, gamma, beta, y, HW,
                   ga.P, G, eps, silu, (const float2*)nullptr, 0, 0, st1, st2);
    });
    return hipGetLastError();
}

// ----------------------------------------------------------------- LayerNorm

template <int NV>  // vectors of 8 per lane (C <= NV * 512)
__global__ __launch_bounds__(256) void ln_kernel(const f16* x, const f16* gamma, const f16* beta,
                                                 f16* y, int T, int C, float eps) {
    const int lane = threadIdx.x & 63;
    const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= T) return;
    const int V = C / 8;
    float v[NV][8];
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int vi = lane + i * 64;
        if (vi < V) {
            uint4 raw = *(const uint4*)(x + (int64_t)t * C + vi * 8);
            const f16* hv = (const f16*)&raw;
#pragma unroll
            for (int e = 0; e < 8; ++e) { v[i][e] = (float)hv[e]; s += v[i][e]; }
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[i][e] = 0.f;
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
    const float mean = s / (float)C;
    float q = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i)
        if (lane + i * 64 < V)
#pragma unroll
            for (int e = 0; e < 8; ++e) { const float d = v[i][e] - mean; q += d * d; }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) q += __shfl_xor(q, off);
    const float rstd = rsqrtf(q / (float)C + eps);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int vi = lane + i * 64;
        if (vi < V) {
            uint4 gr = *(const uint4*)(gamma + vi * 8), br = *(const uint4*)(beta + vi * 8);
            const f16* gh = (const f16*)&gr;
            const f16* bh = (const f16*)&br;
            uint4 outv;
            f16* ov = (f16*)&outv;
#pragma unroll
            for (int e = 0; e < 8; ++e) ov[e] = (f16)((v[i][e] - mean) * rstd * (float)gh[e] + (float)bh[e]);
            *(uint4*)(y + (int64_t)t * C + vi * 8) = outv;
        }
    }
}

hipError_t layernorm_launch(const f16* x, const f16* gamma, const f16* beta, f16* y, int T, int C,
                            float eps, hipStream_t s) {
    if (C % 8 || C > 4 * 512) return hipErrorInvalidValue;
    dim3 grid((T + 3) / 4), block(256);
    static const char* kNames[4] = {"ln_kernel<1>", "ln_kernel<2>", "ln_kernel<3>", "ln_kernel<4>"};
    const int v = C <= 512 ? 0 : C <= 1024 ? 1 : C <= 1536 ? 2 : 3;
    launch_timed(kNames[v], 0.0, 4.0 * T * C, [&] {
        if (v == 0) SDU_LAUNCH(ln_kernel<1>, grid, block, 0, s, x, gamma, beta, y, T, C, eps);
        else if (v == 1) SDU_LAUNCH(ln_kernel<2>, grid, block, 0, s, x, gamma, beta, y, T, C, eps);
        else if (v == 2) SDU_LAUNCH(ln_kernel<3>, grid, block, 0, s, x, gamma, beta, y, T, C, eps);
        else SDU_LAUNCH(ln_kernel<4>, grid, block, 0, s, x, gamma, beta, y, T, C, eps);
    });
    return hipGetLastError();
}

}  // namespace sdu
