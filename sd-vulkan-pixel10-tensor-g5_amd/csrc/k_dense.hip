// Dense GEMM for gfx950: C[M,N] = [A | A2][M,K] . W[N,K]^T, fp16 operands, fp32 sums, for K
// (and the split point of a two-source A) a multiple of 64 and N a multiple of 8: every Linear and
// 1x1 conv of the UNet, the text encoder and the decoders.
//
// The product is formed transposed (MFMA rows = output columns): a lane then holds 8
// consecutive columns of its row in two accumulators, so bias, LayerNorm, GEGLU, residual,
// activation, row and channel statistics and the 16-byte stores all work on registers, and
// no wave waits for another between its last MFMA and its stores.
//
// Bound by the LDS reads and DMA waits around the MFMAs at large K (8192 x 4096 x 4096: 242 us,
// 1.14 PFLOP/s, 303 us in gemm_kernel), by the epilogue and its bytes at small K
// (65536 x 2560 x 320 GEGLU 150 us against 221, 65536 x 320 x 320 30 against 37, 16384 x 5120 x
// 640 GEGLU 128 against 172), by one block's latency chain where the shape has few tiles
// (154 x 768 x 768 8.7 against 11.5, a clear launch in both; 7.2 without it).  What gave it: the epilogue in registers (no LDS round trip
// of the tile), the DMA running on across a tile's epilogue, and LDS reads placed among the
// MFMAs.  A 128 x 160 tile spilled and won one shape (16384 x 640 x 3200); rings of 4 to 9
// stages at one block per CU lost 10-30% on operands that come from HBM.
#include "gemm_common.h"

#include <algorithm>
#include <string>

namespace sdu {

// Sum over the 16 lanes of a DPP row, in its last lane (row_shr 1, 2, 4, 8).
__device__ __forceinline__ float row16_sum(float v) {
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x111, 0xf, 0xf, true));
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x112, 0xf, 0xf, true));
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x114, 0xf, 0xf, true));
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x118, 0xf, 0xf, true));
    return v;
}

// Tile MT x NT, WM x WN waves of 16 FM rows x 16 FN columns, K steps of 64
// through a ring of NS stages.  v_mfma_f32_16x16x32_f16 with W as its A operand: fragment row r of
// column tile j is column 32 (j / 2) + 8 (r / 4) + 4 (j % 2) + r % 4 of the wave's, so that
// lane l holds columns 32 (j / 2) + 8 (l / 16) + {0 .. 7} of row l % 16 in tiles j and j + 1.
//
// LDS rows are 128 bytes, 16-byte chunk c of row r at slot c ^ sw(r): sw = r / 2 % 8 for A, and for W
// the same of its fragment row (2 (r / 8 % 4) + r / 2 % 2), which keeps every 16-lane phase of a
// fragment read on distinct banks.
//
// The blocks are persistent (an unsplit launch has at most the resident number of them): the
// DMA runs NS steps ahead across tile boundaries, so a tile's first operands land
// during the previous tile's last steps and epilogue.  DMA past the last tile goes through an
// empty resource, which keeps the wait counts constant; the next half step's fragments are
// read during this one's MFMAs (see conv3_patch_kernel).
// LNC: the LayerNorm consumer (GemmArgs::ln_part).  EP: what the epilogue does after the bias.
enum DenseEp {
    EP_ROWS = 0,   // (+ residual), fp16
    EP_PART = 1,   // the same, keeping row statistics (GemmArgs::row_part)
    EP_STATS = 2,  // the same, keeping channel statistics (GemmArgs::stats)
    EP_GEGLU = 3,  // GEGLU, fp16
    EP_QGELU = 4,  // quick-GELU, fp16
    EP_F32 = 5     // fp32
};
template <int MT, int NT, int WM, int WN, int NS, int WPE, bool LNC, int EP>
__global__ __launch_bounds__(WM* WN * 64) __attribute__((amdgpu_waves_per_eu(WPE)))
void gemm_dense_kernel(GemmArgs a) {
    constexpr int NW = WM * WN, WTM = MT / WM, WTN = NT / WN, FM = WTM / 16, FN = WTN / 16, JP = FN / 2;
    constexpr bool GEGLU = EP == EP_GEGLU;
    constexpr int AI = MT / 8 / NW, BI = NT / 8 / NW, LPT = AI + BI;  // 1 KB DMA instructions per wave and step
    constexpr int ASZ = MT * 128, STAGE = (MT + NT) * 128;            // bytes
    static_assert(WTN == 64 && WTM % 16 == 0 && AI * NW * 8 == MT && BI * NW * 8 == NT, "tile");
    __shared__ __attribute__((aligned(1024))) char smem[NS * STAGE];
    __shared__ float2 red[2][EP == EP_STATS ? WM : 1][EP == EP_STATS ? NT : 1];  // channel statistics of the waves

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave % WM, wn = wave / WM;
    const int lq = lane >> 4, lr = lane & 15;

    const int tiles_n = (a.N + NT - 1) / NT, tiles_m = (a.M + MT - 1) / MT, ntile = tiles_m * tiles_n;
    // rows and columns of virtual block vb (XCD-contiguous tile order)
    auto tile_at = [&](int vb, int& m0, int& n0, int& id) __attribute__((always_inline)) {
        id = xcd_block(ntile, vb);
        int tm, tn;
        if (a.n_major) {
            tn = id / tiles_m;
            tm = id - tn * tiles_m;
        } else {
            tm = id / tiles_n;
            tn = id - tm * tiles_n;
        }
        m0 = __builtin_amdgcn_readfirstlane(tm * MT);
        n0 = __builtin_amdgcn_readfirstlane(tn * NT);
    };
    constexpr uint32_t kOOB = 0x80000000u;
    const int kbeg = blockIdx.z * a.k_per_split;
    const int nk = (min(a.K, kbeg + a.k_per_split) - kbeg) >> 6;

    // ---- DMA: instruction q fills rows 8q .. 8q+7 of its operand tile, lane l row l / 8, slot
    // l % 8; rows past M / N repeat the last one (results never stored).  The issue position:
    // tile ivb, step it, A source.
    uint32_t voA[AI], voB[BI];
    const int crow = lane >> 3;
    int ivb = blockIdx.x, it = 0, im0, in0, iid;
    const f16* asrc;
    int asz, ak;  // source, its bytes, its first K
    auto set_a = [&](bool second) __attribute__((always_inline)) {
        const int ld = second ? a.lda2 : a.lda;
        asrc = second ? a.A2 : a.A;
        asz = a.M * ld * 2;
        ak = second ? a.K1 : 0;
#pragma unroll
        for (int i = 0; i < AI; ++i) {
            const int r = (i * NW + wave) * 8 + crow;
            voA[i] = (uint32_t)(min(im0 + r, a.M - 1) * ld * 2 + (((lane & 7) ^ (r >> 1)) & 7) * 16);
        }
    };
    auto set_tile = [&]() __attribute__((always_inline)) {
        tile_at(ivb, im0, in0, iid);
        set_a(a.A2 && kbeg >= a.K1);
#pragma unroll
        for (int i = 0; i < BI; ++i) {
            const int r = (i * NW + wave) * 8 + crow;
            voB[i] = (uint32_t)(min(in0 + r, a.N - 1) * a.K * 2 + (((lane & 7) ^ (2 * ((r >> 3) & 3) + ((r >> 1) & 1))) & 7) * 16);
        }
    };
    set_tile();
    const int m_first = im0, n_first = in0, id_first = iid;
    const int szB = a.N * a.K * 2;
    auto bdma = [&](__amdgpu_buffer_rsrc_t rs, uint32_t vo, int so, int dst) __attribute__((always_inline)) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)(smem + dst), 16, vo, so, 0, 0);
    };
    auto issue = [&](int so) __attribute__((always_inline)) {
        if (it == nk) {
            it = 0;
            ivb += gridDim.x;
            if (ivb < ntile) set_tile();
        }
        const int k = kbeg + it * 64;
        if (a.A2 && k == a.K1 && it > 0) set_a(true);  // on to the second source
        const bool live = ivb < ntile;
        const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)asrc, (short)0, live ? asz : 0, 0x00020000);
        const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc((void*)a.Wt, (short)0, live ? szB : 0, 0x00020000);
#pragma unroll
        for (int i = 0; i < AI; ++i) bdma(ra, voA[i], (k - ak) * 2, so + (i * NW + wave) * 1024);
#pragma unroll
        for (int i = 0; i < BI; ++i) bdma(rb, voB[i], k * 2, so + ASZ + (i * NW + wave) * 1024);
        ++it;
    };
#pragma nounroll
    for (int p = 0; p < NS; ++p) issue(p * STAGE);

    const int oA0 = (wm * WTM + lr) * 128 + ((lq ^ (lr >> 1)) & 7) * 16;
    const int oB0 = ASZ + (wn * WTN + (lr >> 2) * 8 + (lr & 3)) * 128 + ((lq ^ (2 * ((lr >> 2) & 3) + ((lr >> 1) & 1))) & 7) * 16;
    const int oA[2] = {oA0, oA0 ^ 64}, oB[2] = {oB0, oB0 ^ 64};
    half8 af[2][FM], bf[2][FN];
    auto load = [&](int so, int ks) __attribute__((always_inline)) {
        const char* pA = smem + (oA[ks] + so);
        const char* pB = smem + (oB[ks] + so);
#pragma unroll
        for (int j = 0; j < FN; ++j) bf[ks][j] = *(const half8*)(pB + ((j >> 1) * 32 + (j & 1) * 4) * 128);
#pragma unroll
        for (int i = 0; i < FM; ++i) af[ks][i] = *(const half8*)(pA + i * 2048);
    };
    floatx4 acc[FM][FN];
    auto mfma = [&](int ks) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bf[ks][j], af[ks][i], acc[i][j], 0, 0, 0);
    };
    auto weave = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < FM + FN; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // LDS read
        }
        __builtin_amdgcn_sched_group_barrier(0x008, FM * FN, 0);
    };
    wait_vmcnt_lgkm0<(NS - 1) * LPT>();
    __builtin_amdgcn_s_barrier();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    int so = 0;  // this step's ring stage (bytes)

    for (int vb = blockIdx.x; vb < ntile; vb += gridDim.x) {
    int m0 = m_first, n0 = n_first, bid = id_first;
    if (vb != (int)blockIdx.x) tile_at(vb, m0, n0, bid);
    // epilogue operands: row i * 16 + lr of the wave's rows, columns jp * 32 + 8 lq + {0..7}.
    // Output and residual go through buffer resources of the tile's rows: rows past M are past
    // the resource's range, columns past N get an offset past it (not stored; loads give zeros).
    const int wrow = wm * WTM + lr, mrow = m0 + wrow, ncol = n0 + wn * WTN + lq * 8;
    const int rows = min(MT, a.M - m0);
    uint32_t ocol[JP];  // output column of chunk jp
#pragma unroll
    for (int jp = 0; jp < JP; ++jp) ocol[jp] = ncol + jp * 32 < a.N ? (uint32_t)(GEGLU ? (n0 + wn * WTN) / 2 + jp * 16 + lq * 8 : ncol + jp * 32) : kOOB / 4;
    // the residual, or the LayerNorm consumer's 64-column partials of the row (dealt over its 4
    // lanes), loaded before the K loop (no other block writes them)
    constexpr bool RES = !LNC && (EP == EP_ROWS || EP == EP_PART || EP == EP_STATS);
    constexpr int MAXP = 5;  // K <= 1280
    constexpr bool PRE = RES && EP != EP_STATS;  // (with channel statistics, one row ahead: registers)
    uint4 rres[PRE ? FM : 2][JP];
    float2 lnp[LNC ? FM : 1][MAXP];
    if constexpr (LNC) {
        const int T = a.K >> 6;
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int p = 0; p < MAXP; ++p) {
                const int j = lq + 4 * p;
                lnp[i][p] = j < T ? *(const float2*)(a.ln_part + ((int64_t)j * a.M + min(mrow + i * 16, a.M - 1)) * 2)
                                  : make_float2(0.f, 0.f);
            }
    }
    const __amdgpu_buffer_rsrc_t rsR = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(a.res ? a.res + (int64_t)m0 * a.ldr : a.A), (short)0, a.res ? rows * a.ldr * 2 : 0, 0x00020000);
    auto load_res = [&](int i, int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int jp = 0; jp < JP; ++jp)
            rres[slot][jp] = __builtin_bit_cast(
                uint4, __builtin_amdgcn_raw_buffer_load_b128(rsR, ((wrow + i * 16) * a.ldr + ocol[jp]) * 2, 0, 0));
    };
    if constexpr (PRE) {
#pragma unroll
        for (int i = 0; i < FM; ++i) load_res(i, i);
    }
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = floatx4{};
    load(so, 0);
    // (a later tile's second step landed before the stores of the tile before it)
    const int first_wait = __builtin_amdgcn_readfirstlane(vb != (int)blockIdx.x ? 1 : 0);
#pragma nounroll
    for (int t = 0; t < nk; ++t) {
        const int sn = so == (NS - 1) * STAGE ? 0 : so + STAGE;
        load(so, 1);
        mfma(0);
        weave();
        __builtin_amdgcn_sched_barrier(0);
        // the next step has landed and every wave has read this one
        if (t < first_wait) wait_lgkm0();
        else wait_vmcnt_lgkm0<(NS - 2) * LPT>();
        __builtin_amdgcn_s_barrier();
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        issue(so);
        load(sn, 0);  // (unused after the last step: read again after the epilogue)
        mfma(1);
        weave();
        __builtin_amdgcn_sched_barrier(0);
        so = sn;
    }

    constexpr int QPL = FM * FN;
    if (a.partial && !a.fixup) {
        // split K (one tile per block), reduce kernel: fp32 partial [split][M][N]
        wait_vmcnt_lgkm0<0>();  // no DMA may be in flight when the block's LDS is released
        float* P = a.partial + (int64_t)blockIdx.z * a.M * a.N;
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                const int m = mrow + i * 16, n = ncol + (j >> 1) * 32 + (j & 1) * 4;
                if (m < a.M && n < a.N) *(floatx4*)(P + (int64_t)m * a.N + n) = acc[i][j];
            }
        return;
    }
    if (a.partial) {
        // Split K, in-kernel sum: as in gemm_kernel (device-coherent slot stores, a per-tile
        // arrival counter, the last block sums the slots in slot order).
        constexpr int SLOT = MT * NT, CPOL_SC1 = 1 << 4;
        const __amdgpu_buffer_rsrc_t rsP = __builtin_amdgcn_make_buffer_rsrc(
            (void*)(a.partial + (int64_t)bid * a.splits * SLOT), (short)0, a.splits * SLOT * 4, 0x00020000);
        const uint32_t vo_w = (uint32_t)((wave * QPL * 64 + lane) * 16);
#pragma unroll
        for (int q = 0; q < QPL; ++q)
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[q / FN][q % FN]), rsP, vo_w + q * 1024,
                                                   blockIdx.z * SLOT * 4, CPOL_SC1);
        wait_vmcnt_lgkm0<0>();  // this wave's slot stores are complete
        __syncthreads();
        int* const flag = (int*)smem;
        if (tid == 0) {
            const unsigned prev = __hip_atomic_fetch_add(a.tile_cnt + bid, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const bool last = prev == (unsigned)a.splits - 1;
            if (last) __hip_atomic_store(a.tile_cnt + bid, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            *flag = last;
        }
        __syncthreads();
        if (!*flag) return;
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) acc[i][j] = floatx4{};
        constexpr int QB = 4;  // loads in flight
#pragma nounroll
        for (int z = 0; z < a.splits; ++z) {
#pragma unroll
            for (int q0 = 0; q0 < QPL; q0 += QB) {
                u32x4 pv[QB];
#pragma unroll
                for (int q = 0; q < QB; ++q)
                    pv[q] = __builtin_amdgcn_raw_buffer_load_b128(rsP, vo_w + (q0 + q) * 1024, z * SLOT * 4, CPOL_SC1);
#pragma unroll
                for (int q = 0; q < QB; ++q) acc[(q0 + q) / FN][(q0 + q) % FN] += __builtin_bit_cast(floatx4, pv[q]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }

    // ---- epilogue, in registers
    float ln_r[FM], ln_m[FM];  // rstd, -mean * rstd
    if constexpr (LNC) {
        const float inv_k = 1.0f / (float)a.K;
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            float s1 = 0.f, s2 = 0.f;
#pragma unroll
            for (int p = 0; p < MAXP; ++p) { s1 += lnp[i][p].x; s2 += lnp[i][p].y; }
            s1 += __shfl_xor(s1, 16);
            s2 += __shfl_xor(s2, 16);
            s1 += __shfl_xor(s1, 32);
            s2 += __shfl_xor(s2, 32);
            // one-pass statistics as the reference's layernorm_f32.comp (clamped at 0)
            const float mean = s1 * inv_k;
            ln_r[i] = rsqrtf(fmaxf(s2 * inv_k - mean * mean, 0.f) + a.ln_eps);
            ln_m[i] = -mean * ln_r[i];
        }
    }
    // bias (fp16 and fp32, absent ones through empty resources) and column sums of W
    float badd[JP][8], cs[LNC ? JP : 1][8];
    {
        const __amdgpu_buffer_rsrc_t r1 = __builtin_amdgcn_make_buffer_rsrc((void*)a.bias, (short)0, a.bias ? a.N * 2 : 0, 0x00020000);
        const __amdgpu_buffer_rsrc_t r2 = __builtin_amdgcn_make_buffer_rsrc((void*)a.bias2, (short)0, a.bias2 ? a.N * 4 : 0, 0x00020000);
        const __amdgpu_buffer_rsrc_t r3 = __builtin_amdgcn_make_buffer_rsrc((void*)a.ln_colsum, (short)0, LNC ? a.N * 4 : 0, 0x00020000);
#pragma unroll
        for (int jp = 0; jp < JP; ++jp) {
            const int n = ncol + jp * 32;
            const uint4 bv = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r1, n * 2, 0, 0));
            const f16* bh = (const f16*)&bv;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const floatx4 b2 = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(r2, n * 4 + h * 16, 0, 0));
#pragma unroll
                for (int e = 0; e < 4; ++e) badd[jp][h * 4 + e] = (float)bh[h * 4 + e] + b2[e];
                if constexpr (LNC) {
                    const floatx4 c = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(r3, n * 4 + h * 16, 0, 0));
#pragma unroll
                    for (int e = 0; e < 4; ++e) cs[jp][h * 4 + e] = c[e];
                }
            }
        }
    }
    if constexpr (RES && !PRE) load_res(0, 0);
    wait_vmcnt_lgkm0<0>();  // the DMA in flight (the next tile's first steps) lands before the stores
    auto value = [&](int i, int jp, float (&v)[8]) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            v[e] = acc[i][2 * jp + (e >> 2)][e & 3];
            if constexpr (LNC) v[e] = fmaf(ln_r[i], v[e], ln_m[i] * cs[jp][e]);
            v[e] += badd[jp][e];
        }
    };
    // store one row's 8 values; returns the stored fp16
    constexpr int ESZ = EP == EP_F32 ? 4 : 2;
    const __amdgpu_buffer_rsrc_t rsC = __builtin_amdgcn_make_buffer_rsrc((char*)a.C + (int64_t)m0 * a.ldc * ESZ, (short)0,
                                                                        rows * a.ldc * ESZ, 0x00020000);
    auto store = [&](int i, int jp, const float (&v)[8]) __attribute__((always_inline)) {
        const uint32_t vo = ((uint32_t)(wrow + i * 16) * a.ldc + ocol[jp]) * ESZ;
        uint4 o = make_uint4(0, 0, 0, 0);
        if constexpr (EP == EP_F32) {
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, make_float4(v[0], v[1], v[2], v[3])), rsC, vo, 0, 0);
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, make_float4(v[4], v[5], v[6], v[7])), rsC, vo + 16, 0, 0);
        } else {
            f16* oh = (f16*)&o;
#pragma unroll
            for (int e = 0; e < 8; ++e) oh[e] = (f16)v[e];
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, o), rsC, vo, 0, 0);
        }
        return o;
    };
    if constexpr (GEGLU) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int jp = 0; jp < JP; jp += 2) {
                __builtin_amdgcn_sched_barrier(0);  // one row's values at a time
                float v[8], g[8];
                value(i, jp, v);
                value(i, jp + 1, g);
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] *= gelu_erf(g[e]);
                store(i, jp, v);
            }
    } else {
    // channel statistics (GroupNorm of the consumer): column sums of the wave's rows so far in the
    // current image, slot 0 = the image of the tile's first row, 1 = the next; a 16-row fragment lies
    // in one image (stats_hw % 16 == 0).  The block's waves add up through LDS, so that there is
    // one fp64 atomic per tile and value (one per wave: 52 instead of 24 us for M 8192, N 320,
    // K 1600).
    float st[EP == EP_STATS ? 2 : 1][JP][8];
    const int b0 = EP == EP_STATS ? m0 / a.stats_hw : 0;
    int slot = 0;
    auto flush = [&](int s) __attribute__((always_inline)) {
#pragma unroll
        for (int jp = 0; jp < JP; ++jp)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float t1 = row16_sum(st[0][jp][e]), t2 = row16_sum(st[EP == EP_STATS ? 1 : 0][jp][e]);
                if (lr == 15) red[s][wm][wn * WTN + jp * 32 + lq * 8 + e] = make_float2(t1, t2);
                st[0][jp][e] = 0.f;
                st[EP == EP_STATS ? 1 : 0][jp][e] = 0.f;
            }
    };
    if constexpr (EP == EP_STATS) {
#pragma unroll
        for (int jp = 0; jp < JP; ++jp)
#pragma unroll
            for (int e = 0; e < 8; ++e) { st[0][jp][e] = 0.f; st[1][jp][e] = 0.f; }
    }
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        __builtin_amdgcn_sched_barrier(0);  // one row's values at a time
        const int m = mrow + i * 16, m_f = m0 + wm * WTM + i * 16;
        if constexpr (RES && !PRE) {
            if (i + 1 < FM) load_res(i + 1, (i + 1) & 1);
        }
        if constexpr (EP == EP_STATS) {
            if (slot == 0 && m_f >= (b0 + 1) * a.stats_hw) {
                flush(0);
                slot = 1;
            }
        }
        float s1 = 0.f, s2 = 0.f;  // the row's sums over the wave's 64 columns
#pragma unroll
        for (int jp = 0; jp < JP; ++jp) {
            float v[8];
            value(i, jp, v);
            if constexpr (RES) {
                const f16* rh = (const f16*)&rres[PRE ? i : i & 1][jp];
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] += (float)rh[e];
            }
            if constexpr (EP == EP_QGELU) {
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = apply_act(ACT_QUICK_GELU, v[e]);
            }
            const uint4 o = store(i, jp, v);
            const f16* oh = (const f16*)&o;
            const bool ok = m < a.M && ocol[jp] != kOOB / 4;
            if constexpr (EP == EP_STATS) {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float f = ok ? (float)oh[e] : 0.f;
                    st[0][jp][e] += f;
                    st[1][jp][e] += f * f;
                }
            } else if constexpr (EP == EP_PART) {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float f = ok ? (float)oh[e] : 0.f;
                    s1 += f;
                    s2 += f * f;
                }
            }
        }
        if constexpr (EP == EP_PART) {
            s1 += __shfl_xor(s1, 16);
            s2 += __shfl_xor(s2, 16);
            s1 += __shfl_xor(s1, 32);
            s2 += __shfl_xor(s2, 32);
            const int n = n0 + wn * WTN;
            if (lq == 0 && m < a.M && n < a.N) *(float2*)(a.row_part + ((int64_t)(n >> 6) * a.M + m) * 2) = make_float2(s1, s2);
        }
    }
    if constexpr (EP == EP_STATS) {
        flush(slot);
        if (slot == 0) flush(1);  // (zeros)
        wait_lgkm0();
        __builtin_amdgcn_s_barrier();
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        const int nslot = min(a.M, m0 + MT) - 1 >= (b0 + 1) * a.stats_hw ? 2 : 1;
        for (int q = tid; q < nslot * NT; q += NW * 64) {
            const int s = q / NT, c = q % NT;
            if (n0 + c >= a.N) continue;
            float2 t = red[s][0][c];
#pragma unroll
            for (int w = 1; w < WM; ++w) { t.x += red[s][w][c].x; t.y += red[s][w][c].y; }
            double* d = a.stats + ((int64_t)(b0 + s) * a.N + n0 + c) * 2;
            atomicAdd(d, (double)t.x);
            atomicAdd(d + 1, (double)t.y);
        }
        // (the next tile's epilogue writes red again only after its K loop's barriers)
    }
    }  // !GEGLU
    }  // tiles
}

// Tile shapes: rows, columns, threads
struct DenseCfg {
    int mt, nt, threads, per_cu;  // resident blocks per CU
    const char* name;
};
static const DenseCfg kDense[kNumDense] = {{256, 128, 512, 1, "gemm_dense_kernel<256,128,4,2,3"},
                                           {128, 128, 256, 2, "gemm_dense_kernel<128,128,2,2,2"},
                                           {128, 64, 256, 2, "gemm_dense_kernel<128,64,4,1,3"},
                                           {64, 64, 256, 3, "gemm_dense_kernel<64,64,4,1,3"}};

static int dense_ep(const GemmArgs& a) {
    return a.geglu ? EP_GEGLU : a.stats ? EP_STATS : a.row_part ? EP_PART : a.out_mode == OUT_F32 ? EP_F32 : a.act ? EP_QGELU : EP_ROWS;
}

// Whole K tiles, 8-column chunks, 16-row fragments that lie in one image (channel statistics),
// and the combinations of epilogue options that have a variant.  A tile's 256 output (and
// residual) rows must lie within 1 GiB: the epilogue's byte offsets are 32 bits, and a column past N
// gets one of 1 GiB and up to be past the rows.  (gemm_kernel's are 64 bits.)
bool dense_ok(const GemmArgs& a) {
    if (a.amode != A_DENSE || a.K % 64 || (a.A2 && a.K1 % 64) || a.N % 8) return false;
    if (256LL * a.ldc * (a.out_mode == OUT_F32 ? 4 : 2) > 1 << 30 || (a.res && 256LL * a.ldr * 2 > 1 << 30)) return false;
    if (a.geglu) return !a.res && !a.act && a.out_mode == OUT_F16;
    if (a.ln_part || a.row_part || a.stats)
        return !a.act && a.out_mode == OUT_F16 && !(a.row_part && a.stats) &&
               (a.ln_part ? !a.res && !a.row_part && !a.stats : !a.stats || a.stats_hw % 16 == 0);
    if (a.out_mode == OUT_F32 || a.act) return !a.res && a.out_mode != OUT_F32_NCHW && (a.out_mode == OUT_F16 ? a.act == ACT_QUICK_GELU : !a.act);
    return a.out_mode == OUT_F16;
}

std::string dense_name(int cfg, const GemmArgs& a) {
    return std::string(kDense[cfg].name) + (a.ln_part ? ",1," : ",0,") + std::to_string(dense_ep(a)) + ">";
}

template <int MT, int NT, int WM, int WN, int NS, int WPE>
static void launch(dim3 grid, dim3 blk, const GemmArgs& a, hipStream_t s) {
    switch (dense_ep(a) * 2 + (a.ln_part ? 1 : 0)) {
        case 2 * EP_ROWS: SDU_LAUNCH((gemm_dense_kernel<MT, NT, WM, WN, NS, WPE, false, EP_ROWS>), grid, blk, 0, s, a); break;
        case 2 * EP_ROWS + 1: SDU_LAUNCH((gemm_dense_kernel<MT, NT, WM, WN, NS, WPE, true, EP_ROWS>), grid, blk, 0, s, a); break;
        case 2 * EP_PART: SDU_LAUNCH((gemm_dense_kernel<MT, NT, WM, WN, NS, WPE, false, EP_PART>), grid, blk, 0, s, a); break;
        case 2 * EP_STATS: SDU_LAUNCH((gemm_dense_kernel<MT, NT, WM, WN, NS, WPE, false, EP_STATS>), grid, blk, 0, s, a); break;
        case 2 * EP_GEGLU: SDU_LAUNCH((gemm_dense_kernel<MT, NT, WM, WN, NS, WPE, false, EP_GEGLU>), grid, blk, 0, s, a); break;
        case 2 * EP_GEGLU + 1: SDU_LAUNCH((gemm_dense_kernel<MT, NT, WM, WN, NS, WPE, true, EP_GEGLU>), grid, blk, 0, s, a); break;
        case 2 * EP_QGELU: SDU_LAUNCH((gemm_dense_kernel<MT, NT, WM, WN, NS, WPE, false, EP_QGELU>), grid, blk, 0, s, a); break;
        case 2 * EP_F32: SDU_LAUNCH((gemm_dense_kernel<MT, NT, WM, WN, NS, WPE, false, EP_F32>), grid, blk, 0, s, a); break;
    }
}

void dense_launch(int cfg, const GemmArgs& a, hipStream_t s) {
    const DenseCfg& d = kDense[cfg];
    int tiles = ((a.M + d.mt - 1) / d.mt) * ((a.N + d.nt - 1) / d.nt);
    if (a.splits == 1) tiles = std::min(tiles, 256 * d.per_cu);
    const dim3 grid(tiles, 1, a.splits), blk(d.threads);
    switch (cfg) {
        case 0: launch<256, 128, 4, 2, 3, 2>(grid, blk, a, s); break;
        case 1: launch<128, 128, 2, 2, 2, 2>(grid, blk, a, s); break;
        case 2: launch<128, 64, 4, 1, 3, 2>(grid, blk, a, s); break;
        case 3: launch<64, 64, 4, 1, 3, 3>(grid, blk, a, s); break;
    }
}

}  // namespace sdu
