// 3x3 convolution (pad 1, stride 1) for gfx950 with the input patch resident in LDS.
//
// The implicit-GEMM kernel (k_gemm.hip) moves every input pixel into LDS once per tap: nine
// copies of the A tile per 64 channels.  Here a block owns 64 SUB output pixels as SUB 8x8
// sub-tiles and stages, per 64 input channels, the 10x10 pixels around each sub-tile once;
// the nine taps read their A fragments from that patch at shifted addresses, and only the
// weight tile of each tap streams through the ring.
//
// What bounds it: the MFMAs of a step, plus the DMA prologue and the epilogue of a block.  A
// 256 x 160 step is 1280 cycles of MFMA per SIMD against 660 of LDS reads and about 450 of DMA.
// Measured against the implicit-GEMM kernel's best plan (us; fp16 TFLOP/s of the new one):
//   B=1 128x128 512 -> 512   91 -> 62  (1250)     B=16 32x32 640 -> 640  161 -> 96 (1260)
//   B=1 512x512 128 -> 128  111 -> 85 (910)       B=16 64x64 320 -> 320  170 -> 107 (1130)
//   B=2 64x64 320 -> 320   31.1 -> 19.6 (770)     B=2 32x32 640 -> 640  30.5 -> 23.7 (640)
//   B=2 16x16 1280 -> 1280 30.5 -> 22.8 (660)     B=1 512x512 64 -> 64   53.7 -> 37.2 (520)
// Three versions of the loop, same tiles: branches per step and the wait and barrier at its
// head 117 us (B=16 32x32), the fragment reads moved across the barrier 117 us, the taps
// unrolled into straight-line code 97 us: what cost was the scalar work and the branches
// between the barrier and the first MFMA, where all waves of the block stand.
#include "gemm_common.h"

#include <cstdio>
#include <utility>

namespace sdu {

// f(integral_constant 0), f(1), ... f(N - 1)
template <class F, int... I>
__device__ __forceinline__ void static_for_seq(F&& f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
    static_for_seq(f, std::make_integer_sequence<int, N>{});
}

// Tile: NSUB sub-tiles of TW x TW output pixels (TW 16 or 8) x NT output channels, WM x WN
// waves.  v_mfma_f32_16x16x32_f16: A / B operand lane l holds row / column l % 16, K elements
// 8 (l / 16) .. + 8; accumulator element e of lane l is row 4 (l / 16) + e, column l % 16.
//
// K order: units, each the NTAP taps (9, or the sub-pixel form's 4) of one 64-channel chunk as
// NTAP steps of 64, then the chunks of the dense tail (a 1x1 conv over A2 / A3 at the same
// pixels: the centre tap only, one step).  A split-K block takes a contiguous range of units.
//
// LDS: two patches (this chunk's and the next one's, whose loads are spread over this chunk's
// taps) and a ring of NS weight tiles.  Patch pixel (py, px) of sub-tile s is row
// (s (TW + 2) + py) (TW + 2) + px of 128 bytes; its 16-byte channel chunk c sits at slot
// c ^ sw, sw = px / 2 (+ 4 (py % 2) for TW 8) mod 8.  A 16-lane phase of a 16-byte LDS read is
// lanes 0-3, 12-15 of one half of the wave and 4-11 of the next 16 lanes: fragment rows 0-3
// and 12-15 are the 16 pixels' even ones, 4-11 the odd ones, so each half of a phase covers
// the 8 slots of one 128-byte half of the 256-byte bank period, at every tap.
//
// The loop is straight-line code over a chunk's taps: LDS addresses are six registers (tap
// column, swizzle) plus immediates, weights past the block's range are loaded through an
// empty resource so that every wait counts the same DMA, and the fragments of the next half
// step are read during the MFMAs of this one (the block barrier comes in mid-step, after which
// the next weight tile has landed and the oldest one may be overwritten).
//
// ONE: a conv of one 64-channel chunk without a tail or split: no second patch, so two 16x16 tiles
// of 64 channels fit a CU and one's loads and epilogue run beside the other's taps
// (512x512x64 -> 64 with residual 43 us -> 35, 110 MB at 3.1 TB/s; 300x400 22 -> 18; sub-pixel,
// 256x256x64 to 512x512 50 -> 24).
// DMA instructions a wave may have in flight at the barrier of tap t: those issued after the
// step of the weights of step t + 1, i.e. NS - 2 weight tiles and the patch instructions of the
// last NS - 2 taps (none of them before tap 0, see LASTA); after the last tap only what was
// issued after the next chunk's patch.
template <int NTAP, int NS, int BI, int APT, int AI>
constexpr int dma_ahead(int t) {
    int w = (NS - 2) * BI;
    for (int k = 1; k <= NS - 2; ++k)
        for (int i = (t - k) * APT; t - k >= 0 && i < (t - k + 1) * APT && i < AI; ++i) ++w;
    const int since_patch = (t - 1 - (AI - 1) / APT) * BI;
    return t < NTAP - 1 || w < since_patch ? w : since_patch;
}

template <int TW, int NSUB, int NT, int WM, int WN, int NTAP, int NS, int WPE, bool ONE = false>
__global__ __launch_bounds__(WM* WN * 64) __attribute__((amdgpu_waves_per_eu(WPE)))
void conv3_patch_kernel(GemmArgs a) {
    constexpr int NW = WM * WN, NTH = NW * 64, SPX = TW * TW, MT = SPX * NSUB, WTM = MT / WM, WTN = NT / WN;
    constexpr int FM = WTM / 16, FN = WTN / 16;
    constexpr int PW = TW + 2, PPX = PW * PW;
    constexpr int PQ = (NSUB * PPX * 8 + 63) / 64, AI = (PQ + NW - 1) / NW;  // 1 KB DMA instructions: patch, per wave
    constexpr int BQ = NT / 8, BI = (BQ + NW - 1) / NW;                      // weight tile, per wave
    constexpr int PATCH = PQ * 1024, BST = BQ * 1024;                        // bytes
    constexpr int RING = (ONE ? 1 : 2) * PATCH, SMEM = RING + NS * BST;
    // patch DMA of the next chunk: APT instructions in each of the first taps, none in the last one
    // (a ring of all taps: before the first weights of that chunk are asked for)
    constexpr int APT = NS == NTAP ? (NTAP == 9 ? AI : (AI + 1) / 2) : (AI + NTAP - 3) / (NTAP - 2), LASTA = (AI - 1) / APT;
    static_assert(WTM % 32 == 0 && WTN % 16 == 0 && NTAP % NS == 0 && LASTA <= NTAP - NS + (NTAP == 4) && SMEM <= 160 * 1024, "tile");
    static_assert(SPX % WTM == 0 || (TW == 8 && WTM % 64 == 0), "wave rows");
    __shared__ __attribute__((aligned(1024))) char smem[SMEM];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave % WM, wn = wave / WM;

    // block -> (tile of sub-tiles, column tile); a sub-pixel conv's tiles are phase-major
    const int nbx = (a.Win + TW - 1) / TW, nby = (a.Hin + TW - 1) / TW, spi = nbx * nby, nsub = a.Bn * spi;
    const int tpp = (nsub + NSUB - 1) / NSUB;  // tiles (per phase)
    const int tiles_m = NTAP == 4 ? 4 * tpp : tpp, tiles_n = (a.N + NT - 1) / NT;
    const int bid = xcd_block(tiles_m * tiles_n, blockIdx.x);
    int tm, tn;
    if (a.n_major) {
        tn = bid / tiles_m;
        tm = bid - tn * tiles_m;
    } else {
        tm = bid / tiles_n;
        tn = bid - tm * tiles_n;
    }
    const int phase = NTAP == 4 ? tm / tpp : 0;
    const int sub0 = (tm - phase * tpp) * NSUB, n0 = tn * NT;
    const int oy0 = phase >> 1, ox0 = phase & 1;  // sub-pixel phase: first tap's patch offset

    // a sub-tile's image (-1: past the last one) and top-left pixel
    auto sub_at = [&](int s, int& b, int& y, int& x) __attribute__((always_inline)) {
        const int q = sub0 + s;
        b = q / spi;
        const int r = q - b * spi, by = r / nbx;
        y = by * TW;
        x = (r - by * nbx) * TW;
        if (q >= nsub) b = -1;
    };
    int sb0, sy0, sx0, sb1 = -1, sy1 = 0, sx1 = 0;
    sub_at(0, sb0, sy0, sx0);
    static_assert(NSUB <= 2, "sub-tiles");
    if (NSUB > 1) sub_at(1, sb1, sy1, sx1);

    // ---- DMA lane assignment (buffer_load ... lds: lane l of instruction q lands at byte
    // q * 1024 + l * 16).  Patch: row q * 8 + l / 8, slot l % 8; pixels outside the image (and
    // rows past the patch) read past the resource's range: zeros.  A wave without an
    // instruction q repeats its first one.
    constexpr uint32_t kOOB = 0x80000000u;
    uint32_t a_pix[AI], a_ch[AI];  // byte offset = pixel * (2 * channels) + a_ch
#pragma unroll
    for (int i = 0; i < AI; ++i) {
        const int qi = i * NW + wave < PQ ? i * NW + wave : wave;
        const int row = qi * 8 + (lane >> 3), s = row / PPX, r = row - s * PPX, py = r / PW, px = r - py * PW;
        const int b = s == 0 ? sb0 : sb1, y = (s == 0 ? sy0 : sy1) + py - 1, x = (s == 0 ? sx0 : sx1) + px - 1;
        const bool ok = s < NSUB && b >= 0 && y >= 0 && y < a.Hin && x >= 0 && x < a.Win;
        a_pix[i] = ok ? (b * a.Hin + y) * a.Win + x : 0;
        a_ch[i] = ok ? (((lane & 7) ^ ((px >> 1) + (TW == 8 ? 4 * (py & 1) : 0))) & 7) * 16 : kOOB;
    }
    uint32_t voB[BI];
#pragma unroll
    for (int i = 0; i < BI; ++i) {
        const int qi = i * NW + wave < BQ ? i * NW + wave : wave, row = qi * 8 + (lane >> 3);
        voB[i] = (uint32_t)(((phase * a.N + min(n0 + row, a.N - 1)) * a.K) * 2 + (((lane & 7) ^ (row >> 1)) & 7) * 16);
    }
    const int szA = a.Bn * a.Hin * a.Win * a.Cin * 2, szB = (NTAP == 4 ? 4 : 1) * a.N * a.K * 2;
    auto bdma = [&](__amdgpu_buffer_rsrc_t rs, uint32_t vo, int so, int dst) __attribute__((always_inline)) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)(smem + dst), 16, vo, so, 0, 0);
    };

    // the block's units [ubeg, uend): steps split evenly, at chunk boundaries
    const int nc = a.Cin >> 6, ntail = (a.K >> 6) - nc * NTAP;
    auto bound = [&](int z) __attribute__((always_inline)) {
        const int w = (nc * NTAP + ntail) * z / (int)gridDim.z;
        return w <= nc * NTAP ? (w + NTAP / 2) / NTAP : nc + w - nc * NTAP;
    };
    const int ubeg = __builtin_amdgcn_readfirstlane(bound(blockIdx.z));
    const int uend = __builtin_amdgcn_readfirstlane(bound(blockIdx.z + 1));

    // patch source of unit u (an empty resource past the range)
    struct Src {
        __amdgpu_buffer_rsrc_t rs;
        uint32_t ld;
        int so;
    };
    auto src_of = [&](int u) __attribute__((always_inline)) {
        const f16* p = a.A;
        int ld = a.Cin, so = u * 128, sz = szA;
        if (u >= nc) {
            const int kw = a.K1 + (u - nc) * 64;
            const bool t2 = kw < a.K2;
            p = t2 ? a.A2 : a.A3;
            ld = t2 ? a.lda2 : a.lda3;
            so = (kw - (t2 ? a.K1 : a.K2)) * 2;
            sz = a.M * ld * 2;
        }
        return Src{__builtin_amdgcn_make_buffer_rsrc((void*)p, (short)0, u < uend ? sz : 0, 0x00020000), (uint32_t)ld * 2, so};
    };
    auto issue_a = [&](const Src& s, int i, int buf) __attribute__((always_inline)) {
        const int qi = i * NW + wave < PQ ? i * NW + wave : wave;
        bdma(s.rs, __umul24(a_pix[i], s.ld) + a_ch[i], s.so, buf * PATCH + qi * 1024);
    };
    const __amdgpu_buffer_rsrc_t rsB = __builtin_amdgcn_make_buffer_rsrc((void*)a.Wt, (short)0, szB, 0x00020000);
    auto issue_b = [&](__amdgpu_buffer_rsrc_t rs, int kw, int st) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < BI; ++i) {
            const int qi = i * NW + wave < BQ ? i * NW + wave : wave;
            bdma(rs, voB[i], kw * 2, RING + st * BST + qi * 1024);
        }
    };
    // K offset of the weights d steps after the first step of unit u (d < NTAP), and whether
    // the block has that step
    auto kw_of = [&](int u, int d, bool& in) __attribute__((always_inline)) {
        const bool conv = u < nc;
        in = conv ? u < uend : u + d < uend;
        return conv ? d * a.Cin + u * 64 : a.K1 + (u - nc + d) * 64;
    };
    auto issue_b_at = [&](int u, int d, int st) __attribute__((always_inline)) {
        bool in;
        const int kw = kw_of(u, d, in);
        issue_b(__builtin_amdgcn_make_buffer_rsrc((void*)a.Wt, (short)0, in ? szB : 0, 0x00020000), kw, st);
    };

    // ---- epilogue threads: thread t owns the 8 columns oc .. of rows r0 + k * RSTEP of each
    // staged pass (PR rows: 32 of every wave row)
    constexpr int PR = WM * 32, NP = WTM / 32, CPR = NT / 8, RSTEP = NTH / CPR, MAXR = (PR + RSTEP - 1) / RSTEP;
    const int oc = (tid % CPR) * 8, r0 = tid / CPR, n = n0 + oc;
    const bool ep_on = tid < RSTEP * CPR && n < a.N;
    // input pixel of tile row r (row-major in its sub-tile; -1 outside the image) and its image
    auto locate = [&](int r, int& img) __attribute__((always_inline)) {
        const int s = r / SPX, y = (s == 0 ? sy0 : sy1) + (r % SPX) / TW, x = (s == 0 ? sx0 : sx1) + r % TW;
        img = s == 0 ? sb0 : sb1;
        return img >= 0 && y < a.Hin && x < a.Win ? (img * a.Hin + y) * a.Win + x : -1;
    };

    floatx4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = floatx4{};

    // ---- main loop
    const int lq = lane >> 4, lr = lane & 15;
    // pixel (row-major in the fragment's 16) of fragment row r: rows 4q .. 4q+3 are pixels
    // fpix(q) + 0, 2, 4, 6
    auto fpix = [](int q) __attribute__((always_inline)) { return q < 2 ? q : 11 - q; };  // 0, 1, 9, 8
    const int wrow = wm * WTM;
    int oA[3][2], oB[2];  // LDS byte positions: [tap column][swizzle half], [half of the step]
    {
        const int fp = fpix(lr >> 2) + 2 * (lr & 3);
        const int y = (wrow % SPX) / TW + (TW == 8 ? fp >> 3 : 0), x = TW == 8 ? fp & 7 : fp;
#pragma unroll
        for (int kx = 0; kx < 3; ++kx) {
            const int px = x + kx + (NTAP == 4 && kx < 2 ? ox0 : 0);
            const int sw = (px >> 1) + (TW == 8 ? 4 * ((y + oy0) & 1) : 0);
            oA[kx][0] = ((wrow / SPX * PW + y + oy0) * PW + px) * 128 + ((lq ^ sw) & 7) * 16;
            oA[kx][1] = oA[kx][0] ^ 64;
        }
        oB[0] = RING + (wn * WTN + lr) * 128 + ((lq ^ (lr >> 1)) & 7) * 16;
        oB[1] = oB[0] ^ 64;
    }
    half8 af[2][FM], bf[2][FN];
    // the fragments of half ks of tap (ky, kx), weights in ring stage st
    auto load = [&](int ky, int kx, int st, int ks) __attribute__((always_inline)) {
        const char* pA = smem + oA[kx][TW == 8 ? (ky & 1) ^ ks : ks] + ky * PW * 128;
        const char* pB = smem + oB[ks] + st * BST;
#pragma unroll
        for (int i = 0; i < FM; ++i)
            af[ks][i] = *(const half8*)(pA + (TW == 8 ? (i >> 2) * PPX + (i & 3) * 2 * PW : i * PW) * 128);
#pragma unroll
        for (int j = 0; j < FN; ++j) bf[ks][j] = *(const half8*)(pB + j * 2048);
    };
    auto mfma = [&](int ks) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[ks][i], bf[ks][j], acc[i][j], 0, 0, 0);
    };
    // interleave the half step's LDS reads with its MFMAs
    auto weave = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < FM + FN; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // LDS read
        }
        __builtin_amdgcn_sched_group_barrier(0x008, FM * FN, 0);
    };
    auto flip = [&](int by) __attribute__((always_inline)) {
#pragma unroll
        for (int kx = 0; kx < 3; ++kx) {
            oA[kx][0] += by;
            oA[kx][1] += by;
        }
    };
    if (ubeg < uend) {
        const Src s0 = src_of(ubeg);
#pragma unroll
        for (int i = 0; i < AI; ++i) issue_a(s0, i, 0);
#pragma unroll
        for (int d = 0; d < NS; ++d) issue_b_at(ubeg, d, d);
        int pbuf = 0, u = ubeg;
        if (u < nc) {
            wait_vmcnt_lgkm0<(NS - 1) * BI>();
            __builtin_amdgcn_s_barrier();
            __atomic_signal_fence(__ATOMIC_SEQ_CST);
            load(0, 0, 0, 0);
        }
        for (; u < uend && u < nc; ++u) {
            const Src sn = src_of(u + 1);
            static_for<NTAP>([&](auto tap_c) __attribute__((always_inline)) {
                constexpr int tap = decltype(tap_c)::value, TR = NTAP == 9 ? 3 : 2;
                load(tap / TR, tap % TR, tap % NS, 1);
                mfma(0);
                weave();
                __builtin_amdgcn_sched_barrier(0);
                wait_vmcnt_lgkm0<dma_ahead<NTAP, NS, BI, APT, ONE ? 0 : AI>(tap)>();
                __builtin_amdgcn_s_barrier();
                __atomic_signal_fence(__ATOMIC_SEQ_CST);
                if constexpr (tap + NS < NTAP) issue_b(rsB, (tap + NS) * a.Cin + u * 64, tap % NS);
                else issue_b_at(u + 1, tap + NS - NTAP, tap % NS);
#pragma unroll
                for (int i = tap * APT; !ONE && i < (tap + 1) * APT && i < AI; ++i) issue_a(sn, i, pbuf ^ 1);
                if constexpr (tap + 1 < NTAP) {
                    load((tap + 1) / TR, (tap + 1) % TR, (tap + 1) % NS, 0);
                } else {
                    if constexpr (!ONE) flip(pbuf ? -PATCH : PATCH);
                    load(0, 0, 0, 0);  // (unused after the last unit and before the tail)
                }
                mfma(1);
                weave();
                __builtin_amdgcn_sched_barrier(0);
            });
            pbuf ^= 1;
        }
        // the dense tail: centre tap, its patch and weights one step ahead
        for (int st = 0, j = 0; !ONE && u < uend; ++u, ++j) {
            wait_vmcnt_lgkm0<0>();
            __builtin_amdgcn_s_barrier();
            __atomic_signal_fence(__ATOMIC_SEQ_CST);
            const Src sn = src_of(u + 1);
#pragma unroll
            for (int i = 0; i < AI; ++i) issue_a(sn, i, pbuf ^ 1);
            if (j > 0) issue_b_at(u, NS - 1, st == 0 ? NS - 1 : st - 1);
            oB[0] += st * BST;
            oB[1] += st * BST;
            load(1, 1, 0, 0);
            load(1, 1, 0, 1);
            oB[0] -= st * BST;
            oB[1] -= st * BST;
            mfma(0);
            mfma(1);
            __atomic_signal_fence(__ATOMIC_SEQ_CST);
            flip(pbuf ? -PATCH : PATCH);
            pbuf ^= 1;
            st = st == NS - 1 ? 0 : st + 1;
        }
        wait_vmcnt_lgkm0<0>();  // no DMA may land in the LDS the epilogue uses
    }
    __syncthreads();

    constexpr int QPL = FM * FN;  // float4 quads per lane
    if (a.partial && !a.fixup) {
        // split K, reduce kernel: fp32 partial [split][M][N], rows by pixel
        float* P = a.partial + (int64_t)blockIdx.z * a.M * a.N;
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                int img;
                const int m = locate(wrow + i * 16 + fpix(lq) + 2 * e, img);
#pragma unroll
                for (int j = 0; j < FN; ++j) {
                    const int c = n0 + wn * WTN + j * 16 + lr;
                    if (m >= 0 && c < a.N) P[(int64_t)m * a.N + c] = acc[i][j][e];
                }
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
        __syncthreads();        // ... for every wave
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
        for (int z = 0; z < a.splits; ++z) {
            u32x4 pv[QPL];
#pragma unroll
            for (int q = 0; q < QPL; ++q)
                pv[q] = __builtin_amdgcn_raw_buffer_load_b128(rsP, vo_w + q * 1024, z * SLOT * 4, CPOL_SC1);
#pragma unroll
            for (int q = 0; q < QPL; ++q) acc[q / FN][q % FN] += __builtin_bit_cast(floatx4, pv[q]);
        }
    }

    // ---- epilogue: the fp32 tile through LDS in NP passes of PR rows (rows wm * WTM + ip * 32 +
    // [0, 32) of every wave row), 8 columns of one row per thread and step
    constexpr int CST = NT + 4;  // padded fp32 row stride
    static_assert(PR * CST * 4 <= SMEM, "staged pass fits the LDS");
    static_assert(NTH * 32 * 4 <= SMEM, "statistics flush fits the LDS");
    float* Cs = (float*)smem;
    float badd[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) badd[e] = 0.f;
    if (ep_on) {
        if (a.bias) {
            const uint4 bv = *(const uint4*)(a.bias + n);
            const f16* bh = (const f16*)&bv;
#pragma unroll
            for (int e = 0; e < 8; ++e) badd[e] = (float)bh[e];
        }
        if (a.bias2) {
#pragma unroll
            for (int e = 0; e < 8; ++e) badd[e] += a.bias2[n + e];
        }
    }
    const bool do_st = a.stats != nullptr;
    float st[2][2][8];
#pragma unroll
    for (int sl = 0; sl < 2; ++sl)
#pragma unroll
        for (int e = 0; e < 8; ++e) { st[sl][0][e] = 0.f; st[sl][1][e] = 0.f; }
#pragma unroll
    for (int ip = 0; ip < NP; ++ip) {
        int pix[MAXR], img[MAXR];
        uint4 rres[MAXR];
#pragma unroll
        for (int k = 0; k < MAXR; ++k) {
            const int sr = r0 + k * RSTEP;
            pix[k] = -1;
            rres[k] = make_uint4(0, 0, 0, 0);
            if (!ep_on || sr >= PR) continue;
            pix[k] = locate((sr >> 5) * WTM + ip * 32 + (sr & 31), img[k]);
            if (a.res && pix[k] >= 0) rres[k] = *(const uint4*)(a.res + (int64_t)pix[k] * a.ldr + n);
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    Cs[(wm * 32 + i * 16 + fpix(lq) + 2 * e) * CST + wn * WTN + j * 16 + lr] = acc[ip * 2 + i][j][e];
        __syncthreads();
#pragma unroll
        for (int k = 0; k < MAXR; ++k) {
            if (pix[k] < 0) continue;
            float v[8];
            ld8(Cs + (r0 + k * RSTEP) * CST + oc, v);
            const f16* rh = (const f16*)&rres[k];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] += badd[e];
            if (a.res) {
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] += (float)rh[e];
            }
            if (a.act) {
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = apply_act(a.act, v[e]);
            }
            int64_t mo = pix[k];
            if (NTAP == 4) {  // the phase's pixel of the upsampled image
                const int q = pix[k] - img[k] * a.Hin * a.Win, iy = q / a.Win, ix = q - iy * a.Win;
                mo = ((int64_t)img[k] * a.Ho + 2 * iy + oy0) * a.Wo + 2 * ix + ox0;
            }
            if (a.out_mode == OUT_F16) {
                uint4 o;
                f16* oh = (f16*)&o;
#pragma unroll
                for (int e = 0; e < 8; ++e) oh[e] = (f16)v[e];
                *(uint4*)((f16*)a.C + mo * a.ldc + n) = o;
                if (do_st) {
                    const bool s1 = img[k] != sb0;
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const float f = (float)oh[e];
                        if (s1) { st[1][0][e] += f; st[1][1][e] += f * f; }
                        else { st[0][0][e] += f; st[0][1][e] += f * f; }
                    }
                }
            } else {
                float* cp = (float*)a.C + mo * a.ldc + n;
                *(float4*)cp = make_float4(v[0], v[1], v[2], v[3]);
                *(float4*)(cp + 4) = make_float4(v[4], v[5], v[6], v[7]);
            }
        }
    }
    if (do_st) stats_flush<NTH, CPR>(a, st, sb0, NSUB > 1 && sb1 > sb0 ? 2 : 1, n0, (float*)smem);
}

// Tile shapes: sub-tile side, sub-tiles, columns, threads
struct PatchCfg {
    int tw, nsub, nt, threads;
    const char* name[2];
};
static const PatchCfg kPatch[kNumPatch] = {
    {16, 1, 128, 512, {"conv3_patch_kernel<16,1,128,4,2,9>", "conv3_patch_kernel<16,1,128,4,2,4>"}},
    {16, 1, 160, 512, {"conv3_patch_kernel<16,1,160,4,2,9>", ""}},
    {8, 2, 80, 256, {"conv3_patch_kernel<8,2,80,4,1,9>", "conv3_patch_kernel<8,2,80,4,1,4>"}},
    {8, 2, 64, 256, {"conv3_patch_kernel<8,2,64,4,1,9>", "conv3_patch_kernel<8,2,64,4,1,4>"}},
    {8, 2, 64, 256, {"conv3_patch_kernel<8,2,64,4,1,9,9>", ""}},
    {8, 1, 64, 256, {"conv3_patch_kernel<8,1,64,2,2,9,9>", ""}},
    {8, 1, 32, 128, {"conv3_patch_kernel<8,1,32,2,1,9,9>", ""}},
    {16, 1, 64, 512, {"conv3_patch_kernel<16,1,64,4,2,9,3,1>", "conv3_patch_kernel<16,1,64,4,2,4,4,1>"}}};

const char* conv_patch_name(int cfg, bool subpix) { return kPatch[cfg].name[subpix]; }

// (four 160-wide weight tiles do not fit the LDS; the shapes with a ring of all nine taps' weights
// have no four-tap form)
bool conv_patch_one_chunk(int cfg) { return cfg == 7; }

bool conv_patch_subpix(int cfg) { return cfg != 1 && (cfg < 4 || cfg == 7); }

int conv_patch_tiles_m(int cfg, const GemmArgs& a) {
    const PatchCfg& p = kPatch[cfg];
    const int nsub = a.Bn * ((a.Hin + p.tw - 1) / p.tw) * ((a.Win + p.tw - 1) / p.tw);
    return (nsub + p.nsub - 1) / p.nsub * (a.subpix ? 4 : 1);
}

void conv_patch_launch(int cfg, const GemmArgs& a, hipStream_t s) {
    const PatchCfg& p = kPatch[cfg];
    const dim3 grid(conv_patch_tiles_m(cfg, a) * ((a.N + p.nt - 1) / p.nt), 1, a.splits), blk(p.threads);
    switch (cfg * 2 + (a.subpix ? 1 : 0)) {
        case 0: SDU_LAUNCH((conv3_patch_kernel<16, 1, 128, 4, 2, 9, 3, 2>), grid, blk, 0, s, a); break;
        case 1: SDU_LAUNCH((conv3_patch_kernel<16, 1, 128, 4, 2, 4, 4, 2>), grid, blk, 0, s, a); break;
        case 2: SDU_LAUNCH((conv3_patch_kernel<16, 1, 160, 4, 2, 9, 3, 2>), grid, blk, 0, s, a); break;
        case 4: SDU_LAUNCH((conv3_patch_kernel<8, 2, 80, 4, 1, 9, 3, 2>), grid, blk, 0, s, a); break;
        case 5: SDU_LAUNCH((conv3_patch_kernel<8, 2, 80, 4, 1, 4, 4, 1>), grid, blk, 0, s, a); break;
        case 6: SDU_LAUNCH((conv3_patch_kernel<8, 2, 64, 4, 1, 9, 3, 2>), grid, blk, 0, s, a); break;
        case 8: SDU_LAUNCH((conv3_patch_kernel<8, 2, 64, 4, 1, 9, 9, 1>), grid, blk, 0, s, a); break;
        case 10: SDU_LAUNCH((conv3_patch_kernel<8, 1, 64, 2, 2, 9, 9, 1>), grid, blk, 0, s, a); break;
        case 15: SDU_LAUNCH((conv3_patch_kernel<16, 1, 64, 4, 2, 4, 4, 4, true>), grid, blk, 0, s, a); break;
        case 14: SDU_LAUNCH((conv3_patch_kernel<16, 1, 64, 4, 2, 9, 3, 4, true>), grid, blk, 0, s, a); break;
        case 12: SDU_LAUNCH((conv3_patch_kernel<8, 1, 32, 2, 1, 9, 9, 1>), grid, blk, 0, s, a); break;
        case 7: SDU_LAUNCH((conv3_patch_kernel<8, 2, 64, 4, 1, 4, 4, 1>), grid, blk, 0, s, a); break;
    }
}

}  // namespace sdu
