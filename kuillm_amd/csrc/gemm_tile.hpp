// MFMA GEMM for the sizes between the decode GEMMs and the 256x256-tile
// kernels: `gemm_tile_kernel`, output tiles of BM x BN chosen per call.
#pragma once

#include "common.hpp"

namespace kuiops {

struct GemmArgs {
    int64_t M, N, K;
    const void *A; int64_t lda, stride_a;
    const void *B; int64_t ldb, stride_b;
    void *out; int64_t ldo, stride_o;
    const void *cin; int64_t ldcin; int c_kind;
    float alpha, beta;
    int64_t k_per_split;   // multiple of 64 (gemm_tile_kernel: of its K step)
    int splits;
    int tiles_m, tiles_n;
    int vec_store;         // 16-byte row-segment epilogue (ldo, N % 8 == 0, aligned out)
    int raster;            // tile order within a batch entry: 0 = groups of 8 tile-rows, 1 = row by row
    float *partial;        // split-K workspace [splits][M][N]
};

typedef __attribute__((address_space(3))) char lds_char;
typedef short s16x4 __attribute__((ext_vector_type(4)));

// Generic -> LDS address-space cast.  A direct cast keeps the pointer's
// provenance (an integer round trip would hide which LDS array it points
// into, and the compiler would then make every LDS read wait for all
// in-flight LDS-DMA loads).
__device__ __forceinline__ lds_char *to_lds(const void *p) {
    return (lds_char *)(const_cast<void *>(p));
}

// Global -> LDS copy (buffer_load ... lds): a wave-uniform descriptor
// (SGPRs), a per-lane 32-bit byte offset and a uniform byte offset, so the
// K-step advance costs no per-lane address registers.  16 bytes per lane go
// to dst + 16 * lane; reads past `bytes` return 0.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void *base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ void dma16_buf(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff, const void *dst) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void *)to_lds(dst), 16,
                                             (int)voff, (int)soff, 0, 0);
}

// Uniform (wave-invariant) pointer kept in SGPRs: buffer descriptors built
// from it need no per-lane waterfall loop around each DMA.
__device__ __forceinline__ const char *uniform_ptr(const char *p) {
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return reinterpret_cast<const char *>(((uint64_t)hi << 32) | lo);
}

// 4-byte form (64 x 4 bytes to dst + 4 * lane).
__device__ __forceinline__ void dma4_buf(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff, const void *dst) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void *)to_lds(dst), 4,
                                             (int)voff, (int)soff, 0, 0);
}

// vmcnt-only wait (expcnt / lgkmcnt left at their maxima), N < 64.
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    static_assert(N >= 0 && N < 64, "vmcnt out of range");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// Batched tile order: the linear id runs over batch x tiles; after the XCD
// remap (dispatch is round-robin over the 8 XCDs) each batch entry's tiles
// are contiguous (so one XCD's L2 holds its A and B), and tiles are grouped
// by 8 tile-rows within the entry.
__device__ __forceinline__ void tile_coords_batched(int bid, int nblocks, int tiles_m, int tiles_n,
                                                    int &tm, int &tn, int &bz, int raster = 0) {
    const int xcd = bid & 7, idx = bid >> 3;
    const int q = nblocks >> 3, r = nblocks & 7;
    const int pid = xcd * q + (xcd < r ? xcd : r) + idx;
    const int per = tiles_m * tiles_n;
    bz = pid / per;
    const int t = pid - bz * per;
    if (raster) {
        // row by row: the tiles one XCD runs at once lie side by side, so
        // their row segments of the output form whole rows
        tm = t / tiles_n;
        tn = t - tm * tiles_n;
        return;
    }
    const int G = 8;
    const int width = G * tiles_n;
    const int group = t / width;
    const int first_m = group * G;
    const int gsz = min(tiles_m - first_m, G);
    const int in_group = t - group * width;
    tm = first_m + in_group % gsz;
    tn = in_group / gsz;
}

// 16-byte-chunk swizzle of a row-major B row k of BN columns in LDS.  A
// ds_read_b64_tr_b16 serves 4 rows x 64 bytes per cycle; the 64-byte units
// of rows k .. k + 3 must fall on the four quarters of the 64 banks (256
// bytes): rows of 128 or 384 bytes alternate between two quarters by
// themselves and need one more bit, longer rows (multiples of 256) need two.
template <int BN>
__device__ __forceinline__ int swz_brow(int k) {
    return BN % 128 ? ((k >> 1) & 1) << 2 : (k & 3) << 2;
}

// gemm_tile_kernel: BM x BN output tiles (WM x WN waves of TM x TN 32x32
// accumulators; WK = 2 gives each half of the waves one of a stage's two 64-k
// slices), NS LDS-DMA stages, any M, N and K % 8 == 0.
//
// What bounds it: the loads.  A CU holds about 32 KB of loads in flight
// whatever the kernel asks for (buffer_load to LDS or to registers, 4 to 16
// waves, 2 to 16 stages: 45-53 GB/s per CU from HBM with 32 or 70 CUs loading,
// 128 GB/s from a warm L2), so the time is the tile's bytes over that rate.
// Deeper stages, a whole stage of fragments held in registers and touching
// weight lines ahead of the DMA (each of the work-groups sharing them a part)
// were within 5% of this form; larger tiles are what helps, and K splits where
// they leave CUs idle.  Register-staged tiles of the same size
// (gemm_mfma_kernel) wait for a whole load latency per stage: 512 x 11264 x
// 2048 49 -> 32 us.
template <typename T, bool BCOL, typename Tout, int WM, int WN, int WK, int TM, int TN, int NS, bool SPLIT>
__global__ __launch_bounds__(WM * WN * WK * 64) void gemm_tile_kernel(GemmArgs a) {
    constexpr int NW = WM * WN * WK;                 // waves
    constexpr int BM = WM * TM * 32, BN = WN * TN * 32, BK = 64 * WK;
    constexpr int ASUB = BM * 128, BSUB = BN * 128;  // bytes of one 64-k slice
    constexpr int SB = (ASUB + BSUB) * WK;           // bytes per stage
    constexpr int DA = BM * WK / 8 / NW, DB = BN * WK / 8 / NW;   // 1 KB DMA blocks per wave and stage
    constexpr int CPB = BN / 8;                      // 16-byte chunks per row-major B row
    static_assert(BM * WK / 8 % NW == 0 && BN * WK / 8 % NW == 0, "DMA split");
    static_assert(NS == 3 || NS == 4, "stages");
    typedef typename Mfma<T>::frag frag;
    // One array per stage: the compiler tracks LDS-DMA writes per underlying
    // object, so reads of one stage need not wait for the DMA filling another.
    __shared__ __attribute__((aligned(1024))) char s0[SB], s1[SB], s2[SB], s3[NS > 3 ? SB : 16];
    char *const S[4] = {s0, s1, s2, s3};

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wk = wave / (WM * WN), wm = wave / WN % WM, wn = wave % WN;
    int tm, tn, bz;
    tile_coords_batched(blockIdx.x, gridDim.x, a.tiles_m, a.tiles_n, tm, tn, bz, a.raster);
    tm = __builtin_amdgcn_readfirstlane(tm);
    tn = __builtin_amdgcn_readfirstlane(tn);
    bz = __builtin_amdgcn_readfirstlane(bz);
    const int64_t M = a.M, N = a.N, lda = a.lda, ldb = a.ldb;
    const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
    const int split = SPLIT ? blockIdx.y : 0;
    const int kbeg = SPLIT ? (int)(split * a.k_per_split) : 0;
    const int kend = SPLIT ? (int)min(a.K, kbeg + a.k_per_split) : (int)a.K;
    const int nk = (kend - kbeg + BK - 1) / BK;

    const T *Ab = reinterpret_cast<const T *>(a.A) + bz * a.stride_a + m0 * lda + kbeg;
    const T *Bb = reinterpret_cast<const T *>(a.B) + bz * a.stride_b + (BCOL ? n0 * ldb + kbeg : kbeg * ldb + n0);
    // Descriptors end at the operand's last element; kOut is an offset past
    // every descriptor (reads zeros).
    constexpr uint32_t kOut = 0x80000000u;
    const int64_t endA = ((M - 1 - m0) * lda + (kend - kbeg)) * 2;
    const int64_t endB = (BCOL ? (N - 1 - n0) * ldb + (kend - kbeg) : (kend - kbeg - 1) * ldb + N - n0) * 2;
    const __amdgpu_buffer_rsrc_t rsA = make_rsrc(uniform_ptr(reinterpret_cast<const char *>(Ab)), (uint32_t)min(endA, (int64_t)0x7fffffff));
    const __amdgpu_buffer_rsrc_t rsB = make_rsrc(uniform_ptr(reinterpret_cast<const char *>(Bb)), (uint32_t)min(endB, (int64_t)0x7fffffff));

    // K-contiguous rows (128 bytes): chunk c of row r sits at c ^ swzK(r).
    auto swzK = [](int r) { return (r >> 1) & 7; };
    uint32_t goffA[DA], goffB[DB];
    int kA[DA], kB[DB];           // k of the lane's chunk within the stage
#pragma unroll
    for (int j = 0; j < DA; ++j) {
        const int blk = wave * DA + j, sub = blk / (BM / 8);
        const int r = (blk % (BM / 8)) * 8 + (lane >> 3);
        kA[j] = sub * 64 + (((lane & 7) ^ swzK(r)) << 3);
        goffA[j] = m0 + r < M ? (uint32_t)((r * lda + kA[j]) * 2) : kOut;
    }
#pragma unroll
    for (int j = 0; j < DB; ++j) {
        const int blk = wave * DB + j;
        if constexpr (BCOL) {
            const int sub = blk / (BN / 8);
            const int r = (blk % (BN / 8)) * 8 + (lane >> 3);
            kB[j] = sub * 64 + (((lane & 7) ^ swzK(r)) << 3);
            goffB[j] = n0 + r < N ? (uint32_t)((r * ldb + kB[j]) * 2) : kOut;
        } else {
            const int ch = blk * 64 + lane, k = ch / CPB;
            const int c = (ch % CPB) ^ swz_brow<BN>(k & 63);
            kB[j] = k;
            goffB[j] = n0 + c * 8 < N ? (uint32_t)((k * ldb + c * 8) * 2) : kOut;
        }
    }
    const uint32_t stepA = BK * 2;
    const uint32_t stepB = BCOL ? (uint32_t)(BK * 2) : (uint32_t)(BK * ldb * 2);
    const int kspan = kend - kbeg;
    // DMA blocks b0 .. b1 - 1 (A's, then B's) of stage kt into buffer st.
    // Chunks past K are switched off by their offset (they read zeros without
    // memory traffic), so no DMA is conditional and the waits count exactly;
    // stages past the last read nothing.
    constexpr int PER = DA + DB;
    auto issue = [&](int kt, char *st, int b0, int b1) __attribute__((always_inline)) {
        const int left = kspan - kt * BK;
        const uint32_t ka = left > 0 ? (uint32_t)kt * stepA : 0u, kb = left > 0 ? (uint32_t)kt * stepB : 0u;
#pragma unroll
        for (int b = b0; b < b1; ++b) {
            if (b < DA) {
                dma16_buf(rsA, kA[b] < left ? goffA[b] : kOut, ka, st + (wave * DA + b) * 1024);
            } else {
                const int j = b - DA;
                dma16_buf(rsB, kB[j] < left ? goffB[j] : kOut, kb, st + ASUB * WK + (wave * DB + j) * 1024);
            }
        }
    };

    const int lrow = lane & 31, lk = lane >> 5;
    int offA[4], offB[BCOL ? 4 : TN];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
        const int r = wm * TM * 32 + lrow;
        offA[kk] = wk * ASUB + r * 128 + (((2 * kk + lk) ^ swzK(r)) << 4);
    }
    if constexpr (BCOL) {
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
            const int r = wn * TN * 32 + lrow;
            offB[kk] = ASUB * WK + wk * BSUB + r * 128 + (((2 * kk + lk) ^ swzK(r)) << 4);
        }
    } else {
        const int G = lane >> 4, q = lane & 15;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int kr = 8 * (G >> 1) + (q >> 2);
            const int n = wn * TN * 32 + j * 32 + 16 * (G & 1) + 4 * (q & 3);
            offB[j] = ASUB * WK + wk * BSUB + kr * (BN * 2) + (((n >> 3) ^ swz_brow<BN>(kr)) << 4) + ((n >> 2) & 1) * 8;
        }
    }

    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

    // Operands are swapped (B first): a lane's accumulator holds one output
    // row and 4 consecutive columns per 8-column group.
    frag fa[2][TM], fb[2][TN];
    auto rd = [&](const char *st, int kk, int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
            fa[slot][i] = as_frag<frag>(*reinterpret_cast<const u32x4 *>(st + offA[kk] + i * 32 * 128));
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            if constexpr (BCOL) {
                fb[slot][j] = as_frag<frag>(*reinterpret_cast<const u32x4 *>(st + offB[kk] + j * 32 * 128));
            } else {
                const s16x4 t0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (__attribute__((address_space(3))) s16x4 *)to_lds(st + offB[j] + kk * 16 * (BN * 2)));
                const s16x4 t1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (__attribute__((address_space(3))) s16x4 *)to_lds(st + offB[j] + (kk * 16 + 4) * (BN * 2)));
                const u32x2 h0 = __builtin_bit_cast(u32x2, t0), h1 = __builtin_bit_cast(u32x2, t1);
                fb[slot][j] = as_frag<frag>(u32x4{h0[0], h0[1], h1[0], h1[1]});
            }
        }
    };
    // MFMAs of one 16-k step from fragment slot `slot`, with the LDS reads of
    // the next step and `ndma` DMA instructions spread between them.
    constexpr int NM = TM * TN, NRD = TM + (BCOL ? 1 : 2) * TN;
    auto mm = [&](int slot, int ndma) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = Mfma<T>::m32(fb[slot][j], fa[slot][i], acc[i][j]);
#pragma unroll
        for (int t = 0; t < NM; ++t) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
#pragma unroll
            for (int u = NRD * t / NM; u < NRD * (t + 1) / NM; ++u) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
#pragma unroll
            for (int u = ndma * t / NM; u < ndma * (t + 1) / NM; ++u) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // Stage kt in slot sl of the ring, its first fragments already read.  The
    // reads of each 16-k step go out under the MFMAs of the step before; ahead
    // of the last step every wave waits for its DMA of the next stage and the
    // work-group meets, so the next stage's first reads and the refill of this
    // stage's buffer (half of its DMA here, half under the next stage's first
    // step) run under MFMAs too.
    constexpr int H = (PER + 1) / 2;
    auto step = [&](int kt, int sl) __attribute__((always_inline)) {
        char *const cur = S[sl], *const nxt = S[(sl + 1) % NS], *const prv = S[(sl + NS - 1) % NS];
        rd(cur, 1, 1);
        issue(kt + NS - 1, prv, H, PER);
        mm(0, PER - H);
        rd(cur, 2, 0);
        mm(1, 0);
        rd(cur, 3, 1);
        mm(0, 0);
        wait_vmcnt<(NS - 2) * PER>();               // this wave's DMA of stage kt + 1
        __builtin_amdgcn_s_waitcnt(0xc07f);         // and its LDS reads of stage kt
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        rd(nxt, 0, 0);
        issue(kt + NS, cur, 0, H);
        mm(1, H);
    };

#pragma unroll
    for (int s = 0; s < NS - 1; ++s) issue(s, S[s], 0, PER);
    issue(NS - 1, S[NS - 1], 0, H);
    wait_vmcnt<(NS - 2) * PER + H>();
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    rd(S[0], 0, 0);
    // Whole rounds of the stage ring, then the rest (no branch inside the
    // loop: the compiler's wait insertion is not path-sensitive and would
    // make LDS reads wait for all DMA in flight).
    int kt = 0;
    for (; kt + NS <= nk; kt += NS) {
#pragma unroll
        for (int s = 0; s < NS; ++s) step(kt + s, s);
    }
#pragma unroll
    for (int s = 0; s < NS - 1; ++s)
        if (kt + s < nk) step(kt + s, s);
    wait_vmcnt<0>();
    __syncthreads();

    // The K slices of a WK = 2 work-group meet in LDS (slice 0 + slice 1).
    if constexpr (WK == 2) {
        float *red = reinterpret_cast<float *>(s0) + (wave % (WM * WN)) * (TM * TN * 1024);
        static_assert(WM * WN * TM * TN * 4096 <= SB, "slice sums fit a stage");
        if (wk == 1) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int g = 0; g < 4; ++g)
                        *reinterpret_cast<f32x4 *>(red + ((i * TN + j) * 4 + g) * 256 + lane * 4) =
                            f32x4{acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
        }
        __syncthreads();
        if (wk == 0) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const f32x4 v = *reinterpret_cast<const f32x4 *>(red + ((i * TN + j) * 4 + g) * 256 + lane * 4);
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[i][j][4 * g + e] += v[e];
                    }
        }
    }

    const Tout *cin = reinterpret_cast<const Tout *>(a.cin);
    // the 4 output values of columns col .. col + 3 (row, col in the matrix)
    auto value4 = [&](int i, int j, int g, int64_t row, int64_t col, float v[4]) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = a.alpha * acc[i][j][4 * g + e];
        if (a.c_kind == KUIOPS_C_ROW) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] += col + e < N ? a.beta * to_f32(cin[col + e]) : 0.f;
        } else if (a.c_kind == KUIOPS_C_FULL && row < M) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] += col + e < N ? a.beta * to_f32(cin[row * a.ldcin + col + e]) : 0.f;
        }
    };
    if constexpr (SPLIT || sizeof(Tout) == 4) {
        // fp32 partials (or outputs): 16 bytes per lane
        float *out = SPLIT ? a.partial + (int64_t)split * M * N : reinterpret_cast<float *>(a.out) + bz * a.stride_o;
        const int64_t ldo = SPLIT ? N : a.ldo;
        if (wk == 0) {
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                const int64_t row = m0 + wm * TM * 32 + i * 32 + lrow;
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const int64_t col = n0 + wn * TN * 32 + j * 32 + 8 * g + 4 * lk;
                        float v[4];
                        if constexpr (SPLIT) {
#pragma unroll
                            for (int e = 0; e < 4; ++e) v[e] = acc[i][j][4 * g + e];
                        } else {
                            value4(i, j, g, row, col, v);
                        }
                        if (row >= M) continue;
                        float *p = out + row * ldo + col;
                        if (a.vec_store && col + 3 < N) {
                            *reinterpret_cast<f32x4 *>(p) = f32x4{v[0], v[1], v[2], v[3]};
                        } else {
#pragma unroll
                            for (int e = 0; e < 4; ++e)
                                if (col + e < N) p[e] = v[e];
                        }
                    }
            }
        }
    } else {
        // The rows of accumulator row i (32 per wave row) pass through LDS
        // (16-byte chunks XOR-swizzled by row) and leave as whole row
        // segments, 16 bytes per lane; i alternates between two stage arrays,
        // so one barrier separates a pass's writes from its reads.
        Tout *out = reinterpret_cast<Tout *>(a.out) + bz * a.stride_o;
        constexpr int RB = BN * 2, ROWS = WM * 32, CPR = BN / 8;
        static_assert(ROWS * RB <= SB, "row band fits a stage");
        if constexpr (WK == 2) __syncthreads();
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            char *band = i & 1 ? s0 : s1;
            if (wk == 0) {
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const int r = wm * 32 + lrow, cl = wn * TN * 32 + j * 32 + 8 * g + 4 * lk;
                        float v[4];
                        value4(i, j, g, m0 + wm * TM * 32 + i * 32 + lrow, n0 + cl, v);
                        typedef Tout t4 __attribute__((ext_vector_type(4)));
                        t4 w;
#pragma unroll
                        for (int e = 0; e < 4; ++e) w[e] = from_f32<Tout>(v[e]);
                        *reinterpret_cast<u32x2 *>(band + r * RB + (((cl >> 3) ^ (r & 7)) << 4) + lk * 8) =
                            __builtin_bit_cast(u32x2, w);
                    }
            }
            __syncthreads();
            for (int ch = tid; ch < ROWS * CPR; ch += NW * 64) {
                const int r = ch / CPR, c = ch % CPR;
                const int64_t row = m0 + (r >> 5) * TM * 32 + i * 32 + (r & 31), col = n0 + c * 8;
                if (row >= M || col >= N) continue;
                const u32x4 v = *reinterpret_cast<const u32x4 *>(band + r * RB + ((c ^ (r & 7)) << 4));
                if (a.vec_store) {
                    *reinterpret_cast<u32x4 *>(out + row * a.ldo + col) = v;
                } else {
                    const Tout *e8 = reinterpret_cast<const Tout *>(&v);
                    for (int e = 0; e < 8; ++e)
                        if (col + e < N) out[row * a.ldo + col + e] = e8[e];
                }
            }
        }
    }
}

// Sums split-K partials in split order, then applies alpha / beta / addend.
// Four columns per thread (VEC: N % 4 == 0, an output aligned for it), 64 of
// them across and 4 rows per work-group; the partials of up to four splits
// are loaded before they are added.
template <typename Tout, bool VEC>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(GemmArgs a) {
    constexpr int V = VEC ? 4 : 1;
    const int64_t total = a.M * a.N;
    const int64_t col = ((int64_t)blockIdx.x * 64 + (threadIdx.x & 63)) * V;
    if (col >= a.N) return;
    const Tout *cin = reinterpret_cast<const Tout *>(a.cin);
    for (int64_t row = (int64_t)blockIdx.y * 4 + (threadIdx.x >> 6); row < a.M; row += (int64_t)gridDim.y * 4) {
        const float *p = a.partial + row * a.N + col;
        float s[V];
#pragma unroll
        for (int e = 0; e < V; ++e) s[e] = 0.f;
        for (int z = 0; z < a.splits; z += 4) {
            float t[4][V];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (z + i >= a.splits) {
#pragma unroll
                    for (int e = 0; e < V; ++e) t[i][e] = 0.f;
                } else if constexpr (VEC) {
                    const f32x4 v = *reinterpret_cast<const f32x4 *>(p + (z + i) * total);
#pragma unroll
                    for (int e = 0; e < V; ++e) t[i][e] = v[e];
                } else {
                    t[i][0] = p[(z + i) * total];
                }
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int e = 0; e < V; ++e) s[e] += t[i][e];
        }
        Tout o[V];
#pragma unroll
        for (int e = 0; e < V; ++e) {
            float v = a.alpha * s[e];
            if (a.c_kind == KUIOPS_C_FULL) v += a.beta * to_f32(cin[row * a.ldcin + col + e]);
            else if (a.c_kind == KUIOPS_C_ROW) v += a.beta * to_f32(cin[col + e]);
            o[e] = from_f32<Tout>(v);
        }
        Tout *out = reinterpret_cast<Tout *>(a.out) + row * a.ldo + col;
        if constexpr (VEC) {
            typedef Tout tv __attribute__((ext_vector_type(4)));
            *reinterpret_cast<tv *>(out) = tv{o[0], o[1], o[2], o[3]};
        } else {
            *out = o[0];
        }
    }
}

}  // namespace kuiops
