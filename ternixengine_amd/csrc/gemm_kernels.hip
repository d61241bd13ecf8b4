// gemm_kernels.hip -- gfx950 LDS-tiled int8-MFMA GEMM kernels (M > 32, and 33..64 narrow tiles) for
// the ternary matmul, and their launcher.  Shared helpers, the weight layout and the decode forms are
// described in kernel_common.h.

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdlib.h>

#include <algorithm>
#include <type_traits>

#include "kernel_common.h"
#include "ternary_kernels.h"

namespace ternix_hip {
namespace {

// ------------------------------------------------------------------------------------------------
// LDS-tiled GEMM (prefill shapes).
//
// Workgroup tile BM x (4*BNB) outputs, BNB packed byte-columns, k-step 64.  4 waves in a 2 x 2 grid,
// wave tile (BM/2) rows x (BNB/2) byte-columns; per k-step a wave issues (BM/32) x (BNB/32) x 4
// MFMAs.  A tile in LDS: BM rows x 64 bytes, 16-byte chunks XOR-swizzled by (row/4)%4 so the 16 rows
// read by one ds_read_b128 land on distinct banks.  W tile in LDS is stored transposed (byte-column
// major, the 64 k-rows of a byte-column contiguous, pitch 80 bytes) so a lane's B fragment is one
// ds_read_b128; the transpose is done in registers (v_perm) between the global load and the LDS
// store.  Two LDS stages: global loads of step s+1 are issued before the MFMAs of step s.
// ------------------------------------------------------------------------------------------------

constexpr int GM_THREADS = 256;
constexpr int WT_PITCH = 80;  // bytes per transposed byte-column (64 k-rows + 16 pad)

template <int BM, int BNB, bool ALIGNED_W, bool ALIGNED_A>
__global__ __launch_bounds__(GM_THREADS) void gemm_kernel(const int8_t* __restrict__ A, const uint8_t* __restrict__ B,
                                                          int32_t* __restrict__ C, int M, int K, int N,
                                                          int tiles_n, int k_begin, int k_end, int accumulate,
                                                          int vec_store, int k_split, OutScale os) {
    if (gridDim.y > 1) {  // split-K: this workgroup's k-range, partial tile in slab blockIdx.y
        k_begin += (int)blockIdx.y * k_split;
        k_end = min(k_end, k_begin + k_split);
        C += (size_t)blockIdx.y * (size_t)M * (size_t)N;
    }
    constexpr int WM = BM / 2;            // rows per wave
    constexpr int WB = BNB / 2;           // byte-columns per wave
    constexpr int MT = WM / 16;           // m-tiles per wave
    constexpr int GT = WB / 16;           // 16-byte-column groups per wave
    constexpr int A_CHUNKS = BM * 4;      // 16-byte chunks per A stage
    constexpr int A_PER_T = A_CHUNKS / GM_THREADS;
    constexpr int W_JOBS = (BNB / 4) * 16;  // (dword column, row quad) jobs per W stage
    constexpr int W_PER_T = (W_JOBS + GM_THREADS - 1) / GM_THREADS;
    static_assert(A_CHUNKS % GM_THREADS == 0, "A tile must split evenly");

    __shared__ __attribute__((aligned(16))) int8_t sA[2][BM * 64];
    __shared__ __attribute__((aligned(16))) uint8_t sW[2][BNB * WT_PITCH];

    const int NB = N >> 2;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int q = lane & 15, kb = lane >> 4;

    // Block -> tile: consecutive block ids are dealt round-robin over the 8 XCDs; regroup so that
    // each XCD works on a contiguous run of tiles (neighbouring tiles share A rows / W columns in
    // that XCD's L2).
    const int nblocks = gridDim.x;
    const int bid = blockIdx.x;
    const int per_xcd = (nblocks + 7) >> 3;
    const int xcd = bid & 7, slot = bid >> 3;
    int tile = xcd * per_xcd + slot;
    if ((nblocks & 7) != 0) tile = bid;  // uneven split: keep the plain order
    const int tm = tile / tiles_n, tn = tile % tiles_n;
    const int row0 = tm * BM;
    const int bc0 = tn * BNB;
    // k-steps cover [k_begin, k_end); k_begin % 64 == 0.  Loads treat k >= k_end as zero.
    const int nsteps = (k_end - k_begin + 63) >> 6;

    v4i areg[A_PER_T];
    uint32_t wreg[W_PER_T][4];

    auto gload = [&](int s) {
        const int k0 = k_begin + s * 64;
#pragma unroll
        for (int p = 0; p < A_PER_T; ++p) {
            const int c = tid + p * GM_THREADS;
            const int r = c >> 2, ch = c & 3;
            areg[p] = load_a16_range<ALIGNED_A>(A, row0 + r, k0 + ch * 16, M, K, k_end);
        }
#pragma unroll
        for (int p = 0; p < W_PER_T; ++p) {
            const int job = tid + p * GM_THREADS;
            if (job < W_JOBS) {
                const int dc = job % (BNB / 4), rq = job / (BNB / 4);
#pragma unroll
                for (int r = 0; r < 4; ++r) wreg[p][r] = load_w4<ALIGNED_W>(B, k0 + 4 * rq + r, bc0 + 4 * dc, k_end, NB);
            }
        }
    };
    auto sstore = [&](int buf) {
#pragma unroll
        for (int p = 0; p < A_PER_T; ++p) {
            const int c = tid + p * GM_THREADS;
            const int r = c >> 2, ch = c & 3;
            const int sw = ch ^ ((r >> 2) & 3);
            *reinterpret_cast<v4i*>(&sA[buf][r * 64 + sw * 16]) = areg[p];
        }
#pragma unroll
        for (int p = 0; p < W_PER_T; ++p) {
            const int job = tid + p * GM_THREADS;
            if (job < W_JOBS) {
                const int dc = job % (BNB / 4), rq = job / (BNB / 4);
                uint32_t c0, c1, c2, c3;
                transpose4x4(wreg[p][0], wreg[p][1], wreg[p][2], wreg[p][3], c0, c1, c2, c3);
                uint8_t* base = &sW[buf][(4 * dc) * WT_PITCH + 4 * rq];
                *reinterpret_cast<uint32_t*>(base) = c0;
                *reinterpret_cast<uint32_t*>(base + WT_PITCH) = c1;
                *reinterpret_cast<uint32_t*>(base + 2 * WT_PITCH) = c2;
                *reinterpret_cast<uint32_t*>(base + 3 * WT_PITCH) = c3;
            }
        }
    };

    v4i acc[MT][GT][4];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int g = 0; g < GT; ++g)
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[t][g][j] = v4i{0, 0, 0, 0};

    if (nsteps > 0) {
        gload(0);
        sstore(0);
    }
    __syncthreads();

    for (int s = 0; s < nsteps; ++s) {
        const int buf = s & 1;
        if (s + 1 < nsteps) gload(s + 1);

        // B fragments for this wave: GT groups of 16 byte-columns, 16 k-rows each.
        v4i bfr[GT][4];
#pragma unroll
        for (int g = 0; g < GT; ++g) {
            const int col = wn * WB + g * 16 + q;
            const v4i x4 = *reinterpret_cast<const v4i*>(&sW[buf][col * WT_PITCH + kb * 16]);
#pragma unroll
            for (int rq = 0; rq < 4; ++rq) {
                const uint32_t x = (uint32_t)x4[rq];
                bfr[g][0][rq] = (int)((x << 6) & 0xC0C0C0C0u);
                bfr[g][1][rq] = (int)((x << 4) & 0xC0C0C0C0u);
                bfr[g][2][rq] = (int)((x << 2) & 0xC0C0C0C0u);
                bfr[g][3][rq] = (int)(x & 0xC0C0C0C0u);
            }
        }
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            const int r = wm * WM + t * 16 + q;
            const int sw = kb ^ ((r >> 2) & 3);
            const v4i a = *reinterpret_cast<const v4i*>(&sA[buf][r * 64 + sw * 16]);
#pragma unroll
            for (int g = 0; g < GT; ++g)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[t][g][j] = mfma_i8(a, bfr[g][j], acc[t][g][j]);
        }

        if (s + 1 < nsteps) sstore(buf ^ 1);
        __syncthreads();
    }

    // Epilogue: element i of tile (t, g, j) is row 4*kb + i of m-tile t, column 4*(byte-col) + j.
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int row = row0 + wm * WM + t * 16 + 4 * kb + i;
            if (row >= M) continue;
#pragma unroll
            for (int g = 0; g < GT; ++g) {
                const int bcol = bc0 + wn * WB + g * 16 + q;
                if (bcol >= NB) continue;
                v4i v = {acc[t][g][0][i] >> 6, acc[t][g][1][i] >> 6, acc[t][g][2][i] >> 6, acc[t][g][3][i] >> 6};
                if (os.Y) {  // dequantised float output: y = c * (row_scale[row] * w_scale)
                    store_scaled(os, row, N, 4 * bcol, v, vec_store);
                    continue;
                }
                int32_t* out = C + (size_t)row * (size_t)N + 4 * bcol;
                if (vec_store) {
                    if (accumulate) v += *reinterpret_cast<const v4i*>(out);
                    __builtin_nontemporal_store(v, reinterpret_cast<v4i*>(out));  // streamed, not re-read
                } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j) out[j] = accumulate ? out[j] + v[j] : v[j];
                }
            }
        }
}

constexpr int GF_BNB = 64;

__device__ __forceinline__ int gf_swz_a(int r) { return (r >> 1) & 7; }
__device__ __forceinline__ int gf_swz_w(int r) { return ((r >> 1) & 3) ^ ((r >> 4) & 1); }
// W swizzle for a given stage-row width: 64-byte rows as gf_swz_w; 32-byte rows (two chunks) keep the
// 8 rows of one transposing read on distinct banks by their pitch alone and flip the chunk for the
// second 16-row half of a wave's k-block, which is read in the same pass.
template <int BNB>
__device__ __forceinline__ int swz_w(int r) { return BNB == 64 ? gf_swz_w(r) : (BNB == 32 ? ((r >> 4) & 1) : 0); }

// ------------------------------------------------------------------------------------------------
// GEMM on v_mfma_i32_16x16x64_i8: the 64-row tiles of 256 columns (4 waves, 64 x 64 outputs each, two
// workgroups per CU) and the 64 x 64 tiles of up to 64 rows.  K % BK == 0, aligned A and W.
//   * A and W both go global -> LDS with direct 16-byte loads (global_load_lds_dwordx4): no registers
//     held, so NS stages are in flight.  Each wave instruction fills 64 consecutive 16-byte LDS slots; the
//     bank-conflict swizzles are applied by choosing which global chunk each lane loads.
//   * A rows (128 bytes per stage): chunk c of row r at position c ^ ((r/2) % 8), so the 16 rows of
//     one ds_read_b128 fragment read fall on distinct banks.
//   * W rows stay row-major: 64-byte rows keep chunk c of row r at c ^ ((r/2) % 4) ^ ((r/16) % 2).  The
//     first term spreads the 8 rows one 16-lane group reads over 32 banks; the second gives the group of
//     the next 16 rows the other 32 (measured: no LDS bank conflicts left).  B fragments are read with
//     ds_read_b64_tr_b8, which transposes bytes within each 16-lane group: result lane j, byte i = byte
//     (j % 8) of the 8 bytes addressed by lane 2i + j/8.  Lane x addresses k-row (x/2) at byte offset
//     8*(x%2) of its 16-byte-column group, so lane q receives byte-column q of 8 consecutive k-rows; two
//     reads give the 16 k-rows of its MFMA B operand, with no VALU transpose and no transposed stores.
//   * every LDS fragment read is inline assembly, so the only LDS waits are the explicit ones;
//   * the fragments of the next MFMA k-step are read while the MFMAs of the current one run
//     (two register sets, alternating);
//   * the stage barrier (stage s+1 landed everywhere, stage s free for reuse) and the DMA issue of
//     stage s+NS happen before the last k-step's MFMAs of stage s, and the first fragments of
//     stage s+1 are read right after it, so the MFMA pipe never waits for a fresh stage's reads.
// ------------------------------------------------------------------------------------------------
template <int MT, int GT>
struct PipeFrag {
    v4i a[MT];
    uint64_t lo[GT], hi[GT];
};

template <int BM, int WGN, int NS, int BK, int NWV, int BNB, bool TILED, int GM = 4>
__global__ __launch_bounds__(64 * NWV) __attribute__((amdgpu_waves_per_eu(2)))
void gemm_pipe16_kernel(const int8_t* __restrict__ A, const uint8_t* __restrict__ B, int32_t* __restrict__ C, int M,
                      int K, int N, int tiles_n, int k_begin, int k_end, int accumulate, int vec_store,
                      int k_split, OutScale os, int group_m) {
    if (gridDim.y > 1) {  // split-K: this workgroup's k-range, partial tile in slab blockIdx.y
        k_begin += (int)blockIdx.y * k_split;
        k_end = min(k_end, k_begin + k_split);
        C += (size_t)blockIdx.y * (size_t)M * (size_t)N;
    }
    constexpr int THR = 64 * NWV;           // threads per workgroup
    constexpr int CW = BNB / 16;            // 16-byte chunks per W stage row
    constexpr int WGM = NWV / WGN;
    constexpr int WM = BM / WGM;
    constexpr int MT = WM / 16;
    constexpr int GT = CW / WGN;
    constexpr int KS = BK / 64;
    constexpr int CPR = BK / 16;
    constexpr int A_STAGE = BM * BK;
    constexpr int W_STAGE = BK * BNB;
    constexpr int NA = A_STAGE / 16 / THR;
    constexpr int NW = W_STAGE / 16 / THR;
    static_assert(KS % 2 == 0, "fragment sets alternate per k-step");
    static_assert(NA >= 1 && NW >= 1 && GT >= 1, "tile too small for the workgroup");
    __shared__ __attribute__((aligned(16))) int8_t sA0[A_STAGE];
    __shared__ __attribute__((aligned(16))) int8_t sA1[A_STAGE];
    __shared__ __attribute__((aligned(16))) int8_t sA2[A_STAGE];
    __shared__ __attribute__((aligned(16))) int8_t sA3[NS > 3 ? A_STAGE : 16];
    __shared__ __attribute__((aligned(16))) uint8_t sW0[W_STAGE];
    __shared__ __attribute__((aligned(16))) uint8_t sW1[W_STAGE];
    __shared__ __attribute__((aligned(16))) uint8_t sW2[W_STAGE];
    __shared__ __attribute__((aligned(16))) uint8_t sW3[NS > 3 ? W_STAGE : 16];
    auto stage_a = [&](int i) -> int8_t* { return i == 0 ? sA0 : (i == 1 ? sA1 : (i == 2 ? sA2 : sA3)); };
    auto stage_w = [&](int i) -> uint8_t* { return i == 0 ? sW0 : (i == 1 ? sW1 : (i == 2 ? sW2 : sW3)); };

    const int NB = N >> 2;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WGN, wn = wave % WGN;
    const int q = lane & 15, kb = lane >> 4;

    const int tiles_m = (M + BM - 1) / BM;
    int tm, tn;
    {
        const int t = xcd_linear(blockIdx.x, gridDim.x);
        const int G_M = group_m > 0 ? group_m : GM;  // row tiles per group of the tile order
        const int first_m = (t / (G_M * tiles_n)) * G_M;
        const int gm = min(tiles_m - first_m, G_M);
        const int local = t % (G_M * tiles_n);
        tm = first_m + local % gm;
        tn = local / gm;
    }
    const int row0 = tm * BM;
    const int bc0 = tn * BNB;
    const int nst = (k_end - k_begin) / BK;

    uint32_t a_off[NA];
#pragma unroll
    for (int p = 0; p < NA; ++p) {
        const int slot = (p * NWV + wave) * 64 + lane;
        const int r = slot / CPR, pos = slot % CPR;
        const int grow = min(row0 + r, M - 1);
        a_off[p] = (uint32_t)grow * (uint32_t)K + (uint32_t)(((pos & ~7) | ((pos & 7) ^ gf_swz_a(r))) * 16);
    }
    uint32_t w_off[NW];
#pragma unroll
    for (int p = 0; p < NW; ++p) {
        const int slot = (p * NWV + wave) * 64 + lane;
        const int r = slot / CW, pos = slot % CW;
        w_off[p] = TILED ? tile64_offset((bc0 >> 4) + (pos ^ swz_w<BNB>(r)), r, K >> 6)
                         : (uint32_t)r * (uint32_t)NB + (uint32_t)(bc0 + (pos ^ swz_w<BNB>(r)) * 16);
    }
    auto issue = [&](int st, int buf) {
        const int sc = min(st, nst - 1);
        const int8_t* abase = A + k_begin + (size_t)sc * BK;
        int8_t* adst = stage_a(buf);
#pragma unroll
        for (int p = 0; p < NA; ++p) lds_dma16(abase + a_off[p], adst + (p * NWV + wave) * 1024);
        const uint8_t* wbase = TILED ? B + (size_t)((k_begin + sc * BK) >> 6) * 1024
                                     : B + (size_t)(k_begin + sc * BK) * (size_t)NB;
        uint8_t* wdst = stage_w(buf);
#pragma unroll
        for (int p = 0; p < NW; ++p) lds_dma16(wbase + w_off[p], wdst + (p * NWV + wave) * 1024);
    };

    // Per-lane fragment offsets inside a stage.  A: row wm*WM + 16t + q, chunk kk*4 + kb (the swizzle
    // depends on the row only through (row/2) % 8, the same for all t).  W: k-row 64kk + 16kb + q/2
    // (+8 for the second read), 16-byte group wn*GT + g (swizzle through (row/2) % 4, the same for all
    // kk and for the +8 row).
    uint32_t a_lane[KS];
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) {
        const int r = wm * WM + q;
        const int c = kk * 4 + kb;
        a_lane[kk] = (uint32_t)(r * BK + 16 * ((c & ~7) | ((c & 7) ^ gf_swz_a(r))));
    }
    uint32_t w_lane[GT];
#pragma unroll
    for (int g = 0; g < GT; ++g) {
        const int cg = wn * GT + g;
        const int r0 = kb * 16 + (q >> 1);
        w_lane[g] = (uint32_t)(r0 * BNB + 16 * (cg ^ swz_w<BNB>(r0)) + 8 * (q & 1));
    }
    auto read = [&](PipeFrag<MT, GT>& f, int buf, int kk) {
        const uint32_t ab = lds_u32(stage_a(buf)) + a_lane[kk];
#pragma unroll
        for (int t = 0; t < MT; ++t) f.a[t] = lds_read_b128_asm(ab + (uint32_t)(t * 16 * BK));
        const uint32_t wb = lds_u32(stage_w(buf)) + (uint32_t)(kk * 64 * BNB);
#pragma unroll
        for (int g = 0; g < GT; ++g) {
            f.lo[g] = lds_read_tr8_asm(wb + w_lane[g]);
            f.hi[g] = lds_read_tr8_asm(wb + w_lane[g] + 8 * BNB);
        }
    };
    // All LDS reads issued so far have returned; the empty asm statements tie each fragment register
    // to that point, so no use of them is scheduled before it.
    auto wait_frag = [&](PipeFrag<MT, GT>& f) {
        TX_LGKMCNT0();
#pragma unroll
        for (int t = 0; t < MT; ++t) __asm__ volatile("" : "+v"(f.a[t]));
#pragma unroll
        for (int g = 0; g < GT; ++g) __asm__ volatile("" : "+v"(f.lo[g]), "+v"(f.hi[g]));
    };

    v4i acc[MT][GT][4];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int g = 0; g < GT; ++g)
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[t][g][j] = v4i{0, 0, 0, 0};

    auto mfmas = [&](const PipeFrag<MT, GT>& f) {
#pragma unroll
        for (int g = 0; g < GT; ++g) {
            const uint32_t x4[4] = {(uint32_t)f.lo[g], (uint32_t)(f.lo[g] >> 32), (uint32_t)f.hi[g],
                                    (uint32_t)(f.hi[g] >> 32)};
            v4i bfr[4];
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4) {
                const uint32_t x = x4[r4];
                bfr[0][r4] = (int)((x << 6) & 0xC0C0C0C0u);
                bfr[1][r4] = (int)((x << 4) & 0xC0C0C0C0u);
                bfr[2][r4] = (int)((x << 2) & 0xC0C0C0C0u);
                bfr[3][r4] = (int)(x & 0xC0C0C0C0u);
            }
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[t][g][j] = mfma_i8(f.a[t], bfr[j], acc[t][g][j]);
        }
    };

    PipeFrag<MT, GT> f0, f1;
    // Prologue: all NS stages in flight, wait for stage 0, first fragments.
#pragma unroll
    for (int p = 0; p < NS; ++p) issue(p, p);
    TX_VMCNT((NS - 1) * (NA + NW));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    read(f0, 0, 0);

    // One stage in buffer h (a literal at every call site).  Fragment set f0 serves even k-steps.
    auto stage = [&](int st, int h) {
#pragma unroll
        for (int kk = 0; kk < KS; ++kk) {
            PipeFrag<MT, GT>& cur = (kk & 1) ? f1 : f0;
            PipeFrag<MT, GT>& nxt = (kk & 1) ? f0 : f1;
            wait_frag(cur);
            __builtin_amdgcn_sched_barrier(0);
            if (kk + 1 < KS) {
                read(nxt, h, kk + 1);
            } else if (st + 1 < nst) {
                TX_VMCNT((NS - 2) * (NA + NW));  // stage st+1 has landed (NS-2 later stages may not)
                __builtin_amdgcn_s_barrier();     // ... everywhere, and every wave is done reading stage st
                __builtin_amdgcn_sched_barrier(0);
                issue(st + NS, h);
                read(nxt, (h + 1) % NS, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            mfmas(cur);
            // keep the next k-step's wait below these MFMAs (it would otherwise be hoisted among them
            // and wait for the reads just issued)
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    int s = 0;
    for (; s + NS <= nst; s += NS) {
        stage(s + 0, 0);
        stage(s + 1, 1);
        stage(s + 2, 2);
        if (NS > 3) stage(s + 3, 3);
    }
    if (s + 0 < nst) stage(s + 0, 0);
    if (s + 1 < nst) stage(s + 1, 1);
    if (NS > 3 && s + 2 < nst) stage(s + 2, 2);
    float fs[MT][4];  // the float epilogue's row scales, all in flight at once
    if (os.Y) {
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) fs[t][i] = os.rs[min(row0 + wm * WM + t * 16 + 4 * kb + i, M - 1)];
    }
    TX_VMCNT(0);  // no LDS DMA may land after the workgroup exits

#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int row = row0 + wm * WM + t * 16 + 4 * kb + i;
            if (row >= M) continue;
#pragma unroll
            for (int g = 0; g < GT; ++g) {
                const int bcol = bc0 + (wn * GT + g) * 16 + q;
                v4i v = {acc[t][g][0][i] >> 6, acc[t][g][1][i] >> 6, acc[t][g][2][i] >> 6, acc[t][g][3][i] >> 6};
                if (os.Y) {  // dequantised float output: y = c * (row_scale[row] * w_scale)
                    store_scaled_f(os, fs[t][i] * os.ws, row, N, 4 * bcol, v, vec_store);
                    continue;
                }
                int32_t* out = C + (size_t)row * (size_t)N + 4 * bcol;
                if (vec_store) {
                    if (accumulate) v += *reinterpret_cast<const v4i*>(out);
                    __builtin_nontemporal_store(v, reinterpret_cast<v4i*>(out));  // streamed, not re-read
                } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j) out[j] = accumulate ? out[j] + v[j] : v[j];
                }
            }
        }
}

// ------------------------------------------------------------------------------------------------
// GEMM on v_mfma_i32_32x32x32_i8 (K % 16 == 0, K >= BK, NB % 16 == 0, aligned A and W; output columns n_out <= N).
//
// A workgroup is WGM x WGN x WGK waves; a wave computes 32*MT rows x 32 byte-columns (128 outputs), MT x 4
// accumulators of 32x32, over its share of every stage's k-rows.  What bounds it, on MI355X:
//   * Prefill (every CU full): power.  The clock falls to 1.85-2.15 GHz with the MFMA pipes 79 % busy; from
//     registers alone 32x32x32 sustains 4.34 POPS, 16x16x64 3.9.  So the tile spends little energy beside the
//     MFMAs: it is wide in N, since a packed weight byte is four columns (64 x 128 outputs read 64 + 32 bytes of
//     LDS per k-row where a 64 x 64 tile reads 64 + 16 for half the work).
//   * Fewer tiles than CUs: issue.  One wave per SIMD ran at 61 % (decode 17 %, DMA 14 %, barriers 11 %), so the
//     smaller tiles split each stage's k-steps over WGK waves, which sum their tiles through LDS at the end:
//     no partial sums in memory, no second launch, and two or more waves on every SIMD.
// Each MFMA is followed by a share of the other work, so that the pipe always has the next one: half a field of
// the next decode, two of the next k-step's LDS reads (first MFMAs), one or two of the stage's DMAs (its last
// k-step).  DMAs in one burst after the barrier cost 6 % (1024x6912x2560 24.0 -> 22.0 us).
// us before -> after, L2-warm weights: 128x4096x4096 19.3 -> 9.5, 256x4096x11008 20.7 -> 16.7, 1024x6912x2560 31.4 ->
// 22.1, 1024x2560x13824 41 -> 34.5, 2048x4096x14336 126 -> 111 (the card at its slowest; 103 -> 98 otherwise).
// RG: ragged operands (any K >= BK, NB >= BNB, any addresses) read in place.  Every 16-byte chunk lies inside its row,
// since the last stage ends at k_end and the last column tile at NB (both overlap their neighbour; columns done
// twice store the same values), so chunks go through registers with one unaligned load each, no edge cases, and
// from there to the same LDS slots: two stages in LDS, the next two in registers.  Rows of W already done are
// zeroed on the way instead of masked.
// LDS layouts (no bank conflicts): A chunk c of row r at c ^ ((r/2) % 8) for 128-byte rows, c ^ (r % 16) for
// 256-byte ones; W's 32-byte column pairs p of row r at p ^ f(r), f the row bits that make 8 rows of one pair
// cover all 64 banks.  W fragments come from ds_read_b64_tr_b8 (see below): 16-lane groups 0-1 take the two
// halves of a pair for k-rows 0-15, groups 2-3 for rows 16-31, as the MFMA's lanes want them.
// ------------------------------------------------------------------------------------------------
typedef int v16i __attribute__((ext_vector_type(16)));

template <int BK>
__device__ __forceinline__ int gw_swz_a(int r) { return BK == 128 ? ((r >> 1) & 7) : (r & 15); }
template <int BNB>
__device__ __forceinline__ int gw_swz_w(int r) {
    return BNB == 128 ? 2 * ((r >> 1) & 3) : (BNB == 64 ? 2 * ((r >> 2) & 1) : 0);
}

template <int OFF>
__device__ __forceinline__ v4i lds_read_b128_off(uint32_t addr) {
    v4i v;
    __asm__ volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF));
    return v;
}
template <int OFF>
__device__ __forceinline__ uint64_t lds_read_tr8_off(uint32_t addr) {
    uint64_t v;
    __asm__ volatile("ds_read_b64_tr_b8 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF));
    return v;
}

template <int V>
using Int = std::integral_constant<int, V>;

template <int MT>
struct WideFrag {
    v4i a[MT];
    uint64_t lo, hi;
};

template <int WGM, int WGN, int WGK, int MT, int BK, int NS, bool TILED, int GM, bool RG>
__global__ __launch_bounds__(64 * WGM * WGN * WGK) __attribute__((amdgpu_waves_per_eu(2)))
void gemm_pipe_kernel(const int8_t* __restrict__ A, const uint8_t* __restrict__ B, int32_t* __restrict__ C, int M,
                      int K, int N, int n_out, int tiles_n, int k_begin, int k_end, int accumulate, int vec_store,
                      int k_split, OutScale os, int group_m) {
    if (gridDim.y > 1) {  // split-K: this workgroup's k-range, partial tile in slab blockIdx.y
        k_begin += (int)blockIdx.y * k_split;
        k_end = min(k_end, k_begin + k_split);
        C += (size_t)blockIdx.y * (size_t)M * (size_t)n_out;
    }
    constexpr int NWV = WGM * WGN * WGK;
    constexpr int THR = 64 * NWV;
    constexpr int BM = 32 * MT * WGM;
    constexpr int BNB = 32 * WGN;
    constexpr int CW = BNB / 16;           // 16-byte chunks per W stage row
    constexpr int CPR = BK / 16;           // and per A stage row
    constexpr int KS = BK / 32 / WGK;      // 32-row k-steps per wave and stage
    constexpr int A_STAGE = BM * BK;
    constexpr int W_STAGE = BK * BNB;
    constexpr int STAGE = A_STAGE + W_STAGE;
    constexpr int NA = A_STAGE / 16 / THR;
    constexpr int NW = W_STAGE / 16 / THR;
    constexpr int RED = WGK == 1 ? 0 : NWV * (WGK - 1) * (16 / WGK) * 1024;  // bytes of the final exchange
    constexpr int LDS = NS * STAGE > RED ? NS * STAGE : RED;
    static_assert(KS == 2 || KS == 4, "fragment sets alternate per k-step");
    static_assert(NA >= 1 && NW >= 1 && A_STAGE % (16 * THR) == 0 && W_STAGE % (16 * THR) == 0, "uneven stage");
    static_assert(LDS <= 160 * 1024, "LDS");
    __shared__ __attribute__((aligned(256))) uint8_t smem[LDS];

    const int NB = N >> 2;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wk = wave / (WGM * WGN), wmn = wave % (WGM * WGN);
    const int wm = wmn / WGN, wn = wmn % WGN;
    const int r32 = lane & 31, half = lane >> 5, q = lane & 15;

    const int tiles_m = (M + BM - 1) / BM;
    int tm, tn;
    {
        const int t = xcd_linear(blockIdx.x, gridDim.x);
        const int G_M = group_m > 0 ? group_m : GM;  // row tiles per group of the tile order
        const int first_m = (t / (G_M * tiles_n)) * G_M;
        const int gm = min(tiles_m - first_m, G_M);
        const int local = t % (G_M * tiles_n);
        tm = first_m + local % gm;
        tn = local / gm;
    }
    const int row0 = tm * BM;
    const int bc0 = RG ? min(tn * BNB, NB - BNB) : tn * BNB;
    // Stages of BK k-rows; the last one ends at k_end, so where BK does not divide the range it starts inside
    // the stage before, and the rows that one has done are masked out of its weights.
    const int klen = k_end - k_begin;
    const int nst = (klen + BK - 1) / BK;
    const int done = nst * BK - klen;  // k-rows of the last stage that the stage before it has done

    uint32_t a_off[NA];
#pragma unroll
    for (int p = 0; p < NA; ++p) {
        const int slot = (p * NWV + wave) * 64 + lane;
        const int r = slot / CPR, pos = slot % CPR;
        const int grow = min(row0 + r, M - 1);  // rows past M load row M-1; never stored
        a_off[p] = (uint32_t)grow * (uint32_t)K + (uint32_t)((pos ^ gw_swz_a<BK>(r)) * 16);
    }
    uint32_t w_off[NW];
#pragma unroll
    for (int p = 0; p < NW; ++p) {
        const int slot = (p * NWV + wave) * 64 + lane;
        const int r = slot / CW, pos = slot % CW;
        const int c = min((bc0 >> 4) + (pos ^ gw_swz_w<BNB>(r)), (NB >> 4) - 1);  // columns past N: never stored
        if (RG) w_off[p] = (uint32_t)r * (uint32_t)NB + (uint32_t)(bc0 + (pos ^ gw_swz_w<BNB>(r)) * 16);
        else w_off[p] = TILED ? tile64_offset(c, r, K >> 6) : (uint32_t)r * (uint32_t)NB + (uint32_t)(c * 16);
    }
    // DMA instruction d of stage st (A's NA, then W's NW) into the stage buffer at byte `off`.
    // (Stages past the last one repeat it: the load count per stage stays static, and a branch around the
    // loads cost more than the repeats.)
    auto issue = [&](int st, int off, int d) {
        const int k0 = k_begin + min(st * BK, klen - BK);
        if (d < NA) {
            lds_dma16(A + k0 + a_off[d < NA ? d : 0], smem + off + (d * NWV + wave) * 1024);
        } else {
            const int p = d - NA;
            const uint8_t* wbase = TILED ? B + (size_t)(k0 >> 6) * 1024 : B + (size_t)k0 * (size_t)NB;
            lds_dma16(wbase + w_off[p < 0 ? 0 : p], smem + off + A_STAGE + (p * NWV + wave) * 1024);
        }
    };

    // Ragged operands (RG): chunk d of stage st through a register, and from there into the stage buffer.
    auto gload = [&](int st, int d) -> v4i {
        const int k0 = k_begin + min(st * BK, klen - BK);
        const void* src = d < NA ? (const void*)(A + k0 + a_off[d < NA ? d : 0])
                                 : (const void*)(B + (size_t)k0 * (size_t)NB + w_off[d < NA ? 0 : d - NA]);
        v4i v;
        __builtin_memcpy(&v, src, 16);  // any alignment
        return v;
    };
    auto swrite = [&](v4i v, int st, int off, int d) {
        const int slot = ((d < NA ? d : d - NA) * NWV + wave) * 64 + lane;
        if (d >= NA && st == nst - 1 && slot / CW < done) v = v4i{0, 0, 0, 0};  // a k-row the stage before has done
        lds_write_b128_asm(lds_u32(smem) + (uint32_t)(off + (d < NA ? 0 : A_STAGE) + slot * 16), v);
    };

    uint32_t a_lane[KS];
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) {
        const int r = wm * MT * 32 + r32;
        const int c = (wk * KS + kk) * 2 + half;
        a_lane[kk] = lds_u32(smem) + (uint32_t)(r * BK + 16 * (c ^ gw_swz_a<BK>(r)));
    }
    const uint32_t w_lane = lds_u32(smem) + (uint32_t)(((wk * KS * 32) + half * 16 + (q >> 1)) * BNB +
                                       16 * ((2 * wn + ((lane >> 4) & 1)) ^ gw_swz_w<BNB>(q >> 1)) + 8 * (q & 1));
    // Read r (0, 1: the weights' halves; 2 ..: m-tile r - 2) of k-step KK of the stage at byte `off`.
    auto read = [&](auto kc, WideFrag<MT>& f, uint32_t off, int r) {
        constexpr int KK = decltype(kc)::value;
        if (r == 0) f.lo = lds_read_tr8_off<A_STAGE + KK * 32 * BNB>(w_lane + off);
        if (r == 1) f.hi = lds_read_tr8_off<A_STAGE + KK * 32 * BNB + 8 * BNB>(w_lane + off);
        if (r == 2) f.a[0] = lds_read_b128_off<0>(a_lane[KK] + off);
        if constexpr (MT > 1)
            if (r == 3) f.a[1] = lds_read_b128_off<32 * BK>(a_lane[KK] + off);
    };
    // The reads still outstanding may be the MT youngest (the activations); tie the registers to the wait.
    auto wait_w = [&](WideFrag<MT>& f) {
        __builtin_amdgcn_s_waitcnt(0xF | (3 << 14) | (7 << 4) | (MT << 8));
        __asm__ volatile("" : "+v"(f.lo), "+v"(f.hi));
    };
    auto wait_a = [&](WideFrag<MT>& f) {
        TX_LGKMCNT0();
#pragma unroll
        for (int t = 0; t < MT; ++t) __asm__ volatile("" : "+v"(f.a[t]));
    };

    v16i acc[MT][4];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[t][j][i] = 0;

    // Field mask of each k-step: all fields, or none in the last stage's steps that are already done (a lane
    // holds 16 consecutive k-rows of a step, and every k-range is a multiple of 16 rows).
    auto field_mask = [&](bool last, int kk) -> uint32_t {
        return !RG && last && (wk * KS + kk) * 32 + half * 16 < done ? 0u : 0xC0C0C0C0u;
    };
    uint32_t mask[KS];
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) mask[kk] = field_mask(nst == 1, kk);
    v4i b0, b1;                         // decoded fields: one feeds the MFMAs while the next one is made
    auto decode = [&](v4i& b, const WideFrag<MT>& f, int j, int r4, uint32_t m) {
        const uint32_t x = r4 == 0 ? (uint32_t)f.lo : (r4 == 1 ? (uint32_t)(f.lo >> 32)
                                                               : (r4 == 2 ? (uint32_t)f.hi : (uint32_t)(f.hi >> 32)));
        b[r4] = (int)((j == 3 ? x : x << (6 - 2 * j)) & m);
    };
    constexpr int D = NA + NW;      // DMA instructions per stage
    constexpr int SLOTS = 4 * MT;   // MFMAs per k-step
    constexpr int R = 2 + MT;       // LDS reads per k-step

    WideFrag<MT> f0, f1;
    v4i ga[RG ? D : 1], gb[RG ? D : 1];  // RG: the chunks of stages st + 2 (even st: ga) and st + 3
    if constexpr (RG) {
        static_assert(NS == 2 && !TILED, "two stage buffers, two stages in registers");
#pragma unroll
        for (int d = 0; d < D; ++d) ga[d] = gload(0, d);
#pragma unroll
        for (int d = 0; d < D; ++d) gb[d] = gload(1, d);
#pragma unroll
        for (int d = 0; d < D; ++d) {
            swrite(ga[d], 0, 0, d);
            ga[d] = gload(2, d);
        }
#pragma unroll
        for (int d = 0; d < D; ++d) {
            swrite(gb[d], 1, STAGE, d);
            gb[d] = gload(3, d);
        }
        TX_LGKMCNT0();
    } else {
#pragma unroll
        for (int p = 0; p < NS; ++p)
#pragma unroll
            for (int d = 0; d < D; ++d) issue(p, p * STAGE, d);
        TX_VMCNT((NS - 1) * D);
    }
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < R; ++r) read(Int<0>{}, f0, 0, r);
    wait_w(f0);
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) decode(b0, f0, 0, r4, mask[0]);
    wait_a(f0);

    // One 32-row k-step: SLOTS MFMAs, each followed by a share of the next field's decode, of the next
    // k-step's LDS reads (first half) and, in a stage's last k-step, of the DMAs of stage st + NS.
    auto step = [&](auto kc, WideFrag<MT>& cur, WideFrag<MT>& nxt, int st, uint32_t off, uint32_t noff, v4i* g) {
        constexpr int KK = decltype(kc)::value;
        constexpr bool LAST = KK + 1 == KS;
        if constexpr (LAST) {
            // stage st + 1 has landed (the NS - 2 later ones may not)
            if constexpr (!RG) TX_VMCNT((NS - 2) * D);
            __builtin_amdgcn_s_barrier();  // ... everywhere, and every wave is done reading stage st
        }
        if (LAST && done > 0 && st + 2 == nst) {
#pragma unroll
            for (int kk = 0; kk + 1 < KS; ++kk) mask[kk] = field_mask(true, kk);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < SLOTS; ++s) {
            const int j = s / MT, t = s % MT;
            v4i& b = (j & 1) ? b1 : b0;
            v4i& bn = (j & 1) ? b0 : b1;
            acc[t][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(cur.a[t], b, acc[t][j], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            if (s == 3 * MT) wait_w(nxt);
#pragma unroll
            for (int r4 = t * 4 / MT; r4 < (t + 1) * 4 / MT; ++r4)
                decode(bn, j == 3 ? nxt : cur, (j + 1) & 3, r4, mask[j == 3 ? (KK + 1) % KS : KK]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (r / 2 == s) read(Int<(KK + 1) % KS>{}, nxt, LAST ? noff : off, r);
            if constexpr (LAST) {
#pragma unroll
                for (int d = 0; d < D; ++d)
                    if (d * SLOTS / D == s) {
                        if constexpr (RG) {
                            swrite(g[d], st + 2, (int)off, d);
                            g[d] = gload(st + 4, d);
                        } else {
                            issue(st + NS, (int)off, d);
                        }
                    }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        wait_a(nxt);
        if (LAST && done > 0 && st + 2 == nst) mask[KS - 1] = field_mask(true, KS - 1);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto stage = [&](int st, uint32_t off, uint32_t noff, v4i* g) {
        step(Int<0>{}, f0, f1, st, off, noff, g);
        step(Int<1>{}, f1, f0, st, off, noff, g);
        if constexpr (KS == 4) {
            step(Int<2>{}, f0, f1, st, off, noff, g);
            step(Int<3>{}, f1, f0, st, off, noff, g);
        }
    };
    if constexpr (RG) {
        for (int st = 0; st < nst; st += 2) {
            stage(st, 0, STAGE, ga);
            if (st + 1 < nst) stage(st + 1, STAGE, 0, gb);
        }
    } else {
        uint32_t off = 0;
        for (int st = 0; st < nst; ++st) {
            const uint32_t noff = off + STAGE == (uint32_t)(NS * STAGE) ? 0u : off + STAGE;
            stage(st, off, noff, ga);
            off = noff;
        }
    }
    // The float epilogue's row scales, all in flight at once (loaded one by one between the stores they cost a
    // memory latency per row: dequantising 1024x2560x13824 38.3 us against 34 for int32).
    float fs[MT][16];
    if (os.Y) {
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i)
                fs[t][i] = os.rs[min(row0 + (wm * MT + t) * 32 + 8 * (i >> 2) + 4 * half + (i & 3), M - 1)];
    }
    TX_VMCNT(0);  // no LDS DMA may land after the workgroup exits

    // Element i of accumulator (t, j) is row 8*(i/4) + 4*half + i%4 of m-tile t, column 4*r32 + j.
    auto store = [&](int t, int i, v4i v) {
        const int row = row0 + (wm * MT + t) * 32 + 8 * (i >> 2) + 4 * half + (i & 3);
        const int bcol = bc0 + wn * 32 + r32;
        if (row >= M || bcol >= (n_out >> 2)) return;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] >>= 6;
        if (os.Y) {  // dequantised float output: y = c * (row_scale[row] * w_scale)
            store_scaled_f(os, fs[t][i] * os.ws, row, n_out, 4 * bcol, v, vec_store);
            return;
        }
        int32_t* out = C + (size_t)row * (size_t)n_out + 4 * bcol;
        if (vec_store) {
            if (accumulate) v += *reinterpret_cast<const v4i*>(out);
            __builtin_nontemporal_store(v, reinterpret_cast<v4i*>(out));  // streamed, not re-read
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) out[j] = accumulate ? out[j] + v[j] : v[j];
        }
    };
    if constexpr (WGK == 1) {
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) store(t, i, v4i{acc[t][0][i], acc[t][1][i], acc[t][2][i], acc[t][3][i]});
    } else {
        // Each of the WGK waves of one output tile finishes 1/WGK of its elements: per m-tile it leaves the
        // other shares in LDS for their owners and adds what they left for it.
        constexpr int SH = 16 / WGK;  // elements i per share and m-tile
        v4i* ex = reinterpret_cast<v4i*>(smem);  // [wmn][owner][sender slot][SH][64 lanes]
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            __syncthreads();
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int owner = i / SH;
                const int slot = (wk - owner + WGK) % WGK - 1;  // 0 .. WGK-2 for the other waves
                if (owner != wk)
                    ex[(((wmn * WGK + owner) * (WGK - 1) + slot) * SH + i % SH) * 64 + lane] =
                        v4i{acc[t][0][i], acc[t][1][i], acc[t][2][i], acc[t][3][i]};
            }
            __syncthreads();
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int owner = i / SH;
                if (owner != wk) continue;
                v4i v = {acc[t][0][i], acc[t][1][i], acc[t][2][i], acc[t][3][i]};
#pragma unroll
                for (int sl = 0; sl < WGK - 1; ++sl)
                    v += ex[(((wmn * WGK + owner) * (WGK - 1) + sl) * SH + i % SH) * 64 + lane];
                store(t, i, v);
            }
        }
    }
}

// Tile shapes of gemm_pipe_kernel and what they cost (gemm_plan).  us per 256 k-rows of a round: t1 with one
// workgroup on every CU, t2 with per_cu of them; one_cu of t1 on an idle chip; second of the way to t2 where
// the first CUs get a second workgroup.  fixed + a round's start and stores.
struct WideTile {
    int rows, bnb, bk, per_cu;
    float t1, t2, fixed, round, second, one_cu;
};
// Fitted to 5800 timings of 228 shapes (M 33-2048, K 512-16384, N 768-16384, 1-16 splits; root mean square error
// 7 %); the plans it picks are within 1 % of the fastest of these tiles on average.
constexpr WideTile kWide[kWideTiles] = {
    {32, 32, 256, 2, 0.455f, 0.872f, 1.96f, 2.57f, 0.674f, 0.60f},   // 0: 32 x 128, K over 4 waves
    {32, 64, 256, 2, 0.550f, 1.31f, 0.00f, 4.88f, 0.862f, 0.681f},   // 1: 32 x 256, K over 4 of 8 waves
    {64, 64, 256, 1, 0.708f, 0.811f, 2.36f, 4.66f, 1.0f, 0.672f},    // 2: 64 x 256, K over 4 of 8 waves
    {64, 128, 128, 1, 1.34f, 1.60f, 1.89f, 4.65f, 1.0f, 0.698f},     // 3: 64 x 512, K over 2 of 8 waves
    {64, 128, 128, 2, 1.56f, 3.25f, 2.02f, 4.23f, 0.409f, 0.736f},   // 4: 64 x 512, 4 waves, two workgroups per CU
    {64, 64, 128, 2, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f},            // 5: 64 x 256, K over 2 of 4 waves (split plans)
    {128, 64, 128, 1, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f},           // 6: 128 x 256, K over 2 of 8 waves (split plans)
};
// The 64 x 256 tiles of gemm_pipe16_kernel, on the same scale.
constexpr WideTile kPipe64Cost = {64, 64, 128, 2, 1.08f, 1.76f, 0.001f, 4.75f, 0.225f, 0.732f};

template <int WGM, int WGN, int WGK, int MT, int BK, int NS, int GM, bool RG = false>
hipError_t launch_wide(const int8_t* A, const uint8_t* B, int32_t* C, int M, int K, int N, int n_out, int kb, int ke,
                       int acc, int vs, hipStream_t st, const OutScale& os, int splits, int k_split, int tiled,
                       int gm_env) {
    constexpr int BM = 32 * MT * WGM, BNB = 32 * WGN;
    const int tiles_n = (N / 4 + BNB - 1) / BNB;
    const dim3 grid((unsigned)(((M + BM - 1) / BM) * tiles_n), splits), block(64 * WGM * WGN * WGK);
    if constexpr (!RG) {
        if (tiled) {
            hipLaunchKernelGGL((gemm_pipe_kernel<WGM, WGN, WGK, MT, BK, NS, true, GM, false>), grid, block, 0, st, A, B, C, M, K,
                               N, n_out, tiles_n, kb, ke, acc, vs, k_split, os, gm_env);
            return hipGetLastError();
        }
    }
    hipLaunchKernelGGL((gemm_pipe_kernel<WGM, WGN, WGK, MT, BK, NS, false, GM, RG>), grid, block, 0, st, A, B, C, M, K, N,
                       n_out, tiles_n, kb, ke, acc, vs, k_split, os, gm_env);
    return hipGetLastError();
}

template <int BM, int BNB>
hipError_t launch_gemm_t(const int8_t* A, const uint8_t* B, int32_t* C, int M, int K, int N, bool aw, bool aa,
                         int kb, int ke, int acc, hipStream_t st, const OutScale& os, int splits, int k_split) {
    const int NB = N >> 2;
    const int tiles_m = (M + BM - 1) / BM, tiles_n = (NB + BNB - 1) / BNB;
    const dim3 grid(tiles_m * tiles_n, splits), block(GM_THREADS);
    const int vs = ((uintptr_t)(os.Y ? (const void*)os.Y : (const void*)C) % 16) == 0;
    if (aw && aa)
        hipLaunchKernelGGL((gemm_kernel<BM, BNB, true, true>), grid, block, 0, st, A, B, C, M, K, N, tiles_n, kb, ke, acc, vs, k_split, os);
    else if (aw)
        hipLaunchKernelGGL((gemm_kernel<BM, BNB, true, false>), grid, block, 0, st, A, B, C, M, K, N, tiles_n, kb, ke, acc, vs, k_split, os);
    else if (aa)
        hipLaunchKernelGGL((gemm_kernel<BM, BNB, false, true>), grid, block, 0, st, A, B, C, M, K, N, tiles_n, kb, ke, acc, vs, k_split, os);
    else
        hipLaunchKernelGGL((gemm_kernel<BM, BNB, false, false>), grid, block, 0, st, A, B, C, M, K, N, tiles_n, kb, ke, acc, vs, k_split, os);
    return hipGetLastError();
}

}  // namespace

// Narrow 64 x 64 tiles for M <= 64 when they alone fill at most one workgroup per CU (measured on
// MI355X: cfg3 M=64 up 18.0 -> 13.4 us with no K split, 4096^2 at M=64 16.2 -> 9.9 us; with more
// tiles than CUs, e.g. N = 28672, the 256-column tiles are faster).  The gemm_narrow debug switch (0 / 1) turns
// the choice off / on regardless (experiments).
bool gemm_narrow_wanted(int M, int K, int N, int tiled) {
    const int env = debug_get(DBG_GEMM_NARROW);
    const int NB = N >> 2;
    if (env == 0 || NB % 16 != 0 || K % 256 != 0) return false;
    if (env > 0) return true;
    // Row-major weights: not where K is split (K > 4096), where the 256-column tiles with more splits
    // win (on MI355X, cold, 64 / 256 columns: 64x11008x4096 14.4 / 13.1 us, 48x11008x4096 13.8 /
    // 11.9, 40x16384x4096 16.4 / 12.8, 64x16384x8192 30.1 / 21.4, 33x8192x4096 11.5 / 10.5).  The
    // tile-64 layout keeps them (its 1 KB blocks: 64x11008x4096 11.1 against 13.0 us).
    if (M > 64 || (K > 4096 && !tiled)) return false;
    return (long)((M + 63) / 64) * (NB / 16) <= device_cu_count();
}

// Tile height of a split-K launch: 64-row tiles of four waves or 128-row tiles of eight, each with
// the split count sized to one workgroup per CU (at most 16 splits of >= 256 k-rows).  The plan that
// keeps more CUs busy wins; on a tie the 64-row tiles win where they need no split at all on a full
// grid, the 128-row ones where each workgroup carries >= 80 M multiply-adds (their second wave per
// SIMD pays for the larger partials), else the 64-row ones.  On MI355X, cold weights, 64 / 128 rows:
// 128x11008x4096 15.4 / 19.3 us, 256x16384x4096 27.1 / 28.3, 256x8192x2048 14.4 / 19.3, 512x8192x2048
// 18.8 / 22.9 (ties, fewer multiply-adds); 512x11008x4096 33.2 / 32.1, 512x16384x4096 42.8 / 39.7,
// 768x16384x4096 64.1 / 55.1 (ties, more); 384x11008x4096 32.0 / 28.4 (192 against 240 workgroups);
// 1024x11008x4096 45.3 / 49.0 and 1024x16384x4096 65.1 / 62.4 (the 64-row tiles without a split).
int gemm_split_rows(int M, int K, int N) {
    const int bm_env = debug_get(DBG_GEMM_BM);
    if (bm_env == 64 || bm_env == 128) return bm_env;  // tests and measurements
    if (M % 128 != 0) return 64;  // no padding rows
    const long cus = device_cu_count();
    const long smax = std::min<long>(std::max(1, K / 256), 16);
    auto plan = [&](int rows, long* splits) {  // CUs busy in the plan's last wave of workgroups
        const long t = (long)((M + rows - 1) / rows) * (long)((N / 4 + 63) / 64);
        *splits = std::min<long>(t * 2 <= cus ? cus / t : 1, smax);
        const long wgs = t * *splits;
        return wgs % cus == 0 ? cus : wgs % cus;
    };
    long s64 = 1, s128 = 1;
    const long f64 = plan(64, &s64), f128 = plan(128, &s128);
    if (f128 != f64) return f128 > f64 ? 128 : 64;
    if (s64 == 1 && f64 == cus) return 64;
    const double macs = (double)M * (double)N * (double)K / (double)cus;
    return macs >= 80e6 ? 128 : 64;
}

namespace {

// Predicted us of one launch over `len` k-rows (and of the reduce launch with splits > 1).
double wide_cost(const WideTile& w, long M, long N, long len, long splits) {
    const long cus = device_cu_count(), slots = cus * w.per_cu;
    const long wgs = ((M + w.rows - 1) / w.rows) * ((N / 4 + w.bnb - 1) / w.bnb) * splits;
    const long full = wgs / slots, rem = wgs % slots;
    double last = 0.0;
    if (rem > cus) last = w.t1 + (w.t2 - w.t1) * (w.second + (1.0 - w.second) * (double)(rem - cus) / (double)cus);
    else if (rem > 0) last = w.t1 * (w.one_cu + (1.0 - w.one_cu) * (double)rem / (double)cus);
    double t = w.fixed + (double)(full + (rem > 0)) * w.round + (double)len / 256.0 * ((double)full * w.t2 + last);
    if (splits > 1) t += 2.5 + (0.787 * (double)splits + 0.621) * (double)M * (double)N * 1e-6;
    return t;
}

// K over `splits` ranges of whole 64-row blocks, none shorter than `least` rows; fewer where they do not fit.
void split_k(int K, long splits, int least, GemmPlan* p) {
    for (; splits > 1; --splits) {
        const int ks = (int)((K / splits + (K % splits != 0) + 63) / 64 * 64);
        const int n = (K + ks - 1) / ks;
        if (n > 1 && K - (n - 1) * ks >= least) {
            p->splits = n;
            p->k_split = ks;
            return;
        }
    }
    p->splits = 1;
    p->k_split = 0;
}

// Sizes the ragged tiles take: a whole stage, a whole tile of columns, 32-bit offsets.
bool ragged_ok(int M, int K, int N) {
    return M > 0 && K >= 256 && N / 4 >= 64 && (size_t)M * (size_t)K < ((size_t)1 << 32) &&
           (size_t)256 * (size_t)(N / 4) < ((size_t)1 << 32);
}

// The split count of the row-tile plan (gemm_split_rows): one workgroup per CU, at most 16 splits of >= 256 rows.
int row_tile_splits(int M, int K, int N, int bm, int col_tiles) {
    // K <= 4096: the reduce launch and the partial sums cost more than the idle CUs (measured on
    // MI355X, cold weights: 40x1024x4096 7.6 -> 4.9 us without the split, 64x2560x6912 11.8 -> 8.8,
    // 256x1024x11008 31.1 -> 9.7, 256x4096x11008 35.2 -> 25.0; from K = 6144 the split wins:
    // 128x11008x4096 59.0 -> 22.4 us).
    if (K <= 4096) return 1;
    const long tiles = (long)((M + bm - 1) / bm) * col_tiles, cus = device_cu_count();
    return (int)std::max<long>(1, std::min<long>({tiles * 2 <= cus ? cus / tiles : 1, (long)K / 256, 16L}));
}

}  // namespace

// Which kernel a GEMM call runs and how it splits K (the single place the choice is made).
GemmPlan gemm_plan(const int8_t* A, const uint8_t* B, int M, int K, int N, int tiled, bool may_split, bool padded) {
    GemmPlan p;
    const int NB = N >> 2;
    const bool aligned = (uintptr_t)A % 16 == 0 && (uintptr_t)B % 16 == 0 && (size_t)M * (size_t)K < ((size_t)1 << 32) &&
                         (size_t)512 * (size_t)NB < ((size_t)1 << 32) && M > 0;
    const bool force_generic = debug_get(DBG_GEMM_GENERIC) == 1;  // tests
    const bool pipe16 = aligned && !padded && K > 0 && K % 128 == 0 && NB % 64 == 0 && (tiled || !force_generic);
    const bool wide = aligned && K >= 128 && K % 16 == 0 && NB % 16 == 0 && (!tiled || K % 64 == 0) &&
                      (tiled || !force_generic);
    // The tile-64 layout is read by the LDS-DMA GEMMs only (whole 128-row stages, at most 4 GiB of W).
    if (tiled && (!pipe16 || (size_t)K * (size_t)NB >= ((size_t)1 << 32))) {
        p.choice = GemmChoice::Invalid;
        return p;
    }
    const int splits_env = debug_get(DBG_GEMM_SPLITS);  // tests
    auto forced = [&](long s) { return splits_env > 0 ? (long)splits_env : s; };
    const int tile_rg = debug_get(DBG_GEMM_BM, 1) - kWideTiles;  // tests and measurements
    if (tile_rg >= 0 && tile_rg < kRaggedTiles && !tiled && ragged_ok(M, K, N)) {
        p.choice = (GemmChoice)((int)GemmChoice::Ragged0 + tile_rg);
        if (may_split) split_k(K, forced(1), 256, &p);
        return p;
    }
    if (!pipe16 && !wide) {
        if (may_split) split_k(K, forced(row_tile_splits(M, K, N, gemm_split_rows(M, K, N), (NB + 63) / 64)), 64, &p);
        return p;  // Generic
    }
    // 64 x 64 output tiles (16 bytes of every weight row): enough workgroups without a K split where
    // the 256-column tiles would need one; one m-tile per wave, 256-deep stages.
    if (pipe16 && (M <= 64 || debug_get(DBG_GEMM_NARROW) > 0) && gemm_narrow_wanted(M, K, N, tiled)) {
        p.choice = GemmChoice::Narrow64;
        long s = forced(row_tile_splits(M, K, N, 64, NB / 16));
        if (may_split && s > 1) {  // whole 256-row stages
            p.k_split = (int)((K + s - 1) / s + 255) / 256 * 256;
            p.splits = (K + p.k_split - 1) / p.k_split;
        }
        return p;
    }
    auto use_wide = [&](int i, long s) {
        p.choice = (GemmChoice)((int)GemmChoice::Wide0 + i);
        if (may_split) split_k(K, s, kWide[i].bk, &p);
    };
    auto use_pipe64 = [&](long s) {
        p.choice = GemmChoice::Pipe64;
        if (may_split && s > 1) {  // whole 128-row stages
            p.k_split = (int)((K + s - 1) / s + 127) / 128 * 128;
            p.splits = (K + p.k_split - 1) / p.k_split;
        }
    };
    const int bm_env = debug_get(DBG_GEMM_BM), tile_env = debug_get(DBG_GEMM_BM, 1);  // tests and measurements
    if (wide && tile_env >= 0 && tile_env < kWideTiles && K >= kWide[tile_env].bk) {
        use_wide(tile_env, forced(1));
        return p;
    }
    const int bm = gemm_split_rows(M, K, N);
    const long rows_splits = forced(row_tile_splits(M, K, N, bm, (NB + 63) / 64));
    if (bm_env > 0) {
        if (bm_env == 64 && pipe16) use_pipe64(rows_splits);
        else if (wide) use_wide(bm_env == 64 ? 5 : 6, rows_splits);
        else use_pipe64(rows_splits);
        return p;
    }
    // Four or more splits above 64 rows keep the tile height and the split count of gemm_split_rows, which
    // the plan descriptions promise; the model below would pick 5-16 % faster plans there (512x11008x4096
    // 32.0 against 28.4 us, 256x8192x2048 15.4 against 13.5).  128-row tiles are tile 6 (against eight waves
    // of 64 x 64: 512x11008x4096 33.9 -> 32.0, 512x16384x4096 46.1 -> 39.3), 64-row ones tile 5 from 1024 k-rows a
    // split (256x16384x4096 28.4 -> 25.5, 256x11008x4096 23.0 -> 21.6; shorter ranges stay, 128x6912x2560 13.0
    // against 13.9).
    if (M > 64 && pipe16 && rows_splits >= 4 && may_split) {
        if (bm == 128) use_wide(6, rows_splits);
        else if (K / rows_splits >= 1024) use_wide(5, rows_splits);
        else use_pipe64(rows_splits);
        return p;
    }
    // gemm_pipe16_kernel's tiles take what is within 7 % of a tie: they are level or ahead there (2048x4096x4096 30.4
    // against 32.0 us, 512x2560x13824 20.3 / 21.3, 512x4096x11008 25.9 / 27.7), on every other choice behind.
    const long cus = device_cu_count();
    double best = pipe16 ? 0.93 * wide_cost(kPipe64Cost, M, N, K, 1) : 1e30;
    int tile = -1;
    long splits = 1;
    for (int i = 0; wide && i < 5; ++i) {
        if (K < kWide[i].bk) continue;
        const long tiles = (long)((M + kWide[i].rows - 1) / kWide[i].rows) * (long)((NB + kWide[i].bnb - 1) / kWide[i].bnb);
        for (const long s : {1L, 2L, 3L, 4L, 6L, 8L, 12L, 16L}) {
            // a split where K is long, each range at least 512 rows, and up to two rounds of two per CU
            if (s > 1 && (!may_split || K <= 4096 || K / s < 512 || tiles * s > 4 * cus)) break;
            const double t = wide_cost(kWide[i], M, N, (K + s - 1) / s, s);
            if (t < best) best = t, tile = i, splits = s;
        }
    }
    if (tile < 0) use_pipe64(1);
    else use_wide(tile, forced(splits));
    if (splits_env > 0 && tile < 0) use_pipe64(splits_env);
    return p;
}

// Ragged tiles, where one round of workgroups holds the whole output: the padded copy (6.6 us for 129x8191x2052) costs
// more than their unaligned loads.  Over more rounds the copy is read often enough to pay (400x1001x5004, 260 tiles,
// 16.8 against 14.4 us).  On MI355X, warm, us, padded copy / in place: 129x8191x2052 18.6 / 15.0, 65x4093x4100 15.1 / 12.0,
// 33x12001x3004 21.0 / 14.6, 513x8481x804 22.9 / 17.6, 257x1001x5004 12.0 / 9.7, 33x1001x516 8.4 / 8.8.
GemmPlan gemm_ragged_plan(int M, int K, int N, bool may_split) {
    // Fitted to 780 timings of 108 ragged shapes (rms error 9 %), as kWide.
    static constexpr WideTile cost[kRaggedTiles] = {
        {32, 32, 256, 2, 0.631f, 1.40f, 2.43f, 4.22f, 1.0f, 0.809f},
        {32, 64, 256, 2, 0.745f, 1.93f, 0.0f, 6.83f, 0.915f, 0.707f},
    };
    GemmPlan p;
    p.choice = GemmChoice::Invalid;
    const bool forced = debug_get(DBG_GEMM_BM) > 0 || debug_get(DBG_GEMM_BM, 1) >= 0 || debug_get(DBG_GEMM_GENERIC) == 1 ||
                        debug_get(DBG_GEMM_NARROW) >= 0 || debug_get(DBG_GEMM_SPLITS) > 0;  // tests of the other kernels
    if (!ragged_ok(M, K, N) || forced) return p;
    const long cus = device_cu_count();
    double best = 1e30;
    for (int i = 0; i < kRaggedTiles; ++i) {
        const long tiles = (long)((M + cost[i].rows - 1) / cost[i].rows) * (long)((N / 4 + cost[i].bnb - 1) / cost[i].bnb);
        for (const long s : {1L, 2L, 3L, 4L, 6L, 8L, 12L, 16L}) {
            if (tiles * s > cus || (s > 1 && (!may_split || K / s < 384))) break;
            const double t = wide_cost(cost[i], M, N, (K + s - 1) / s, s);
            if (t >= best) continue;
            best = t;
            p.choice = (GemmChoice)((int)GemmChoice::Ragged0 + i);
            split_k(K, s, 256, &p);
        }
    }
    return p;
}

const char* gemm_choice_name(GemmChoice c) {
    switch (c) {
        case GemmChoice::Narrow64: return "gemm_pipe_kernel<64 rows x 64 cols, 4 waves, 16x16x64>";
        case GemmChoice::Pipe64: return "gemm_pipe_kernel<64 rows x 256 cols, 4 waves, 16x16x64>";
        case GemmChoice::Wide0: return "gemm_pipe_kernel<32 rows x 128 cols, K over 4 waves>";
        case GemmChoice::Wide1: return "gemm_pipe_kernel<32 rows x 256 cols, K over 4 of 8 waves>";
        case GemmChoice::Wide2: return "gemm_pipe_kernel<64 rows x 256 cols, K over 4 of 8 waves>";
        case GemmChoice::Wide3: return "gemm_pipe_kernel<64 rows x 512 cols, K over 2 of 8 waves>";
        case GemmChoice::Wide4: return "gemm_pipe_kernel<64 rows x 512 cols, 4 waves>";
        case GemmChoice::Wide5: return "gemm_pipe_kernel<64 rows x 256 cols, K over 2 of 4 waves>";
        case GemmChoice::Wide6: return "gemm_pipe_kernel<128 rows x 256 cols, K over 2 of 8 waves>";
        case GemmChoice::Ragged0: return "gemm_pipe_kernel ragged<32 rows x 128 cols, K over 4 waves>";
        case GemmChoice::Ragged1: return "gemm_pipe_kernel ragged<32 rows x 256 cols, K over 4 of 8 waves>";
        case GemmChoice::Generic: return "gemm_kernel<128 rows x 256 cols, register-staged>";
        default: return "invalid";
    }
}

hipError_t launch_gemm(const GemmPlan& p, const int8_t* A, const uint8_t* B, int32_t* C, int M, int K, int N, int k_begin,
                       int k_end, int accumulate, hipStream_t st, const OutScale& os, int tiled, int n_out) {
    const int NB = N >> 2, splits = p.splits, k_split = p.k_split;
    if (n_out <= 0) n_out = N;
    const int vs = ((uintptr_t)(os.Y ? (const void*)os.Y : (const void*)C) % 16) == 0;
    const int tiles_n = NB / GF_BNB;
    const int gm_env = std::max(0, debug_get(DBG_GEMM_GM));  // tests and measurements: tile-order group
    if (n_out != N && p.choice < GemmChoice::Wide0) return hipErrorInvalidValue;
#define TX_WIDE(...) \
    launch_wide<__VA_ARGS__>(A, B, C, M, K, N, n_out, k_begin, k_end, accumulate, vs, st, os, splits, k_split, tiled, gm_env)
    switch (p.choice) {
        case GemmChoice::Invalid: return hipErrorInvalidValue;
        case GemmChoice::Generic: {
            const bool aw = (NB % 4 == 0) && ((uintptr_t)B % 4 == 0);
            const bool aa = (K % 16 == 0) && ((uintptr_t)A % 16 == 0);
            return launch_gemm_t<128, 64>(A, B, C, M, K, N, aw, aa, k_begin, k_end, accumulate, st, os, splits, k_split);
        }
        case GemmChoice::Narrow64: {
            const dim3 gridn((unsigned)(((M + 63) / 64) * (NB / 16)), splits);
            if (tiled)
                hipLaunchKernelGGL((gemm_pipe16_kernel<64, 1, 3, 256, 4, 16, true>), gridn, dim3(256), 0, st, A, B, C, M,
                                   K, N, NB / 16, k_begin, k_end, accumulate, vs, k_split, os, gm_env);
            else
                hipLaunchKernelGGL((gemm_pipe16_kernel<64, 1, 3, 256, 4, 16, false>), gridn, dim3(256), 0, st, A, B, C,
                                   M, K, N, NB / 16, k_begin, k_end, accumulate, vs, k_split, os, gm_env);
            return hipGetLastError();
        }
        case GemmChoice::Pipe64: {
            // Tiles are visited in groups of 8 row tiles per column band (512 rows): measured on MI355X with
            // cold weights, 2048x4096x4096 28.4 -> 27.0 us against groups of 4.
            const dim3 grid64((unsigned)(((M + 63) / 64) * tiles_n), splits);
            if (tiled)
                hipLaunchKernelGGL((gemm_pipe16_kernel<64, 4, 3, 128, 4, 64, true, 8>), grid64, dim3(256), 0, st, A, B,
                                   C, M, K, N, tiles_n, k_begin, k_end, accumulate, vs, k_split, os, gm_env);
            else
                hipLaunchKernelGGL((gemm_pipe16_kernel<64, 4, 3, 128, 4, 64, false, 8>), grid64, dim3(256), 0, st, A, B,
                                   C, M, K, N, tiles_n, k_begin, k_end, accumulate, vs, k_split, os, gm_env);
            return hipGetLastError();
        }
        case GemmChoice::Wide0: return TX_WIDE(1, 1, 4, 1, 256, 4, 8);
        case GemmChoice::Wide1: return TX_WIDE(1, 2, 4, 1, 256, 3, 8);
        case GemmChoice::Wide2: return TX_WIDE(1, 2, 4, 2, 256, 4, 8);
        case GemmChoice::Wide3: return TX_WIDE(1, 4, 2, 2, 128, 4, 8);
        case GemmChoice::Wide4: return TX_WIDE(1, 4, 1, 2, 128, 3, 8);
        case GemmChoice::Wide5: return TX_WIDE(1, 2, 2, 2, 128, 3, 8);
        case GemmChoice::Wide6: return TX_WIDE(2, 2, 2, 2, 128, 4, 4);
        case GemmChoice::Ragged0: return TX_WIDE(1, 1, 4, 1, 256, 2, 8, true);
        default: return TX_WIDE(1, 2, 4, 1, 256, 2, 8, true);
    }
#undef TX_WIDE
}

}  // namespace ternix_hip
