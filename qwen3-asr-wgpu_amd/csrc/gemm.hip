// gemm.hip -- the prefill projections' GEMM on fp16 MFMA (gfx950):
//   C[m][n] = f16(sum_k A[m][k] * B[n][k]  (+ C[m][n]))
// or, for gate|up, C[m][n] = f16(SiLU(gate) * up) of the rounded products.
// A: activation rows [M][K], B: weight rows [N][K] (checkpoint layout), both
// K-contiguous; f32 accumulation, one rounding of the f32 result (with the
// residual added in f32 first when accumulating) -- the rounding points of
// the reference's batched projections (cpu_decoder.rs:45-62 batch_dot_acc,
// 398-449; dispatched on the GPU by decoder.rs:3580-4162).
//
// Two kernels of one design, for tiles of 128 x 256 and more (gemm_big_kernel)
// and down to 64 x 64 (gemm_small_kernel); launch_gemm_f16 chooses per shape by
// a cost model.  K steps of 64; four waves, each computing tiles of
// v_mfma_f32_32x32x16_f16 as D = B A^T, so that a lane ends with four
// consecutive columns of a row.  Both operand tiles go global -> LDS by direct
// copies (buffer_load ... lds, one 1 KB block per wave instruction) into a ring
// of stages; the copies are inline asm waited for by count, and the barriers
// are bare, so several steps' copies stay in flight across them.  LDS row
// layout (both operands): row r is 128 bytes (64 k), its 16-byte chunk c at slot
// c ^ ((r >> 1) & 7), so an operand read (16 consecutive rows, one chunk)
// covers 16 distinct 16-byte bank groups.  Rows past M are copied from row
// M - 1 (finite values; their outputs are not stored).
// Workgroups are dealt round-robin to the 8 XCDs: when the column blocks
// divide by 8, XCD x takes a contiguous run of them and walks them in groups
// of a few row blocks, so the tiles an XCD runs at one time share a few A
// and B blocks in its L2.
// Every output sums over K in one fixed order whatever the tile.
// Figures (us, one MI355X, both builds in turn, against the two-stage ping-pong
// and slice-by-slice loops before; weight matrices rotated so that they come
// from HBM): 4269 x 12288 x 2048 209 -> 189, 4269 x 4096 x 2048 85 -> 69, 4269 x 2048 x
// 2048 + residual 52 -> 42, 4269 x 2048 x 6144 + residual 142 -> 106, 420 x 12288 x
// 2048 39.5 -> 32.6, 420 x 4096 x 2048 18.6 -> 15.9, 420 x 2048 x 2048 + residual 11.4 ->
// 11.0, 420 x 2048 x 6144 + residual 29.0 -> 28.0, 131 x 1024 x 3072 + residual 15.0 -> 14.1;
// one matrix, in the memory-side cache: the last three 10.7 -> 9.3, 25.4 -> 21.1, 14.5 -> 11.5.

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <type_traits>

#include "kernels.hpp"

namespace qasr {

namespace {

constexpr int kBK = 64;             // k per step
constexpr int kRowBytes = kBK * 2;  // 128 bytes of one row per step
constexpr int kSlices = kBK / 16;   // MFMA k-slices per step
constexpr int kGroupRows = 4;       // row blocks per group of an XCD's tile walk

__device__ __forceinline__ float16v mfma32(const half8v& a, const half8v& b, const float16v& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ int slot_of(int row, int chunk) { return chunk ^ ((row >> 1) & 7); }

// s_waitcnt vmcnt(VM) lgkmcnt(0): at most VM vector memory operations of this
// wave still in flight, and no LDS operation.
template <int VM>
__device__ __forceinline__ void wait_vm_lgkm0() {
    static_assert(VM >= 0 && VM <= 63, "vmcnt range");
    __builtin_amdgcn_s_waitcnt(0x0070 | (VM & 15) | ((VM >> 4) << 14));
}

// A bare workgroup barrier: the caller has waited for what must have landed
// (a __syncthreads() would also drain the LDS reads still wanted in flight).
__device__ __forceinline__ void bare_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// dma16 (common.hpp) with the step's byte offset in a scalar register.
__device__ __forceinline__ void dma16_at(const u32x4v& rsrc, int voff, int soff, uint32_t lds) {
    asm volatile("buffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(voff), "s"(rsrc), "s"(soff), "{m0}"(lds)
                 : "memory");
}

// kGemmGlu: weight row of B row r of a block whose first column is n0 (of N):
// groups of 16 gate rows and the up rows of the same 16 columns in turn.
__device__ __forceinline__ int glu_row(int n0, int r, int N) {
    return ((r >> 4) & 1) * (N / 2) + n0 / 2 + (r >> 5) * 16 + (r & 15);
}

// Block coordinates of workgroup bid over nmt row and nnt column blocks (see
// the XCD note above).
__device__ __forceinline__ void tile_of(int bid, int nmt, int nnt, int& mt, int& nt) {
    if (nnt % 8 == 0) {
        const int x = bid & 7, j = bid >> 3, nper = nnt >> 3;
        const int grp = j / (kGroupRows * nper);
        const int gr = min(kGroupRows, nmt - grp * kGroupRows);
        const int r = j - grp * kGroupRows * nper;
        mt = grp * kGroupRows + r % gr;
        nt = x * nper + r / gr;
    } else {
        mt = bid % nmt;
        nt = bid / nmt;
    }
}

// The wave's outputs, from D = B A^T tiles: acc[i][j][e] is row m0 + 32 i +
// l32, column n0 + 32 j + 8 (e / 4) + 4 g + e % 4 (four consecutive columns of
// a row per lane).  Each 32-row strip goes through the wave's own LDS region
// `ep` and out as whole row pieces of 16 bytes a lane (without: 2-byte stores,
// and 256 x 256 x 2048 tiles took ~3 us longer each); with the residual the
// strip is staged in f32 and all its C pieces are requested before the first
// use (one memory round trip per strip).  Rows past M are not stored.
// kGemmGlu: the 32 B rows of tile j are 16 gate rows and the same 16 columns'
// up rows (glu_row), so a lane holds gate in elements 0..7 and up in 8..15 and
// writes h = f16(SiLU(gate) up), both rounded to f16 first, to columns n0 + 16 j
// + 8 (e / 4) + 4 g + e % 4, e < 8, of C [M][N / 2].
template <int MT, int NT, int OUT>
struct Epilogue {
    static constexpr bool ACC = OUT == kGemmAcc, GLU = OUT == kGemmGlu;
    static constexpr int kCols = GLU ? 16 * NT : 32 * NT;
    static constexpr int kRow = ACC ? kCols * 4 + 16 : kCols * 2 + 16;  // padded LDS row, bytes
    static constexpr int kBytes = 32 * kRow;                            // per wave
    static constexpr int kPer = kCols / 8;                              // 8-column pieces per row
    static constexpr int kIt = 32 * kPer / 64;                          // pieces per lane and strip

    static __device__ __forceinline__ void run(float16v (&acc)[MT][NT], char* ep, f16* __restrict__ C, int M,
                                               int N, int m0, int n0, int lane) {
        const int g = lane >> 5, l32 = lane & 31;
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            H8 old[ACC ? kIt : 1];
            if constexpr (ACC) {
#pragma unroll
                for (int it = 0; it < kIt; ++it) {
                    const int p = 64 * it + lane, m = min(m0 + 32 * i + p / kPer, M - 1);
                    old[it].u = *reinterpret_cast<const uint4*>(C + (int64_t)m * N + n0 + (p % kPer) * 8);
                }
            }
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int q = 0; q < (GLU ? 2 : 4); ++q) {
                    const int col = (GLU ? 16 : 32) * j + 8 * q + 4 * g;
                    if constexpr (GLU) {
                        half4v h;
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            h[e] = f16_of_f32(silu_times((float)(f16)acc[i][j][4 * q + e], (float)(f16)acc[i][j][8 + 4 * q + e]));
                        *reinterpret_cast<half4v*>(ep + l32 * kRow + col * 2) = h;
                    } else if constexpr (ACC) {
                        *reinterpret_cast<float4*>(ep + l32 * kRow + col * 4) =
                            make_float4(acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]);
                    } else {
                        half4v h;
#pragma unroll
                        for (int e = 0; e < 4; ++e) h[e] = (f16)acc[i][j][4 * q + e];
                        *reinterpret_cast<half4v*>(ep + l32 * kRow + col * 2) = h;
                    }
                }
            __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the strip is in LDS
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int it = 0; it < kIt; ++it) {
                const int p = 64 * it + lane, r = p / kPer, c8 = p % kPer;
                const int m = m0 + 32 * i + r;
                H8 o;
                if constexpr (ACC) {
                    const float4 lo = *reinterpret_cast<const float4*>(ep + r * kRow + c8 * 32);
                    const float4 hi = *reinterpret_cast<const float4*>(ep + r * kRow + c8 * 32 + 16);
                    const float v[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
                    for (int e = 0; e < 8; ++e) o.e[e] = (f16)((float)old[it].e[e] + v[e]);
                } else {
                    o.u = *reinterpret_cast<const uint4*>(ep + r * kRow + c8 * 16);
                }
                if (m < M) *reinterpret_cast<uint4*>(C + (int64_t)m * N + n0 + c8 * 8) = o.u;
            }
            __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): reads done before the next strip's writes
            __builtin_amdgcn_wave_barrier();
        }
    }
};

// ---- large tiles -------------------------------------------------------------
// Four waves in a WGM x (4 / WGM) grid, one per SIMD: 2 x 2, the largest wave
// tile, so the fewest LDS operand bytes per MFMA, or 1 x 4 for 160 rows (five
// 32-row tiles a wave; 4,269 rows of 2,048 columns are then 216 blocks of 256
// CUs, not 184 of 192 rows: K = 6144 with the residual 112-115 -> 107 us).  What bounds it is the
// copies: a CU takes in at most ~85 GB/s of them (a copy-only loop of these
// tiles), 0.75 us for the 64 KB of a 256 x 256 step against 0.85 us of MFMAs,
// so they have to run all the time.  With two stages of both operands they
// could only be issued once a step's reads were done, and had to land before
// the next step's: 1.4 us a step.  Three stages of A, and of B where LDS holds
// them (144 KB with 128 rows, 156 KB with 160; two stages of B with 192 rows, 136 KB,
// and 256, 160 KB), keep a third of a step or more queued across the barrier: 1.1 us (4269 x 2048 x 6144 with the
// residual, this tile: 149 -> 118 us).
//
// Steps: slice ks + 1's operand reads go out one per MFMA under slice ks's
// MFMAs.  In slice 3, after MFMA kBar, the wave waits for its copies of step
// t + 1 and its own reads of step t; past the barrier every wave is done with
// step t's buffers, so its stage of B and A is refilled (with steps t + NB and
// t + 3), the copies spread over the MFMAs up to the next barrier: B first, at
// every second MFMA, then A.
constexpr int kBar = 2;

template <int BM, int BN, int NB, int WGM, int OUT>
__global__ __launch_bounds__(256, 1) void gemm_big_kernel(const f16* __restrict__ A, const f16* __restrict__ B,
                                                          f16* __restrict__ C, int M, int N, int K) {
    constexpr int WGN = 4 / WGM, WM = BM / WGM, WN = BN / WGN;
    constexpr int MT = WM / 32, NT = WN / 32;
    static_assert(MT * 32 * WGM == BM && NT * 32 * WGN == BN, "wave tile of whole 32 x 32 MFMA tiles");
    constexpr int ACOPY = BM / 32, BCOPY = BN / 32;  // copies per wave and step
    constexpr int S = MT * NT;                       // MFMAs per slice
    constexpr int NA = 3;
    constexpr int kABuf = BM * kRowBytes, kBBuf = BN * kRowBytes;
    static_assert((NB == 2 || NB == 3) && NA * kABuf + NB * kBBuf <= 160 * 1024, "LDS");
    static_assert(S >= MT + NT && S > kBar, "one operand read per MFMA of a slice");
    // Position of a copy in MFMAs since the barrier: B copy j at 1 + 2 j, A
    // copies evenly over the rest, the last before slice 3.
    constexpr int kPosA0 = 2 * BCOPY + 2, kPosEnd = 4 * S - kBar;
    constexpr int kStrA = (kPosEnd - kPosA0) / ACOPY;
    static_assert(kStrA >= 1, "copies fit a step");
    constexpr int kEarlyB = (S - kBar) / 2 < BCOPY ? (S - kBar) / 2 : BCOPY;  // B copies inside slice 3
    __shared__ __attribute__((aligned(16))) char smem[NA * kABuf + NB * kBBuf];
    static_assert(4 * Epilogue<MT, NT, OUT>::kBytes <= NA * kABuf + NB * kBBuf, "epilogue staging fits");
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WGN, wn = wave % WGN;
    const int g = lane >> 5, l32 = lane & 31;
    int mt, nt;
    tile_of(blockIdx.x, (M + BM - 1) / BM, N / BN, mt, nt);
    const int m0 = mt * BM, n0 = nt * BN;

    const u32x4v ares = make_rsrc_words(A, M * K * 2);
    const u32x4v bres = make_rsrc_words(B, N * K * 2);
    // Copy j of wave w fills LDS bytes [(4 j + w) KB, +1 KB) of a stage:
    // 16-byte unit p = 64 (4 j + w) + lane, row p / 8, slot p % 8.
    int aoff[ACOPY], boff[BCOPY];
#pragma unroll
    for (int j = 0; j < ACOPY; ++j) {
        const int p = 64 * (4 * j + wave) + lane, row = p >> 3;
        aoff[j] = min(m0 + row, M - 1) * K * 2 + slot_of(row, p & 7) * 16;
    }
#pragma unroll
    for (int j = 0; j < BCOPY; ++j) {
        const int p = 64 * (4 * j + wave) + lane, row = p >> 3;
        boff[j] = (OUT == kGemmGlu ? glu_row(n0, row, N) : n0 + row) * K * 2 + slot_of(row, p & 7) * 16;
    }
    const uint32_t alds = lds_addr(smem) + wave * 1024, blds = alds + NA * kABuf;
    auto copy_a = [&](int t, int buf, int j) { dma16_at(ares, aoff[j], t * kRowBytes, alds + buf + j * 4096); };
    auto copy_b = [&](int t, int buf, int j) { dma16_at(bres, boff[j], t * kRowBytes, blds + buf + j * 4096); };

    // Operand addresses of slice ks within a stage (row tile i: + 4 KB i).
    int ao[kSlices], bo[kSlices];
#pragma unroll
    for (int ks = 0; ks < kSlices; ++ks) {
        const int ra = wm * WM + l32, rb = wn * WN + l32;
        ao[ks] = ra * kRowBytes + slot_of(ra, 2 * ks + g) * 16;
        bo[ks] = NA * kABuf + rb * kRowBytes + slot_of(rb, 2 * ks + g) * 16;
    }
    half8v fa[2][MT], fb[2][NT];
    // Read x of slice ks (a0, b0 .. b(NT-1), a1 ..); after the slice's last its
    // addresses step, in place, by da and db to the next step's stage (an
    // address made in a register that MFMAs in flight still read would wait
    // for them).
    auto read = [&](int da, int db, int ks, int q, int x) {
        if (x == 0 || x > NT) {
            const int i = x == 0 ? 0 : x - NT;
            fa[q][i] = *(const half8v*)(smem + ao[ks] + i * 4096);
        } else {
            fb[q][x - 1] = *(const half8v*)(smem + bo[ks] + (x - 1) * 4096);
        }
        if (x == MT + NT - 1) {
            ao[ks] += da;
            bo[ks] += db;
            asm volatile("" : "+v"(ao[ks]), "+v"(bo[ks]));
        }
    };
    float16v acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = (float16v){};

    // Step t.  a0 .. a2, b0 .. b2: stage offsets of steps t, t + 1, t + 2 (NB ==
    // 2: b2 == b0); the stage of step t - 1 is a2, and b2 or (NB == 2) b1.
    // F: its copies: bit 0 the rest of B(t - 1 + NB) and bit 1 A(t + 2) under
    // slices 0..2, bit 2 B(t + NB) after the barrier; bit 3: the last step.
    auto step = [&](int t, int a0, int a1, int a2, int b0, int b1, int b2, auto Flags) {
        constexpr int F = decltype(Flags)::value;
#pragma unroll
        for (int ks = 0; ks < kSlices; ++ks) {
#pragma unroll
            for (int m = 0; m < S; ++m) {
                const int i = m / NT, j = m % NT, q = ks & 1;
                acc[i][j] = mfma32(fb[q][j], fa[q][i], acc[i][j]);  // D = B A^T
                __builtin_amdgcn_sched_barrier(0);
                if (ks < kSlices - 1) {
                    if (m < MT + NT) read(a1 - a0, b1 - b0, ks + 1, q ^ 1, m);
                    const int pos = S - kBar + ks * S + m;
                    if ((F & 1) && (pos & 1) && pos >= 1 + 2 * kEarlyB && (pos - 1) / 2 < BCOPY)
                        copy_b(t - 1 + NB, NB == 3 ? b2 : b1, (pos - 1) / 2);
                    if ((F & 2) && pos >= kPosA0 && (pos - kPosA0) % kStrA == 0 && (pos - kPosA0) / kStrA < ACOPY)
                        copy_a(t + 2, a2, (pos - kPosA0) / kStrA);
                } else if (!(F & 8)) {
                    if (m == kBar) {
                        wait_vm_lgkm0<F == 7 ? (NB == 2 ? ACOPY : ACOPY + BCOPY) : 0>();
                        bare_barrier();
                    }
                    if (m >= kBar) {
                        if (m - kBar < MT + NT) read(a2 - a1, b2 - b1, 0, 0, m - kBar);
                        if (m == S - 1)
#pragma unroll
                            for (int x = S - kBar; x < MT + NT; ++x) read(a2 - a1, b2 - b1, 0, 0, x);
                    }
                    const int pos = m - kBar;
                    if ((F & 4) && pos > 0 && (pos & 1) && (pos - 1) / 2 < kEarlyB) copy_b(t + NB, b0, (pos - 1) / 2);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    using Full = std::integral_constant<int, 7>;
    const int nk = K / kBK;  // >= NB (Tile::min_steps)
#pragma unroll
    for (int j = 0; j < ACOPY; ++j) copy_a(0, 0, j);
#pragma unroll
    for (int j = 0; j < BCOPY; ++j) copy_b(0, 0, j);
#pragma unroll
    for (int j = 0; j < ACOPY; ++j) copy_a(1, kABuf, j);
    if constexpr (NB == 3)
#pragma unroll
        for (int j = 0; j < BCOPY; ++j) copy_b(1, kBBuf, j);
#pragma unroll
    for (int j = 0; j < kEarlyB; ++j) copy_b(NB - 1, (NB - 1) * kBBuf, j);
    wait_vm_lgkm0<ACOPY + (NB == 3 ? BCOPY : 0) + kEarlyB>();
    bare_barrier();
#pragma unroll
    for (int x = 0; x < MT + NT; ++x) read(kABuf, kBBuf, 0, 0, x);
    __builtin_amdgcn_sched_barrier(0);
    int t = 0, a0 = 0, a1 = kABuf, a2 = 2 * kABuf, b0 = 0, b1 = kBBuf, b2 = NB == 3 ? 2 * kBBuf : 0;
    auto advance = [&]() {
        const int x = a0, y = b0;
        a0 = a1;
        a1 = a2;
        a2 = x;
        b0 = b1;
        b1 = b2;
        b2 = NB == 3 ? y : b0;
        ++t;
    };
    while (t + NB < nk) {
        step(t, a0, a1, a2, b0, b1, b2, Full{});
        advance();
    }
    if constexpr (NB == 3) {
        step(t, a0, a1, a2, b0, b1, b2, std::integral_constant<int, 3>{});
        advance();
        step(t, a0, a1, a2, b0, b1, b2, std::integral_constant<int, 0>{});
    } else {
        step(t, a0, a1, a2, b0, b1, b2, std::integral_constant<int, 1>{});
    }
    advance();
    step(t, a0, a1, a2, b0, b1, b2, std::integral_constant<int, 8>{});
    __syncthreads();  // every wave is past its last operand reads
    Epilogue<MT, NT, OUT>::run(acc, smem + wave * Epilogue<MT, NT, OUT>::kBytes, C, M, OUT == kGemmGlu ? N / 2 : N,
                               m0 + wm * WM, (n0 + wn * WN) / (OUT == kGemmGlu ? 2 : 1), lane);
}

// ---- small tiles -------------------------------------------------------------
// Waves in a 2 x WGN grid.  Their K steps are short (a 64 x 64 step is 128
// MFMA cycles per SIMD against ~380 of LDS traffic), so what counts is that no
// LDS or memory latency is waited for: a whole step's operands are read into
// registers under the previous step's MFMAs (one barrier per step, where a
// read of each 16-k slice under the slice before it waited four LDS latencies:
// 131 x 1024 x 3072 14.6 -> 11.8 us, 420 x 2048 x 6144 26.2 -> 22.4 us with the weights
// in the memory-side cache), and
// NS stages keep NS - 2 steps of copies in flight.
// SLICED: each slice is read under the MFMAs of the slice before it.  Where
// some CUs have two workgroups, the other one covers the LDS latencies and
// whole-step reads only queue up behind each other.  64 x 64 tiles, one to 1.5
// a CU, whole-step reads -> slices, us, weights from HBM and (in brackets) in the
// memory-side cache: 576 x 2048 x 2048 + residual 14.7 -> 13.9 (13.1 -> 11.7),
// 576 x 2048 x 6144 + residual 39.5 -> 37.7 (36.8 -> 36.3), 192 x 6144 x 1024 11.1 ->
// 10.9 (7.7 -> 7.3); only with few row blocks and weights from HBM are slices slower:
// 384 x 4096 x 2048 17.4 -> 17.9 (13.3 -> 12.2).  At one tile a CU (495 x 2048 x 2048
// 11.3 (9.4) -> 11.4 (10.6)) and near two (1007 rows 18.2 -> 18.5) whole steps are faster.
template <int BM, int BN, int NS, int WGN, bool SLICED, int OUT>
__global__ __launch_bounds__(128 * WGN, 1) void gemm_small_kernel(const f16* __restrict__ A, const f16* __restrict__ B,
                                                                  f16* __restrict__ C, int M, int N, int K) {
    constexpr int kWaves = 2 * WGN;
    constexpr int WM = BM / 2, WN = BN / WGN;
    constexpr int MT = WM / 32, NT = WN / 32;
    static_assert(MT >= 1 && NT >= 1, "wave tile of whole 32 x 32 MFMA tiles");
    constexpr int ACOPY = BM * kRowBytes / 1024 / kWaves;  // copy instructions per wave and step
    constexpr int BCOPY = BN * kRowBytes / 1024 / kWaves;
    static_assert(ACOPY * kWaves * 1024 == BM * kRowBytes && BCOPY * kWaves * 1024 == BN * kRowBytes,
                  "whole 1 KB copy blocks per wave");
    constexpr int kStepCopies = ACOPY + BCOPY;
    static_assert(NS >= 2 && NS <= 6 && (NS - 1) * kStepCopies <= 63, "copy stages");
    constexpr int kABuf = BM * kRowBytes, kBBuf = BN * kRowBytes;
    __shared__ __attribute__((aligned(16))) char smem[NS * (kABuf + kBBuf)];
    static_assert(kWaves * Epilogue<MT, NT, OUT>::kBytes <= NS * (kABuf + kBBuf), "epilogue staging fits");
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WGN, wn = wave % WGN;
    const int g = lane >> 5, l32 = lane & 31;
    int mt, nt;
    tile_of(blockIdx.x, (M + BM - 1) / BM, N / BN, mt, nt);
    const int m0 = mt * BM, n0 = nt * BN;

    const u32x4v ares = make_rsrc_words(A, M * K * 2);
    const u32x4v bres = make_rsrc_words(B, N * K * 2);
    int aoff[ACOPY], boff[BCOPY];  // as in gemm_big_kernel
#pragma unroll
    for (int j = 0; j < ACOPY; ++j) {
        const int p = 64 * (kWaves * j + wave) + lane, row = p >> 3;
        aoff[j] = min(m0 + row, M - 1) * K * 2 + slot_of(row, p & 7) * 16;
    }
#pragma unroll
    for (int j = 0; j < BCOPY; ++j) {
        const int p = 64 * (kWaves * j + wave) + lane, row = p >> 3;
        boff[j] = (OUT == kGemmGlu ? glu_row(n0, row, N) : n0 + row) * K * 2 + slot_of(row, p & 7) * 16;
    }
    const uint32_t alds = lds_addr(smem) + wave * 1024, blds = alds + NS * kABuf;
    auto copy_step = [&](int t, int buf) {
        const int kb = t * kRowBytes;
#pragma unroll
        for (int j = 0; j < ACOPY; ++j) dma16_at(ares, aoff[j], kb, alds + buf * kABuf + j * kWaves * 1024);
#pragma unroll
        for (int j = 0; j < BCOPY; ++j) dma16_at(bres, boff[j], kb, blds + buf * kBBuf + j * kWaves * 1024);
    };
    int ao[kSlices], bo[kSlices];
#pragma unroll
    for (int ks = 0; ks < kSlices; ++ks) {
        const int ra = wm * WM + l32, rb = wn * WN + l32;
        ao[ks] = ra * kRowBytes + slot_of(ra, 2 * ks + g) * 16;
        bo[ks] = NS * kABuf + rb * kRowBytes + slot_of(rb, 2 * ks + g) * 16;
    }
    float16v acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = (float16v){};
    // At most `steps` steps' copies of this wave in flight, no LDS read.
    auto wait_steps = [&](int steps) {
        if (NS > 4 && steps >= 4)
            wait_vm_lgkm0<(NS > 4 ? 4 : 0) * kStepCopies>();
        else if (NS > 3 && steps >= 3)
            wait_vm_lgkm0<(NS > 3 ? 3 : 0) * kStepCopies>();
        else if (NS > 2 && steps >= 2)
            wait_vm_lgkm0<(NS > 2 ? 2 : 0) * kStepCopies>();
        else if (steps >= 1)
            wait_vm_lgkm0<kStepCopies>();
        else
            wait_vm_lgkm0<0>();
    };
    const int nk = K / kBK;
    const int npro = nk < NS ? nk : NS;  // steps copied ahead
    for (int t = 0; t < npro; ++t) copy_step(t, t);
    wait_steps(npro - 1 < 4 ? npro - 1 : 4);
    bare_barrier();
    auto next = [&](int b) { return b + 1 == NS ? 0 : b + 1; };
    if constexpr (SLICED) {
        half8v fa[2][MT], fb[2][NT];
        auto read_slice = [&](int buf, int ks) {
#pragma unroll
            for (int i = 0; i < MT; ++i) fa[ks & 1][i] = *(const half8v*)(smem + buf * kABuf + ao[ks] + i * 4096);
#pragma unroll
            for (int i = 0; i < NT; ++i) fb[ks & 1][i] = *(const half8v*)(smem + buf * kBBuf + bo[ks] + i * 4096);
        };
        auto mfma_slice = [&](int ks) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j)
                    acc[i][j] = mfma32(fb[ks & 1][j], fa[ks & 1][i], acc[i][j]);  // D = B A^T
            __builtin_amdgcn_sched_barrier(0);
        };
        read_slice(0, 0);
        for (int t = 0, buf = 0; t < nk; ++t) {
            __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): slice 0
#pragma unroll
            for (int ks = 0; ks + 1 < kSlices; ++ks) {
                read_slice(buf, ks + 1);
                mfma_slice(ks);
            }
            // Once every wave has its last reads of step t and its copies of
            // step t + 1, that step's first slice is read and stage buf refilled
            // (reads first: 559 x 2048 x 2048 in the cache 12.9 -> 12.1 us).
            if (t + 1 < nk) {
                wait_steps(min(t + NS - 1, nk - 1) - (t + 1));
                bare_barrier();
                const int done = buf;
                buf = next(buf);
                read_slice(buf, 0);
                __builtin_amdgcn_sched_barrier(0);
                if (t + NS < nk) copy_step(t + NS, done);
            }
            mfma_slice(kSlices - 1);
        }
        bare_barrier();  // every wave has its last operand reads
    } else {
        half8v fa[2][kSlices][MT], fb[2][kSlices][NT];
        // The addresses step to the next stage (buf + 1, or back to 0) in place: an
        // address made in a register the MFMAs in flight still read would wait for
        // them (420 x 2048 x 6144: 25 against 21.5 us).
        auto read_step = [&](int buf, int q) {
            const int da = buf == NS - 1 ? -(NS - 1) * kABuf : kABuf;
            const int db = buf == NS - 1 ? -(NS - 1) * kBBuf : kBBuf;
#pragma unroll
            for (int ks = 0; ks < kSlices; ++ks) {
#pragma unroll
                for (int i = 0; i < MT; ++i) fa[q][ks][i] = *(const half8v*)(smem + ao[ks] + i * 4096);
#pragma unroll
                for (int i = 0; i < NT; ++i) fb[q][ks][i] = *(const half8v*)(smem + bo[ks] + i * 4096);
                ao[ks] += da;
                bo[ks] += db;
                asm volatile("" : "+v"(ao[ks]), "+v"(bo[ks]));
            }
        };
        auto mfma_step = [&](int q) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int ks = 0; ks < kSlices; ++ks)
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int j = 0; j < NT; ++j) acc[i][j] = mfma32(fb[q][ks][j], fa[q][ks][i], acc[i][j]);  // D = B A^T
            __builtin_amdgcn_sched_barrier(0);
        };
        read_step(0, 0);
        // Step t (stage buf, operands in registers q): its reads and the copies of
        // step t + 1 have landed in every wave, so stage buf takes step t + NS and
        // step t + 1 is read under this step's MFMAs.
        int t = 0, buf = 0;
        for (; t + 1 + NS < nk; t += 2) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                wait_vm_lgkm0<(NS - 2) * kStepCopies>();
                bare_barrier();
                copy_step(t + u + NS, buf);
                buf = next(buf);
                read_step(buf, u ^ 1);
                mfma_step(u);
            }
        }
        for (; t < nk; t += 2) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                if (t + u < nk) {
                    const int newest = min(t + u + NS - 1, nk - 1);  // last step copied
                    wait_steps(newest - (t + u + 1));
                    bare_barrier();
                    if (t + u + NS < nk) copy_step(t + u + NS, buf);
                    buf = next(buf);
                    if (t + u + 1 < nk) read_step(buf, u ^ 1);
                    mfma_step(u);
                }
            }
        }
    }
    // (Whole-step reads: every wave's last returned before the last step's barrier.)
    Epilogue<MT, NT, OUT>::run(acc, smem + wave * Epilogue<MT, NT, OUT>::kBytes, C, M, OUT == kGemmGlu ? N / 2 : N,
                               m0 + wm * WM, (n0 + wn * WN) / (OUT == kGemmGlu ? 2 : 1), lane);
}

struct GemmCall {
    const f16* A;
    const f16* B;
    f16* C;
    int M, N, K;
    GemmOut out;
    int64_t cus;
    hipStream_t stream;
};

template <int BM, int BN, int NB, int WGM>
hipError_t launch_big(const GemmCall& c) {
    const dim3 grid((unsigned)(((c.M + BM - 1) / BM) * (c.N / BN)));
    if (c.out == kGemmAcc)
        hipLaunchKernelGGL((gemm_big_kernel<BM, BN, NB, WGM, kGemmAcc>), grid, dim3(256), 0, c.stream, c.A, c.B, c.C, c.M, c.N, c.K);
    else if (c.out == kGemmGlu)
        hipLaunchKernelGGL((gemm_big_kernel<BM, BN, NB, WGM, kGemmGlu>), grid, dim3(256), 0, c.stream, c.A, c.B, c.C, c.M, c.N, c.K);
    else
        hipLaunchKernelGGL((gemm_big_kernel<BM, BN, NB, WGM, kGemmStore>), grid, dim3(256), 0, c.stream, c.A, c.B, c.C, c.M, c.N, c.K);
    return hipGetLastError();
}

template <int BM, int BN, int NS, int WGN, bool SLICED>
hipError_t launch_small(const GemmCall& c) {
    const dim3 grid((unsigned)(((c.M + BM - 1) / BM) * (c.N / BN)));
    if (c.out == kGemmAcc)
        hipLaunchKernelGGL((gemm_small_kernel<BM, BN, NS, WGN, SLICED, kGemmAcc>), grid, dim3(128 * WGN), 0, c.stream, c.A, c.B, c.C, c.M, c.N, c.K);
    else if (c.out == kGemmGlu)
        hipLaunchKernelGGL((gemm_small_kernel<BM, BN, NS, WGN, SLICED, kGemmGlu>), grid, dim3(128 * WGN), 0, c.stream, c.A, c.B, c.C, c.M, c.N, c.K);
    else
        hipLaunchKernelGGL((gemm_small_kernel<BM, BN, NS, WGN, SLICED, kGemmStore>), grid, dim3(128 * WGN), 0, c.stream, c.A, c.B, c.C, c.M, c.N, c.K);
    return hipGetLastError();
}

// Block tiles.  `occ` workgroups of a tile fit a CU (LDS).  A workgroup takes
// fix + (K / 64) step us: the large tiles, alone on a CU, run in whole rounds
// of one per CU; the small ones take step[0] alone and step[1] two to a CU
// (in between, as the square root of the share of CUs with two), and fill in
// behind each other, so a last part round costs little more than its share.
// The figures are sweeps of every tile over the 1.7B and 0.6B projections at 64
// to 4,269 rows and a 16384 x 12288 x 2048 product, weights coming from HBM.
// 160 x 256 is charged what it takes at K = 6144 (105-110 us a busy round, 108 here),
// which is more than it takes at K = 1024 and 2048 (21 and 37 us, 26 and 43 here):
// with 5.5 + 0.97 a step it is also chosen for second launches of a row split, whose
// rounds overlap the first's, and those were up to 6% slower (3400 x 6144 x 1024
// 42.3 -> 44.9 us).  So it serves N = 2048 with a long K, one round of it for
// 4,097 to 5,120 rows.
struct Tile {
    int bm, bn, occ;
    float fix, step[2];
    int min_steps;  // K steps the kernel needs: its stages of B when large (launch_tile)
};
constexpr Tile kTiles[] = {{256, 256, 1, 6.5f, {1.50f, 0.0f}, 2},
                       {192, 256, 1, 6.0f, {1.10f, 0.0f}, 2},
                       {128, 256, 1, 5.5f, {0.82f, 0.0f}, 3},
                       {64, 128, 2, 4.0f, {0.40f, 0.62f}, 1},
                       {128, 64, 2, 4.0f, {0.38f, 0.62f}, 1},
                       {64, 64, 2, 3.5f, {0.25f, 0.44f}, 1},
                       {160, 256, 1, 10.0f, {1.02f, 0.0f}, 3}};
constexpr int kNumTiles = (int)(sizeof kTiles / sizeof kTiles[0]);
constexpr float kSecondLaunchUs = 2.0f;

// Kernel instances of kTiles[I]: the sizes come from the table, and its
// min_steps cover the copies that a large tile issues ahead.
template <int I, int NB, int WGM>
hipError_t launch_big_tile(const GemmCall& c) {
    static_assert(kTiles[I].min_steps >= NB, "steps copied ahead");
    return launch_big<kTiles[I].bm, kTiles[I].bn, NB, WGM>(c);
}

template <int I, int NS, int WGN, bool SLICED = false>
hipError_t launch_small_tile(const GemmCall& c) {
    return launch_small<kTiles[I].bm, kTiles[I].bn, NS, WGN, SLICED>(c);
}

hipError_t launch_tile(const Tile& t, const GemmCall& c) {
    static_assert(kNumTiles == 7, "one case per tile");
    switch (&t - kTiles) {
        case 0: return launch_big_tile<0, 2, 2>(c);
        case 1: return launch_big_tile<1, 2, 2>(c);
        case 2: return launch_big_tile<2, 3, 2>(c);
        case 3: return launch_small_tile<3, 3, 2>(c);
        case 4: return launch_small_tile<4, 3, 2>(c);
        case 5: {
            // One to 1.5 tiles a CU: slice by slice (see gemm_small_kernel).
            const int64_t tiles = (int64_t)((c.M + 63) / 64) * (c.N / 64);
            if (tiles > c.cus && 2 * tiles <= 3 * c.cus) return launch_small_tile<5, 4, 2, true>(c);
            return launch_small_tile<5, 4, 2>(c);
        }
        default: return launch_big_tile<6, 3, 1>(c);
    }
}

float tile_us(const Tile& c, int64_t rows, int N, int K, int64_t cus) {
    const int64_t tiles = (rows + c.bm - 1) / c.bm * (N / c.bn);
    const float steps = (float)(K / kBK);
    if (c.occ == 1) return (float)((tiles + cus - 1) / cus) * (c.fix + steps * c.step[0]);
    const float per_cu = (float)tiles / (float)cus;
    if (per_cu <= 1.0f) return c.fix + steps * c.step[0];
    if (per_cu <= 2.0f) return c.fix + steps * (c.step[0] + (c.step[1] - c.step[0]) * std::sqrt(per_cu - 1.0f));
    const float rounds = 0.5f * per_cu;
    return (rounds + 0.5f * (std::ceil(rounds) - rounds)) * (c.fix + steps * c.step[1]);
}

// The tile of least predicted time for `rows` rows.
const Tile& best_tile(int64_t rows, int N, int K, int64_t cus, float* us) {
    const Tile* best = nullptr;
    for (const Tile& c : kTiles) {
        if (K / kBK < c.min_steps) continue;
        const float t = tile_us(c, rows, N, K, cus);
        if (!best || t < *us) {
            best = &c;
            *us = t;
        }
    }
    return *best;
}

}  // namespace

bool gemm_f16_fits(int M, int N, int K) {
    return M > 0 && N > 0 && K > 0 && K % kBK == 0 && N % 256 == 0 &&
           (int64_t)M * K * 2 < (int64_t(1) << 31) && (int64_t)N * K * 2 < (int64_t(1) << 31);
}

hipError_t launch_gemm_f16(const f16* A, const f16* B, f16* C, int M, int N, int K, GemmOut out,
                           int cus, hipStream_t stream) {
    if (!gemm_f16_fits(M, N, K)) return hipErrorInvalidValue;
    const int64_t ncu = std::max(1, cus);
    GemmCall c{A, B, C, M, N, K, out, ncu, stream};
    // QASR_GEMM_TILE = 1..7 forces that tile for all rows (the tests compare
    // them; one whose kernel needs more K steps than there are is not forced).
    const char* forced = std::getenv("QASR_GEMM_TILE");
    const int f = forced ? std::atoi(forced) : 0;
    if (f >= 1 && f <= kNumTiles && K / kBK >= kTiles[f - 1].min_steps) return launch_tile(kTiles[f - 1], c);
    // One tile for all rows, or a tile's whole rounds for the first rows and a
    // second launch with the best tile for the rest, whichever the model calls
    // fastest: 4,269 rows of gate|up are 816 tiles of 256 x 256, 3.2 rounds
    // that take four (199 us); three full rounds over 4,096 rows and small
    // tiles for the other 173 take 189.  Every tile sums each output
    // over K in the same order, so the choice never changes a bit.
    float best_us = 0.0f;
    const Tile* t1 = &best_tile(M, N, K, ncu, &best_us);
    const Tile* t2 = nullptr;
    int m1 = M;
    for (const Tile& c1 : kTiles) {
        if (K / kBK < c1.min_steps) continue;
        const int64_t per_row = N / c1.bn, full = (int64_t)c1.occ * ncu;
        const int64_t rounds = (M / c1.bm) * per_row / full;
        const int64_t rows = rounds * full / per_row * c1.bm;
        if (rows <= 0 || rows >= M) continue;
        float rest = 0.0f;
        const Tile& c2 = best_tile(M - rows, N, K, ncu, &rest);
        const float t = tile_us(c1, rows, N, K, ncu) + rest + kSecondLaunchUs;
        if (t < best_us) {
            best_us = t;
            t1 = &c1;
            t2 = &c2;
            m1 = (int)rows;
        }
    }
    c.M = m1;
    const hipError_t e = launch_tile(*t1, c);
    if (e != hipSuccess || !t2) return e;
    c.A = A + (int64_t)m1 * K;
    c.C = C + (int64_t)m1 * (out == kGemmGlu ? N / 2 : N);
    c.M = M - m1;
    return launch_tile(*t2, c);
}

}  // namespace qasr
