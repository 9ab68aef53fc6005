// bf16 FC on a second operand that is used once, straight from its row-major form: C = PP(A · B) with B [K, N] or [N, K].
//
// Stands in for amx_kernel::Matmul with constB = false (include/kernels_amx.hpp:1045-1315).  A B that is new at every call
// gains nothing from being packed first: packing reads and writes all of it, and the GEMM behind it reads it again.
//
// What bounds it: HBM, as long as the rows of A are few.  A wavefront owns a strip of 128 columns and streams its share of
// K through registers, 32 of k (8 KiB; from [N, K] 64 of k) at a time; nothing goes through LDS on the way.  From [K, N] a
// lane loads 16 bytes (8 columns) of 8 consecutive rows, so that 16 lanes cover 256 contiguous bytes of a row, and turns the 8 x 8 square in
// registers (32 v_perm per 8 KiB, everything else is the naming of registers): MFMA i then multiplies the columns
// 8 r + i, r = 0 ... 15, of the strip.  From [N, K] a lane's 16 bytes are 8 of k of one column already and MFMA i takes
// the columns 16 i + r.  B is the first operand of the 16x16x32 MFMA, 16 rows of A the second; rows of A come from the
// L2 (they are small).  K is split over the wavefronts of a workgroup (summed through LDS) and over up to 16 workgroups
// (summed through a workspace, in slice order, by the one that arrives last).
// Measured against packing first: at unpacked_takes.
#include "common.hpp"

namespace mmx {

struct UnpackedArgs {
    const char* A;
    int64_t lda;  // bytes
    const char* B;
    int64_t ldb;  // bytes
    int M, K, N;
    int mtiles, units, S;  // units = column strips x row tiles x K slices
    char* parts;           // S > 1: the slices' sums
    uint32_t* cnt;         // S > 1: one arrival counter per tile, zero between launches
    Epilogue ep;
};

constexpr int STRIP = 128;           // columns of a workgroup
constexpr int RED_ROW = STRIP + 4;   // floats; the pad spreads 16 rows over the banks
constexpr int MAX_SLICES = 16;
// No launch asks for more than WS_STANDARD_BYTES or uses more: a larger answer would replace the stream's buffer, which a graph
// captured earlier may still write to, and the slices of a call would depend on its history.  (That takes slices from wide
// results only, where the CUs have strips enough: 128 x 8192 x 50304 334 us unsplit, 338 in four.)

// 16 bytes from any address (the hardware takes them at any)
typedef u32x4 __attribute__((aligned(1))) u32x4_any;
__device__ __forceinline__ u32x4 load16(const char* base, uint32_t off) { return *reinterpret_cast<const u32x4_any*>(base + off); }
__device__ __forceinline__ u32x4 stream16(const char* base, uint32_t off) {
    return __builtin_nontemporal_load(reinterpret_cast<const u32x4_any*>(base + off));
}

// One step of a wavefront: 32 of k from [K, N]; 64 of k from [N, K], where that is the 128-byte line of a column: its two
// halves are asked for one right behind the other, so that the second finds the line on its way.
template <bool TR>
constexpr int KSTEP = TR ? 64 : 32;

template <bool TR, int MB>
struct Step {
    u32x4 b[KSTEP<TR> / 4];
    u32x4 a[KSTEP<TR> / 32][MB];
};

// half: the last step of an [N, K] holds 32 of k only (the other half repeats the first and is not multiplied)
template <bool TR, int MB>
__device__ __forceinline__ void load_step(Step<TR, MB>& s, const char* B, int64_t ldb, const uint32_t (&boff)[TR ? 8 : 1], const char* A,
                                          const uint32_t (&aoff)[MB], int step, bool half) {
    const char* aa = A + (int64_t)step * (KSTEP<TR> * 2);
    if constexpr (TR) {
        const char* bb = B + (int64_t)step * (KSTEP<TR> * 2);
        const int second = half ? 0 : 64;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            s.b[2 * i] = load16(bb, boff[i]);
            s.b[2 * i + 1] = load16(bb + second, boff[i]);
        }
#pragma unroll
        for (int mb = 0; mb < MB; mb++) {
            s.a[0][mb] = load16(aa, aoff[mb]);
            s.a[1][mb] = load16(aa + second, aoff[mb]);
        }
    } else {
        const char* bb = B + (int64_t)step * KSTEP<TR> * ldb;
#pragma unroll
        for (int j = 0; j < 8; j++) s.b[j] = stream16(bb + j * ldb, boff[0]);
#pragma unroll
        for (int mb = 0; mb < MB; mb++) s.a[0][mb] = load16(aa, aoff[mb]);
    }
}

template <bool TR, int MB>
__device__ __forceinline__ void multiply_step(const Step<TR, MB>& s, f32x4 (&acc)[8][MB], bool half) {
#pragma unroll
    for (int h = 0; h < KSTEP<TR> / 32; h++) {
        if (h && half) break;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            u32x4 w;
            if constexpr (TR) {
                w = s.b[2 * i + h];
            } else {
#pragma unroll
                for (int p = 0; p < 4; p++)  // rows 2 p and 2 p + 1 of column i: halves of dword i / 2
                    w[p] = __builtin_amdgcn_perm(s.b[2 * p + 1][i >> 1], s.b[2 * p][i >> 1], (i & 1) ? 0x07060302u : 0x05040100u);
            }
#pragma unroll
            for (int mb = 0; mb < MB; mb++)
                acc[i][mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w), __builtin_bit_cast(bf16x8, s.a[h][mb]), acc[i][mb], 0, 0, 0);
        }
    }
}

// TR: B is [N, K]; MB: blocks of 16 rows of A per workgroup; NW: wavefronts.
// (Two workgroups of 64 rows per CU from [K, N]: left to itself the compiler took 374 registers for one, 186 + 188; from [N, K]
// it needs more than the 256 that two would have.  With the stores of four columns at once 65 x 64 x 65536 32 -> 16 us.)
template <bool TR, int MB, int NW>
__global__ __launch_bounds__(64 * NW, MB == 1 && !TR ? 4 : (NW == 8 || !TR ? 2 : 1)) void unpacked_kernel(const UnpackedArgs s) {
    __shared__ __attribute__((aligned(16))) float red[NW][16][RED_ROW];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, g = lane >> 4;
    // workgroups are dealt to the 8 XCDs in turn: one XCD gets neighbouring units, and the row tiles that read the same
    // piece of B are neighbours (m fastest), so that all but one of them find it in the XCD's L2
    const int per_xcd = gridDim.x >> 3;
    const int unit = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
    if (unit >= s.units) return;
    const int mt = unit % s.mtiles, rest = unit / s.mtiles;
    const int slice = rest % s.S, strip = rest / s.S;
    const int m0 = mt * 16 * MB, n0 = strip * STRIP;

    const int steps = (s.K + KSTEP<TR> - 1) / KSTEP<TR>;
    const int per_slice = (steps + s.S - 1) / s.S;
    const int s_lo = slice * per_slice, s_hi = min(s_lo + per_slice, steps);
    const int per_wave = (s_hi - s_lo + NW - 1) / NW;
    const int w_lo = s_lo + wave * per_wave, w_hi = min(w_lo + per_wave, s_hi);

    // columns beyond N and rows beyond M read the last one again; what comes of them is not stored
    uint32_t boff[TR ? 8 : 1], aoff[MB];
    const char* B;
    if constexpr (TR) {
        B = s.B + (int64_t)n0 * s.ldb;
#pragma unroll
        for (int i = 0; i < 8; i++) boff[i] = (uint32_t)(min(n0 + 16 * i + r, s.N - 1) - n0) * (uint32_t)s.ldb + 16 * g;
    } else {
        B = s.B;
        boff[0] = (uint32_t)(8 * g) * (uint32_t)s.ldb + (uint32_t)min(n0 + 8 * r, s.N - 8) * 2;
    }
    const char* A = s.A + (int64_t)m0 * s.lda;
#pragma unroll
    for (int mb = 0; mb < MB; mb++) aoff[mb] = (uint32_t)(min(m0 + 16 * mb + r, s.M - 1) - m0) * (uint32_t)s.lda + 16 * g;

    f32x4 acc[8][MB];
#pragma unroll
    for (int i = 0; i < 8; i++)
#pragma unroll
        for (int mb = 0; mb < MB; mb++) acc[i][mb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    // Two steps in flight per wavefront; a step beyond the share is the last one again and is not multiplied.  Each share
    // starts at another place and wraps around: with sizes that are powers of two the shares would otherwise walk the same
    // memory channels in step (8192 x 8192 in 4 slices, one row of A: 33.7 us without, 27.1 with; other sizes level).
    if (w_lo < w_hi) {
        const int len = w_hi - w_lo, rot = (wave + slice + strip) % len;
        auto at = [&](int t) {
            t = min(t, w_hi - 1) + rot;
            return t >= w_hi ? t - len : t;
        };
        auto half = [&](int step) { return TR && step * KSTEP<TR> + 32 == s.K; };
        Step<TR, MB> s0, s1;
        int t0 = at(w_lo), t1 = 0;
        load_step<TR, MB>(s0, B, s.ldb, boff, A, aoff, t0, half(t0));
        int t = w_lo;
        for (; t + 1 < w_hi; t += 2) {
            t1 = at(t + 1);
            load_step<TR, MB>(s1, B, s.ldb, boff, A, aoff, t1, half(t1));
            __builtin_amdgcn_sched_barrier(0);
            multiply_step<TR, MB>(s0, acc, half(t0));
            __builtin_amdgcn_sched_barrier(0);
            t0 = at(t + 2);
            load_step<TR, MB>(s0, B, s.ldb, boff, A, aoff, t0, half(t0));
            __builtin_amdgcn_sched_barrier(0);
            multiply_step<TR, MB>(s1, acc, half(t1));
            __builtin_amdgcn_sched_barrier(0);
        }
        if (t < w_hi) multiply_step<TR, MB>(s0, acc, half(t0));
    }

    // sums over the wavefronts, one block of 16 rows at a time: PER runs of four columns per thread
    constexpr int PER = 8 / NW;
    f32x4 sum[MB][PER];
#pragma unroll
    for (int mb = 0; mb < MB; mb++) {
        if (mb) __syncthreads();
        // accumulator v of MFMA i: column 8 (4 g + v) + i of the strip from [K, N], 16 i + 4 g + v from [N, K]; row r
#pragma unroll
        for (int i = 0; i < 8; i++) {
            if constexpr (TR) {
                *reinterpret_cast<f32x4*>(&red[wave][r][16 * i + 4 * g]) = acc[i][mb];
            } else if (i % 4 == 0) {
#pragma unroll
                for (int v = 0; v < 4; v++)
                    *reinterpret_cast<f32x4*>(&red[wave][r][8 * (4 * g + v) + i]) =
                        f32x4{acc[i][mb][v], acc[i + 1][mb][v], acc[i + 2][mb][v], acc[i + 3][mb][v]};
            }
        }
        __syncthreads();
#pragma unroll
        for (int p = 0; p < PER; p++) {
            const int idx = tid + 64 * NW * p;
            f32x4 t = *reinterpret_cast<const f32x4*>(&red[0][idx >> 5][4 * (idx & 31)]);
#pragma unroll
            for (int w = 1; w < NW; w++) t += *reinterpret_cast<const f32x4*>(&red[w][idx >> 5][4 * (idx & 31)]);
            sum[mb][p] = t;
        }
    }

    if (s.S > 1) {
        // The slice's sums go to the workspace at device scope (sc1: to the level that all XCDs share); once they have been
        // acknowledged the slice counts itself in with an atomicInc that wraps to zero at the last arrival.  The last one
        // adds the sums up in slice order, so the result does not depend on who came last; nobody waits.
        constexpr int AUX_SC1 = 16;
        constexpr int UNIT = MB * 16 * STRIP * 4;  // bytes of one slice's sums
        const int tile = strip * s.mtiles + mt;
        __amdgpu_buffer_rsrc_t parts =
            __builtin_amdgcn_make_buffer_rsrc(s.parts + (int64_t)tile * s.S * UNIT, 0, s.S * UNIT, 0x00020000);
#pragma unroll
        for (int mb = 0; mb < MB; mb++)
#pragma unroll
            for (int p = 0; p < PER; p++)
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, sum[mb][p]), parts,
                                                       slice * UNIT + ((mb * PER + p) * 64 * NW + tid) * 16, 0, AUX_SC1);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();  // every wavefront's stores are through, and the reduction scratch is free
        volatile uint32_t* flag = reinterpret_cast<volatile uint32_t*>(&red[0][0][0]);
        if (tid == 0) *flag = atomicInc(s.cnt + tile, (uint32_t)s.S - 1u);
        __syncthreads();
        if (*flag != (uint32_t)s.S - 1u) return;
        asm volatile("" ::: "memory");
        f32x4 total[MB][PER];
        for (int sl = 0; sl < s.S; sl++) {
#pragma unroll
            for (int mb = 0; mb < MB; mb++)
#pragma unroll
                for (int p = 0; p < PER; p++) {
                    const f32x4 v = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                                  parts, sl * UNIT + ((mb * PER + p) * 64 * NW + tid) * 16, 0, AUX_SC1));
                    total[mb][p] = sl == 0 ? v : total[mb][p] + v;
                }
        }
#pragma unroll
        for (int mb = 0; mb < MB; mb++)
#pragma unroll
            for (int p = 0; p < PER; p++) sum[mb][p] = total[mb][p];
    }

    // The post-op runs in a loop that is not unrolled, over sums handed on through LDS: its code is fetched cold by every
    // launch, and 4 MB PER copies of the GELU in line cost the small shapes more than the multiplication.
    f32x4* mine = reinterpret_cast<f32x4*>(&red[0][0][0]) + tid;  // 64 NW apart, each thread its own
    __syncthreads();
#pragma unroll
    for (int mb = 0; mb < MB; mb++)
#pragma unroll
        for (int p = 0; p < PER; p++) mine[(mb * PER + p) * 64 * NW] = sum[mb][p];
    const Epilogue& ep = s.ep;
#pragma unroll 1
    for (int k = 0; k < MB * PER; k++) {
        const int idx = tid + 64 * NW * (k % PER);
        const int n = n0 + 4 * (idx & 31), m = m0 + 16 * (k / PER) + (idx >> 5);
        if (n >= s.N || m >= s.M) continue;
        const int live = min(4, s.N - n);
        const f32x4 t = mine[k * 64 * NW];
        float o[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int c = n + (e < live ? e : 0);
            float v = t[e];
            if (ep.steps & MMX_PP_DEQUANT) v = v * (ep.deq_oc ? ep.deq_oc[c] : ep.deq);
            if (ep.steps & MMX_PP_BIAS) v = v + ep.bias[c];
            o[e] = v;
        }
        if (ep.steps & MMX_PP_GELU) {
#pragma unroll
            for (int e = 0; e < 4; e++) o[e] = gelu_erf_minimax(o[e]);
        }
        if (ep.steps & MMX_PP_QUANT) {
#pragma unroll
            for (int e = 0; e < 4; e++) o[e] = o[e] * (ep.q_oc ? ep.q_oc[n + (e < live ? e : 0)] : ep.q);
        }
        char* row = ep.C + (int64_t)m * ep.ldc;
        if (live == 4) {  // one store, at whatever address a row of C has
            if (ep.out_dtype == MMX_F32) {
                __builtin_memcpy(__builtin_assume_aligned(row + (int64_t)n * 4, 4), o, 16);
            } else if (ep.out_dtype == MMX_BF16) {
                const uint32_t w[2] = {(uint32_t)to_bf16(o[0]) | (uint32_t)to_bf16(o[1]) << 16, (uint32_t)to_bf16(o[2]) | (uint32_t)to_bf16(o[3]) << 16};
                __builtin_memcpy(__builtin_assume_aligned(row + (int64_t)n * 2, 2), w, 8);
            } else {
                const uint32_t w = to_s8_sat_x4(o[0], o[1], o[2], o[3]);
                __builtin_memcpy(row + n, &w, 4);
            }
            continue;
        }
#pragma unroll 1
        for (int e = 0; e < live; e++) {
            if (ep.out_dtype == MMX_BF16) reinterpret_cast<uint16_t*>(row)[n + e] = to_bf16(o[0]);
            else if (ep.out_dtype == MMX_I8) reinterpret_cast<int8_t*>(row)[n + e] = to_s8_sat(o[0]);
            else reinterpret_cast<float*>(row)[n + e] = o[0];
            o[0] = o[1], o[1] = o[2], o[2] = o[3];
        }
    }
}

// How a call is shared out: blocks of 16 rows of A per workgroup, and K slices.
struct Share {
    int row_blocks, slices;
};
static int row_tiles(int M, int row_blocks) { return (M + 16 * row_blocks - 1) / (16 * row_blocks); }
static int tile_count(int M, int N, int row_blocks) { return (N + STRIP - 1) / STRIP * row_tiles(M, row_blocks); }
static size_t slice_sums(int tiles, int row_blocks) { return (size_t)tiles * row_blocks * 16 * STRIP * 4; }
static size_t workspace_of(int M, int N, Share h) {
    return h.slices > 1 ? WS_COUNTER_BYTES + slice_sums(tile_count(M, N, h.row_blocks), h.row_blocks) * h.slices : 0;
}

// The least of an estimate in us, fitted to 20 000 timings (K 32 ... 11008, N 64 ... 65536, M 1 ... 256, both orders of B, every
// number of blocks, ten numbers of slices); over those its choice takes 2.3 % longer than the best one on average, 18 % at the
// 99th percentile.
//   busy: a workgroup alone on its CU takes `first` (start, sums over the wavefronts, post-op) and `step` for a step of each
//   wavefront (from [N, K] a step is twice as long and comes in pieces of 64 bytes); each further one of the CU adds `next`.
//   stream: the chip takes B in at 5 TB/s, and the row tiles behind the first read it again, mostly from the L2.
//   The two hide behind each other in part; each slice adds to the combination.
// Fewer rows per workgroup mean more of them and less for each to do one after another, more rows fewer passes over B:
// 64 x 512 x 512 from [K, N] 10.3 us in workgroups of 64 rows, 5.8 of 16; 64 x 512 x 65536 22 and 38.
static Share choose_share(int M, int K, int N, int transpose, size_t ws_bytes) {
    if (ws_bytes > WS_STANDARD_BYTES) ws_bytes = WS_STANDARD_BYTES;
    static const struct { int row_blocks; float first, step, next; } forms[2][3] = {
        {{1, 0.6f, 1.85f, 1.35f}, {2, 4.9f, 1.55f, 4.6f}, {4, 7.9f, 1.05f, 6.1f}}, {{1, 0.2f, 3.8f, 0.9f}, {2, 0.8f, 5.2f, 3.0f}, {4, 7.2f, 2.45f, 10.6f}}};
    const int steps = transpose ? (K + 63) / 64 : K / 32, cus = num_cus();
    Share best = {4, 1};
    float best_us = 0.0f;
    for (const auto& f : forms[transpose ? 1 : 0]) {
        if ((f.row_blocks == 1 && M > 64) || (f.row_blocks > 1 && M <= 8 * f.row_blocks)) continue;
        const int nw_log2 = f.row_blocks == 4 ? 2 : 3, nw = 1 << nw_log2, tiles = tile_count(M, N, f.row_blocks);
        const size_t slice_bytes = slice_sums(tiles, f.row_blocks);
        if (f.row_blocks == 1 && M > 32 && tiles > 2 * cus) continue;  // (33 x 512 x 131072 from [N, K] 74 us against 54 with 64 rows)
        const float stream_us = 0.8f + (float)K * N * 2e-6f * (1 / 4.35f + (row_tiles(M, f.row_blocks) - 1) / 57.0f);
        int steps_before = 0;
        for (int S = 1; S <= MAX_SLICES; S++) {
            const int per_slice = (steps + S - 1) / S, wave_steps = (per_slice + nw - 1) >> nw_log2;
            if (S > 1 && (2 * per_slice < nw || tiles > WS_MAX_TILES || 2 * tiles * S > 5 * cus || WS_COUNTER_BYTES + slice_bytes * S > ws_bytes)) break;
            if (wave_steps == steps_before || (S - 1) * per_slice >= steps) continue;  // (nothing gained by the slice, or nothing in it)
            steps_before = wave_steps;
            const float work_us = f.step * wave_steps;
            const float busy_us = f.first + work_us + ((tiles * S + cus - 1) / cus - 1) * (f.next + work_us);
            const float us = sqrtf(busy_us * busy_us + stream_us * stream_us) + (S > 1 ? 0.9f + 0.26f * S : 0.0f);
            if (best_us == 0.0f || us < best_us) best = {f.row_blocks, S}, best_us = us;
        }
    }
    return best;
}

// What the kernel can take: whole steps of k, whole pieces of 16 bytes, lane offsets of 32 bits (64 rows of A, 128 of B).
bool unpacked_can(int M, int K, int N, int64_t lda, int64_t ldb, int transpose) {
    return M > 0 && K >= 32 && K % 32 == 0 && N >= 8 && (transpose || N % 8 == 0) && lda <= (1 << 24) && ldb <= (1 << 23);
}

// Whether a call is better off with it than with packing B first.  Device time, pack + GEMM -> this kernel, B new at every
// call: from [K, N] 8192 x 8192 at M = 1 / 64 / 256 73 / 73 / 90 -> 27 / 37 / 84 us, 4096 x 4096 at M = 16 / 128 24 / 28 -> 13 / 20,
// 512 x 640 at M = 64 / 128 9.7 / 9.6 -> 5.9 / 7.4; from [N, K] 8192 x 8192 at M = 1 / 64 / 128 69 / 69 / 74 -> 32 / 37 / 54,
// 4096 x 4096 at M = 16 / 128 24 / 28 -> 12 / 23, 512 x 640 at M = 64 / 128 9.1 / 9.4 -> 7.1 / 8.7.
// (The product behind a packing ran on the tile kernels when this was measured.  With the small tiles behind it, over 260 shapes of
// 33 to 256 rows the way taken is 1.03 of the better one on average: level from [K, N], 1.05 and 1.08 from [N, K] for 65 to 128
// and 129 to 256 rows, at most 1.6, 140 x 608 x 4448 15.2 against 9.5 us: profiles/unpacked_against_packing.txt.)
// Over 4032 shapes (K 32 ... 11008, N 64 ... 131072, M 1 ... 256) the way taken is on average 0.70 of packing, at most 1.15 of it
// (a microsecond, 1 x 4096 x 256 from [N, K] 8.4 and 9.5).  Packing is the faster way
//   where many workgroups of 64 rows have little to multiply (96 x 64 x 65536 15.7 against 16.2 us, from [N, K], whose form takes
//   a CU alone, 17.4 against 24.8), or come one and a half to a CU over a deep K (128 x 2560 x 24576 from [N, K] 62 against 73);
//   for more than 192 rows of a deep K if its slices leave CUs idle (256 x 11008 x 6144 99 against 113);
//   from [N, K] for more than 128 rows, and for a few strips deeper than 8192 (16 x 11008 x 256 14 against 17).
bool unpacked_takes(int M, int K, int N, int64_t lda, int64_t ldb, int transpose) {
    if (!unpacked_can(M, K, N, lda, ldb, transpose) || M > 256) return false;
    const int tiles = tile_count(M, N, 4), cus = num_cus();
    if (transpose) {
        if (M <= 32) return N > 3 * STRIP || K <= 8192;
        return M <= 64 || (M <= 128 && (tiles <= cus || (K >= 2048 && tiles >= 2 * cus)));
    }
    if (M <= 128) return M <= 64 || tiles <= 2 * cus || K >= 128;
    if (tiles > cus) return false;
    return M <= 192 || K <= 4096 || 4 * tiles <= cus || 10 * (cus / tiles * tiles) >= 9 * cus;
}

size_t unpacked_workspace_bytes(int M, int K, int N, int transpose) {
    return workspace_of(M, N, choose_share(M, K, N, transpose, WS_STANDARD_BYTES));
}

int launch_unpacked(const void* A, int64_t lda, const void* B, int64_t ldb, int transpose, int M, int K, int N, const Epilogue& ep, char* ws,
                    size_t ws_bytes, hipStream_t st) {
    const Share h = choose_share(M, K, N, transpose, ws ? ws_bytes : 0);
    UnpackedArgs s;
    s.A = static_cast<const char*>(A);
    s.lda = M == 1 ? 0 : lda;
    s.B = static_cast<const char*>(B);
    s.ldb = ldb;
    s.M = M, s.K = K, s.N = N;
    s.mtiles = row_tiles(M, h.row_blocks);
    s.S = h.slices;
    s.units = tile_count(M, N, h.row_blocks) * s.S;
    s.cnt = reinterpret_cast<uint32_t*>(ws);
    s.parts = ws ? ws + WS_COUNTER_BYTES : nullptr;
    s.ep = ep;
    const dim3 grid((s.units + 7) / 8 * 8);
    char name[64];
    snprintf(name, sizeof name, "unpacked_%s_rows%d_ksplit%d", transpose ? "nk" : "kn", 16 * h.row_blocks, s.S);
    note_kernel(name);
    if (h.row_blocks == 1) {
        if (transpose) unpacked_kernel<true, 1, 8><<<grid, 512, 0, st>>>(s);
        else unpacked_kernel<false, 1, 8><<<grid, 512, 0, st>>>(s);
    } else if (h.row_blocks == 2) {
        if (transpose) unpacked_kernel<true, 2, 8><<<grid, 512, 0, st>>>(s);
        else unpacked_kernel<false, 2, 8><<<grid, 512, 0, st>>>(s);
    } else {
        if (transpose) unpacked_kernel<true, 4, 4><<<grid, 256, 0, st>>>(s);
        else unpacked_kernel<false, 4, 4><<<grid, 256, 0, st>>>(s);
    }
    return check_hip(hipGetLastError(), "unpacked_kernel launch");
}

}  // namespace mmx
