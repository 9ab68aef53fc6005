// One-off weight preparation kernels: repack to MFMA-fragment order, gate/up interleave,
// per-tensor int8 weight compression, packed int8 -> packed bf16.
//
// Stands in for amx_kernel::repackB_1x2 (include/kernels_amx.hpp:761-816), MLP::setup's gate/up
// interleave (tests/amx-mlp.cpp:758-765) and the weight compression inside
// amx_kernel::Matmul<bf16,int8,float> (include/kernels_amx.hpp:1363-1377, 465-523).
#include <type_traits>

#include "common.hpp"

namespace mmx {

// Packed layout: [panel = n/32][f = k/KS][lane][16 B], KS = 32/ES elements, lane = n%32 + 32*((k%KS)/(KS/2)); K is
// padded with zeros to 128 bytes per column, N to 32 columns.  Four fragments (4 KiB of a panel) are 128 bytes of K of
// 32 columns: the unit that both kernels below work in.
//
// What bounds them is memory: every byte is read once and written once, so all that matters is that both sides move
// whole 128-byte lines and that enough of them are in flight.  (One thread per 16-byte slot, gathering its elements one
// by one, asked for 32 bytes of a line per row and instruction from [N, K] and for two bytes per lane from [K, N].)

// All of a row of W to 2 W - 1 bytes, by W bytes from either end; zero behind it.
template <int W>
__device__ __forceinline__ u32x4 load_short_row(const char* row, int len) {
    uint64_t head = 0, tail = 0;
    __builtin_memcpy(&head, __builtin_assume_aligned(row, 1), W);
    __builtin_memcpy(&tail, __builtin_assume_aligned(row + len - W, 1), W);
    tail = (tail >> (8 * (2 * W - len) - 1)) >> 1;  // what lies behind the first W bytes, if anything
    const uint64_t lo = W == 8 ? head : head | tail << (8 * (W & 7)), hi = W == 8 ? tail : 0;
    return u32x4{(uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32)};
}

// N times 16 bytes from byte `at` of the rows at row(0) ... row(N - 1), each of len bytes.  What lies past the end, and a row
// that is not live(i), is zero and not touched.  No load waits for another; what moves the bytes down runs behind all of them,
// and only where the rows end inside the 16.  (Element by element behind tests, each load waited for the one before it: bytes
// from [K, N], K = 512, N = 3001 9.4 us against 4.5 for a thread per slot.)
// RowLength: what the host knows of len (the code for rows shorter than 16 bytes takes registers).
enum RowLength { ANY_ROW, SHORT_ROW, LONG_ROW };  // any, below 16 bytes, 16 and up
template <int ES, RowLength LEN = ANY_ROW, int N, typename Row, typename Live>
__device__ __forceinline__ void load16_rows(u32x4 (&v)[N], int64_t at, int64_t len, Row&& row, Live&& live) {
#pragma unroll
    for (int i = 0; i < N; i++) v[i] = u32x4{0u, 0u, 0u, 0u};
    typedef typename std::conditional<ES == 2, uint16_t, uint8_t>::type elem;
    if (at >= len) return;
    if (LEN == LONG_ROW || (LEN == ANY_ROW && len >= 16)) {
        const int64_t from = at < len - 16 ? at : len - 16;
#pragma unroll
        for (int i = 0; i < N; i++)
            if (live(i)) __builtin_memcpy(&v[i], __builtin_assume_aligned(row(i) + from, ES), 16);
        if (from < at) {
#pragma unroll
            for (int i = 0; i < N; i++) v[i] = settle16_in_row(v[i], (int)(at - from), 16);
        }
    } else if constexpr (LEN == SHORT_ROW) {
        auto all = [&](auto w) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < N; i++)
                if (live(i)) v[i] = load_short_row<decltype(w)::value>(row(i), (int)len);
        };
        if (len >= 8) all(std::integral_constant<int, 8>{});
        else if (len >= 4) all(std::integral_constant<int, 4>{});
        else if (len >= 2) all(std::integral_constant<int, 2>{});
        else all(std::integral_constant<int, 1>{});
    } else {
#pragma unroll
        for (int i = 0; i < N; i++)
            if (live(i)) {
                alignas(16) elem e[16 / ES];
#pragma unroll
                for (int j = 0; j < 16 / ES; j++) e[j] = j * ES < len ? reinterpret_cast<const elem*>(row(i))[j] : (elem)0;
                __builtin_memcpy(&v[i], e, 16);
            }
    }
}
// the same where all of it is there
template <int ES>
__device__ __forceinline__ u32x4 load16(const char* p) {
    u32x4 v;
    __builtin_memcpy(&v, __builtin_assume_aligned(p, ES), 16);
    return v;
}

// [N, K] (a row per column of B): a slot is 16 consecutive bytes of a row, so nothing has to be rearranged in registers.
// A wavefront takes 128 bytes of K of 32 rows: load i covers 8 whole lines (8 rows x 128 bytes), and the lane's 16
// bytes, chunk c of row r, belong at (c / 2) KiB + (r + 32 (c % 2)) * 16 of the panel's 4 KiB - for one c the 8 rows of
// a store are 128 consecutive bytes, whole lines again.  UNR such units per wavefront keep 4 UNR loads in flight.
// PAIR: gate and up interleaved by panel, panel 2p = gate columns [32p, 32p + 32), panel 2p + 1 = up's.
// N = 11008, K = 4096, against a thread per slot: bf16 82 -> 31 us (5.8 TB/s moved), bytes 91 -> 16, gate and up 157 -> 67.
template <int ES, int UNR, bool PAIR, RowLength LEN>
__global__ __launch_bounds__(256) void repack_rows_kernel(const char* __restrict__ B0, const char* __restrict__ B1, int64_t ldb, int kbytes,
                                                          int N, char* __restrict__ out, int kunits, int groups, int flip) {
    const int lane = threadIdx.x & 63;
    const int panel = blockIdx.x / groups;
    const int ku0 = ((blockIdx.x - panel * groups) * 4 + (threadIdx.x >> 6)) * UNR;
    const char* const B = PAIR && (panel & 1) ? B1 : B0;
    const int n0 = (PAIR ? panel >> 1 : panel) * 32;
    const int r8 = lane >> 3, c = lane & 7;
    u32x4 v[UNR][4];
    char* const o = out + ((int64_t)panel * kunits + ku0) * 4096 + (c >> 1) * 1024 + (32 * (c & 1) + r8) * 16;
    auto store = [&](bool whole) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < UNR; u++) {
            if (!whole && ku0 + u >= kunits) break;
            const int kb = (ku0 + u) * 128 + c * 16;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                u32x4 w = v[u][i];
                if (ES == 1 && flip && n0 + 8 * i + r8 < N) {  // (the padding stays zero)
#pragma unroll
                    for (int e = 0; e < 16; e++)
                        if (kb + e < kbytes) w[e >> 2] ^= 0x80u << (8 * (e & 3));
                }
                *reinterpret_cast<u32x4*>(o + u * 4096 + i * 128) = w;
            }
        }
    };
    // (the stores are in both branches, so that each waits for its own load only: behind the join they waited for all,
    // 3001 x 8192 bf16 17.9 us against 16.5)
    if (n0 + 32 <= N && (ku0 + UNR) * 128 <= kbytes) {
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int u = 0; u < UNR; u++) v[u][i] = load16<ES>(B + (int64_t)(n0 + 8 * i + r8) * ldb + (ku0 + u) * 128 + c * 16);
        __builtin_amdgcn_sched_barrier(0);  // (neighbouring lines of a row one right behind the other: unaligned rows share one)
        store(true);
    } else {
#pragma unroll
        for (int u = 0; u < UNR; u++)
            if (ku0 + u < kunits)
                load16_rows<ES, LEN>(v[u], (ku0 + u) * 128 + c * 16, kbytes, [&](int i) { return B + (int64_t)(n0 + 8 * i + r8) * ldb; },
                                     [&](int i) { return n0 + 8 * i + r8 < N; });
        store(false);
    }
}

// [K, N]: a slot's elements lie a row apart, so a lane reads a square - EL rows of 16 bytes, EL = 16 / ES consecutive k
// of as many columns - and transposes it in registers (v_perm_b32: 32 of them for 8 x 8 bf16, 128 for 16 x 16 bytes).
// A load covers 8 rows x 128 bytes.  The EL slots of a lane are those of neighbouring columns, so a direct store would
// scatter 16-byte pieces; the wavefront's slots (8 EL columns x 128 bytes of K) go through its own part of LDS and leave
// as whole fragments.  LDS positions are XORed with the bits above the low four, which spreads the lanes of a write over
// the banks.
// 10240 x 10240, against a thread per slot: bf16 99 -> 90 us (4.7 TB/s moved), bytes 122 -> 35.
template <int ES, RowLength LEN>
__global__ __launch_bounds__(ES == 2 ? 256 : 64) void repack_cols_kernel(const char* __restrict__ B, int64_t ldb, int K, int N,
                                                                         char* __restrict__ out, int kunits, int npanels, int flip) {
    constexpr int EL = 16 / ES;               // columns and k of a lane's square
    constexpr int PANELS = 8 * EL / 32;       // panels per wavefront: 2 (bf16) or 4 (bytes)
    constexpr int WAVES = ES == 2 ? 4 : 1;
    __shared__ __attribute__((aligned(16))) u32x4 slots[WAVES * PANELS * 256];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int ku = blockIdx.x % kunits, pg = (blockIdx.x / kunits) * WAVES + wave;
    const int ng = lane & 7, kg = lane >> 3;
    const int n = pg * (8 * EL) + ng * EL, k = ku * (8 * EL) + kg * EL;
    u32x4 row[EL];
    if ((pg + 1) * (8 * EL) <= N && (ku + 1) * (8 * EL) <= K) {
#pragma unroll
        for (int e = 0; e < EL; e++) row[e] = load16<ES>(B + (int64_t)(k + e) * ldb + (int64_t)n * ES);
    } else {
        load16_rows<ES, LEN>(row, (int64_t)n * ES, (int64_t)N * ES, [&](int e) { return B + (int64_t)(k + e) * ldb; },
                        [&](int e) { return k + e < K; });
    }
    if (ES == 1 && flip) {
#pragma unroll
        for (int e = 0; e < EL; e++)
#pragma unroll
            for (int i = 0; i < 16; i++)
                if (k + e < K && n + i < N) row[e][i >> 2] ^= 0x80u << (8 * (i & 3));
    }
    u32x4* const mine = slots + wave * PANELS * 256;
    auto put = [&](int j, u32x4 slot) {  // the slot of column n + j
        const int col = ng * EL + j;
        const int at = ((col >> 5) * 4 + (kg >> 1)) * 64 + (kg & 1) * 32 + (col & 31);
        mine[at ^ (((at >> 4) ^ (at >> 8)) & 15)] = slot;
    };
    if constexpr (ES == 2) {
#pragma unroll
        for (int d = 0; d < 4; d++) {
            u32x4 lo, hi;
#pragma unroll
            for (int p = 0; p < 4; p++) {
                lo[p] = __builtin_amdgcn_perm(row[2 * p + 1][d], row[2 * p][d], 0x05040100u);
                hi[p] = __builtin_amdgcn_perm(row[2 * p + 1][d], row[2 * p][d], 0x07060302u);
            }
            put(2 * d, lo);
            put(2 * d + 1, hi);
        }
    } else {
#pragma unroll
        for (int d = 0; d < 4; d++) {
            u32x4 s[4];
#pragma unroll
            for (int p = 0; p < 4; p++) {
                const uint32_t a = row[4 * p][d], b = row[4 * p + 1][d], x = row[4 * p + 2][d], y = row[4 * p + 3][d];
                const uint32_t ab01 = __builtin_amdgcn_perm(b, a, 0x05010400u), ab23 = __builtin_amdgcn_perm(b, a, 0x07030602u);
                const uint32_t xy01 = __builtin_amdgcn_perm(y, x, 0x05010400u), xy23 = __builtin_amdgcn_perm(y, x, 0x07030602u);
                s[0][p] = __builtin_amdgcn_perm(xy01, ab01, 0x05040100u);
                s[1][p] = __builtin_amdgcn_perm(xy01, ab01, 0x07060302u);
                s[2][p] = __builtin_amdgcn_perm(xy23, ab23, 0x05040100u);
                s[3][p] = __builtin_amdgcn_perm(xy23, ab23, 0x07060302u);
            }
#pragma unroll
            for (int j = 0; j < 4; j++) put(4 * d + j, s[j]);
        }
    }
    __syncthreads();
#pragma unroll
    for (int p = 0; p < PANELS; p++) {
        const int panel = pg * PANELS + p;
        if (panel >= npanels) break;
        char* const o = out + ((int64_t)panel * kunits + ku) * 4096 + lane * 16;
#pragma unroll
        for (int f = 0; f < 4; f++) {
            const int at = (p * 4 + f) * 64 + lane;
            *reinterpret_cast<u32x4*>(o + f * 1024) = mine[at ^ (((at >> 4) ^ (at >> 8)) & 15)];
        }
    }
}

template <int ES, bool PAIR>
static int launch_repack_rows(const void* B0, const void* B1, int64_t ldb, int K, int N, int npanels, void* out, hipStream_t st, int flip) {
    constexpr int UNR = 2;
    const int kunits = (int)(((int64_t)K * ES + 127) / 128), groups = (kunits + 4 * UNR - 1) / (4 * UNR);
    const int64_t blocks = (int64_t)npanels * groups;
    if (blocks > 0x7fffffff) return set_error(MMX_E_INVALID, "weight matrix too large to repack in one launch");
    const bool is_short = (int64_t)K * ES < 16;
    hipLaunchKernelGGL((is_short ? repack_rows_kernel<ES, UNR, PAIR, SHORT_ROW> : repack_rows_kernel<ES, UNR, PAIR, LONG_ROW>), dim3((unsigned)blocks), dim3(256), 0, st, static_cast<const char*>(B0),
                       static_cast<const char*>(B1), ldb, K * ES, N, static_cast<char*>(out), kunits, groups, flip);
    return check_hip(hipGetLastError(), "repack_rows_kernel launch");
}

template <int ES>
static int launch_repack_cols(const void* B, int64_t ldb, int K, int N, void* out, hipStream_t st, int flip) {
    const int kunits = (int)(((int64_t)K * ES + 127) / 128), npanels = (N + 31) / 32;
    constexpr int WAVES = ES == 2 ? 4 : 1, PER_BLOCK = WAVES * (ES == 2 ? 2 : 4);
    const int64_t blocks = (int64_t)((npanels + PER_BLOCK - 1) / PER_BLOCK) * kunits;
    if (blocks > 0x7fffffff) return set_error(MMX_E_INVALID, "weight matrix too large to repack in one launch");
    const bool is_short = (int64_t)N * ES < 16;
    hipLaunchKernelGGL((is_short ? repack_cols_kernel<ES, SHORT_ROW> : repack_cols_kernel<ES, LONG_ROW>), dim3((unsigned)blocks), dim3(64 * WAVES), 0, st, static_cast<const char*>(B), ldb, K, N,
                       static_cast<char*>(out), kunits, npanels, flip);
    return check_hip(hipGetLastError(), "repack_cols_kernel launch");
}

int launch_repack(int elesz, const void* B, int64_t ldb, int K, int N, int transpose, void* out, hipStream_t st, int flip) {
    if (transpose) return elesz == 2 ? launch_repack_rows<2, false>(B, B, ldb, K, N, (N + 31) / 32, out, st, 0)
                                     : launch_repack_rows<1, false>(B, B, ldb, K, N, (N + 31) / 32, out, st, flip);
    return elesz == 2 ? launch_repack_cols<2>(B, ldb, K, N, out, st, 0) : launch_repack_cols<1>(B, ldb, K, N, out, st, flip);
}

int launch_repack_gate_up(const void* wg, const void* wu, int64_t ldw, int K, int N, void* out, hipStream_t st) {
    return launch_repack_rows<2, true>(wg, wu, ldw, K, N, 2 * N / 32, out, st, 0);
}

// Rows of any alignment and length (16 bytes and more) to rows of `pitch` bytes, a multiple of 128, zero behind their end.
__global__ __launch_bounds__(256) void align_rows_kernel(const char* __restrict__ A, int64_t lda, int pieces, int row_bytes, char* __restrict__ out, int per_row) {
    constexpr int UNR = 4;
    const int i0 = blockIdx.x * (256 * UNR) + threadIdx.x;
    u32x4 v[UNR];
    int at[UNR];
#pragma unroll
    for (int u = 0; u < UNR; u++) {
        const int i = i0 + u * 256 < pieces ? i0 + u * 256 : pieces - 1, m = i / per_row;
        at[u] = (i - m * per_row) * 16;
        v[u] = fetch16_in_row(A + (int64_t)m * lda, at[u], row_bytes);
    }
#pragma unroll
    for (int u = 0; u < UNR; u++)
        if (i0 + u * 256 < pieces) *reinterpret_cast<u32x4*>(out + (int64_t)(i0 + u * 256) * 16) = settle16_in_row(v[u], at[u], row_bytes);
}

int launch_align_rows(const void* A, int64_t lda, int M, int row_bytes, void* out, int pitch, hipStream_t st) {
    const int pieces = M * (pitch / 16);  // (the caller's workspace bounds it)
    hipLaunchKernelGGL(align_rows_kernel, dim3((pieces + 1023) / 1024), dim3(256), 0, st, static_cast<const char*>(A), lda, pieces, row_bytes,
                       static_cast<char*>(out), pitch / 16);
    return check_hip(hipGetLastError(), "align_rows_kernel launch");
}

// ---- per-tensor weight compression ---------------------------------------------------------------
__global__ void zero_u32_kernel(uint32_t* p) { *p = 0u; }

// All three kernels of this section stream bf16 and are bound by memory: a lane takes 16 bytes (8 weights) at a time.  A matrix
// whose rows follow each other without a gap is walked as one row (the host passes rows = 1).
// (11008 x 4096 weights: two bytes per load and a 64-bit division per weight took 217 us for the maxima and 65 for the
// quantisation.)
//   ROWS = false: blockIdx.y walks the rows, one load at a time: 4 MB of loads are in flight over the chip, which is what memory
//   takes; with four loads in a row maxima, quantisation and packing took, launch to launch, 66.3 us for 11008 x 4096, 13.9 for
//   1184 x 4160 and 19.7 for 3000 x 3000, now 61.4, 12.6 and 17.7 (two loads: 61.4, 13.5, 18.2; nontemporal loads and stores, twice
//   as many workgroups, and quantising from the end that was read last are level or behind).  Rows with gaps that are walked like this by
//   the quantiser (from 8192 columns) or by both (from 32768), maxima and quantisation, launch to launch: 4096 x 8192 31.9 -> 29.8,
//   4096 x 11008 43.8 -> 39.5, 11008 x 8200 104 -> 97, 512 x 32768 21.9 -> 19.5, 4 x 100000 12.9 -> 10.3.
//   ROWS = true, for rows with gaps that are too short to fill the four loads of a workgroup: 2^row_log2 lanes share a row, a
//   lane's four loads are of four rows.  (Maxima and quantisation of rows with gaps, a row at a time -> shared out: 1000000 x 8
//   4252 -> 17 us, 131072 x 128 518 -> 20, 16384 x 1024 67 -> 18, 4096 x 4096 31 -> 18; the maxima alone 4096 x 8192 46 -> 31, both kernels.)
constexpr int QUANT_UNR = 4;

template <int THREADS, bool ROWS, typename F>
__device__ __forceinline__ void for_each_8_weights(const char* __restrict__ W, int64_t ldw, int rows, int64_t cols, int row_log2, F&& f) {
    if constexpr (ROWS) {
        const int per_block = THREADS >> row_log2;
        const int64_t step = (int64_t)gridDim.x * per_block, r0 = (int64_t)blockIdx.x * per_block + (threadIdx.x >> row_log2);
        for (int64_t r = r0; r < rows; r += step * QUANT_UNR) {
            for (int64_t c = (int64_t)(threadIdx.x & ((1 << row_log2) - 1)) * 8; c < cols; c += (int64_t)8 << row_log2) {
                u32x4 v[QUANT_UNR];
                load16_rows<2>(v, c * 2, cols * 2, [&](int u) { return W + (r + u * step) * ldw; }, [&](int u) { return r + u * step < rows; });
#pragma unroll
                for (int u = 0; u < QUANT_UNR; u++)
                    if (r + u * step < rows) f(r + u * step, c, v[u]);
            }
        }
    } else {
        const int64_t step = (int64_t)gridDim.x * THREADS;
        for (int r = blockIdx.y; r < rows; r += gridDim.y) {
            const char* const row = W + (int64_t)r * ldw;
            const int64_t first = (int64_t)blockIdx.x * THREADS + threadIdx.x, len = cols * 2;
            if (len < 16) {  // (uniform)
                u32x4 v[1];
                load16_rows<2, SHORT_ROW>(v, first * 16, len, [&](int) { return row; }, [&](int) { return true; });
                if (first * 8 < cols) f(r, first * 8, v[0]);
                continue;
            }
            // One load instruction for the whole wavefront, the row's end in it.  (A draft that loaded the end in a branch of its own gave
            // wrong bytes now and then on the GPU.  Why is not known: compiled again, that form waits for both loads before
            // either is used, and its offsets stay in the row.)
            for (int64_t i = first; i * 8 < cols; i += step) {
                const int64_t at = i * 16, last = len - 16, from = at < last ? at : last;
                u32x4 v = load16<2>(row + from);
                if (from < at) v = settle16_in_row(v, (int)(at - from), 16);
                f(r, i * 8, v);
            }
        }
    }
}

// 8 bytes to columns c .. c + 7 of a row of `cols` (fewer at its end)
__device__ __forceinline__ void store_8_bytes(char* row, int64_t c, int64_t cols, uint32_t lo, uint32_t hi) {
    const uint32_t w[2] = {lo, hi};
    if (c + 8 <= cols) {
        __builtin_memcpy(row + c, w, 8);
    } else {
#pragma unroll
        for (int e = 0; e < 8; e++)
            if (c + e < cols) row[c + e] = (char)(w[e >> 2] >> (8 * (e & 3)));
    }
}

// max |w| over the matrix: the bit pattern of a non-negative float orders like an unsigned integer.
// WORDS: every workgroup leaves its maximum in a word of its own, and the quantising kernel's workgroups take the largest.  Without
// (a scratch of one word) the workgroups' atomics all meet at one address, cleared by a launch before, and take 10 ns each there, so
// there is one workgroup per CU, of 16 wavefronts (2048 workgroups of four: 4096 x 4096 weights in 27 us instead of 10).
constexpr int ABSMAX_THREADS = 1024;
template <bool ROWS, bool WORDS>
__global__ __launch_bounds__(ABSMAX_THREADS) void absmax_kernel(const char* __restrict__ W, int64_t ldw, int rows, int64_t cols, int row_log2,
                                                                uint32_t* out) {
    uint32_t m = 0;
    for_each_8_weights<ABSMAX_THREADS, ROWS>(W, ldw, rows, cols, row_log2, [&](int64_t, int64_t, const u32x4& v) __attribute__((always_inline)) {
#pragma unroll
        for (int d = 0; d < 4; d++) {
            const uint32_t lo = (v[d] << 16) & 0x7fffffffu, hi = v[d] & 0x7fff0000u;
            if (lo <= 0x7f800000u && lo > m) m = lo;  // NaNs do not take part, as with vmaxps/vminps accumulators
            if (hi <= 0x7f800000u && hi > m) m = hi;
        }
    });
    for (int off = 32; off > 0; off >>= 1) {
        const uint32_t o = __shfl_xor(m, off);
        m = o > m ? o : m;
    }
    __shared__ uint32_t of_wave[ABSMAX_THREADS / 64];
    if ((threadIdx.x & 63) == 0) of_wave[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int w = 1; w < ABSMAX_THREADS / 64; w++) m = of_wave[w] > m ? of_wave[w] : m;
        if constexpr (WORDS) out[blockIdx.y * gridDim.x + blockIdx.x] = m;
        else if (m > __hip_atomic_load(out, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(out, m);
    }
}

// q = sat8(rne(w * (127/max))) (include/kernels_amx.hpp:508-523); scales_out = {127/max, max/127}; the maximum is that of `words` words
template <bool ROWS>
__global__ __launch_bounds__(256) void quantize_kernel(const char* __restrict__ W, int64_t ldw, int rows, int64_t cols, int row_log2,
                                                       char* __restrict__ Wq, int64_t ldq, const uint32_t* __restrict__ absmax_bits, int words,
                                                       float* __restrict__ scales_out) {
    uint32_t bits;
    if (words == 1) {
        bits = *absmax_bits;
    } else {
        bits = 0;
        for (int i = threadIdx.x; i < words; i += 256) bits = absmax_bits[i] > bits ? absmax_bits[i] : bits;
        for (int off = 32; off > 0; off >>= 1) {
            const uint32_t o = __shfl_xor(bits, off);
            bits = o > bits ? o : bits;
        }
        __shared__ uint32_t of_wave[4];
        if ((threadIdx.x & 63) == 0) of_wave[threadIdx.x >> 6] = bits;
        __syncthreads();
#pragma unroll
        for (int w = 0; w < 4; w++) bits = of_wave[w] > bits ? of_wave[w] : bits;
    }
    const float amax = u2f(bits);
    const float q = 127 / amax;
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) {
        scales_out[0] = q;
        scales_out[1] = amax / 127;
    }
    for_each_8_weights<256, ROWS>(W, ldw, rows, cols, row_log2, [&](int64_t r, int64_t c, const u32x4& v) __attribute__((always_inline)) {
        uint32_t o[2];
#pragma unroll
        for (int h = 0; h < 2; h++)
            o[h] = to_s8_sat_x4(u2f(v[2 * h] << 16) * q, u2f(v[2 * h] & 0xffff0000u) * q, u2f(v[2 * h + 1] << 16) * q,
                                u2f(v[2 * h + 1] & 0xffff0000u) * q);
        if (c < cols) store_8_bytes(Wq + r * ldq, c, cols, o[0], o[1]);
    });
}

// A matrix without gaps between its rows becomes one row.
static void one_row(int64_t ldw, int64_t ldq, int& rows, int64_t& cols) {
    if (ldw == cols * 2 && ldq == cols) cols *= rows, rows = 1;
}

// How the kernels above walk a matrix, by at most `most` workgroups.  Rows with gaps that are shorter than QUANT_UNR loads of a
// workgroup are shared out (ROWS): the fewest lanes, a power of two, that cover a row, and QUANT_UNR rows per lane at a time; with
// `spread` one while there are fewer than two workgroups for every CU (not for the maxima).
struct QuantWalk {
    bool by_rows;
    int row_log2;
    dim3 grid;
};
static QuantWalk quantize_walk(int rows, int64_t cols, int threads, int most, bool spread) {
    if (rows > 1 && cols < (int64_t)threads * 8 * QUANT_UNR) {
        int log2 = 0;
        while ((8 << log2) < cols && (1 << log2) < threads) log2++;
        const int64_t x1 = (rows + (threads >> log2) - 1) / (threads >> log2), x = (x1 + QUANT_UNR - 1) / QUANT_UNR;
        return {true, log2, dim3((unsigned)(spread && x < 2 * num_cus() ? (x1 < 2 * num_cus() ? x1 : 2 * num_cus()) : (x < most ? x : most)))};
    }
    const int64_t x = (cols + (int64_t)threads * 8 - 1) / ((int64_t)threads * 8);
    const int gx = (int)(x < most ? x : most), gy = most / gx;
    return {false, 0, dim3((unsigned)gx, (unsigned)(rows < gy ? rows : gy))};
}

// scratch: words > 1 means that many, at least as many as there are CUs
int launch_quantize(const void* W, int64_t ldw, int rows, int cols_in, void* Wq, int64_t ldq, float* scales_out,
                    uint32_t* scratch, int words, hipStream_t st) {
    int64_t cols = cols_in;
    one_row(ldw, ldq, rows, cols);
    const QuantWalk m = quantize_walk(rows, cols, ABSMAX_THREADS, num_cus(), false), q = quantize_walk(rows, cols, 256, 2048, true);
    const int used = words > 1 ? (int)(m.grid.x * m.grid.y) : 1;
    if (used > words) return set_error(MMX_E_INVALID, "quantize: %d words of scratch, %d needed", words, used);
    if (words == 1) hipLaunchKernelGGL(zero_u32_kernel, dim3(1), dim3(1), 0, st, scratch);
    const auto absmax = words == 1 ? (m.by_rows ? absmax_kernel<true, false> : absmax_kernel<false, false>)
                                   : (m.by_rows ? absmax_kernel<true, true> : absmax_kernel<false, true>);
    hipLaunchKernelGGL(absmax, m.grid, dim3(ABSMAX_THREADS), 0, st, static_cast<const char*>(W), ldw, rows, cols, m.row_log2, scratch);
    hipLaunchKernelGGL(q.by_rows ? quantize_kernel<true> : quantize_kernel<false>, q.grid, dim3(256), 0, st, static_cast<const char*>(W), ldw,
                       rows, cols, q.row_log2, static_cast<char*>(Wq), ldq, scratch, used, scales_out);
    return check_hip(hipGetLastError(), "quantize kernels launch");
}

// q = trunc(bf16_rne(float(w) * scale)): the element conversion of repackB_1xL<int8_t, L>
// (weight_compression/fc16m.cpp:80-81, "*dst++ = src0[n] * scale" with src0 an ov::bfloat16* and dst an int8_t*: the
// product is a bfloat16 again, include/bf16.hpp:181-183, and its conversion to int8_t goes through float and
// truncates toward zero).  Values the language leaves undefined are defined here: beyond int8's range saturates,
// NaN gives 0.
__device__ __forceinline__ uint32_t scale_trunc(float w, float scale) {
    const float t = from_bf16(to_bf16(w * scale));
    int q = 0;
    if (t == t) q = t >= 127.0f ? 127 : (t <= -128.0f ? -128 : (int)t);  // float -> int: toward zero
    return (uint32_t)q & 0xffu;
}

template <bool ROWS>
__global__ __launch_bounds__(256) void quantize_scale_trunc_kernel(const char* __restrict__ W, int64_t ldw, int rows, int64_t cols,
                                                                   int row_log2, float scale, char* __restrict__ Wq, int64_t ldq) {
    for_each_8_weights<256, ROWS>(W, ldw, rows, cols, row_log2, [&](int64_t r, int64_t c, const u32x4& v) __attribute__((always_inline)) {
        uint32_t o[2] = {0, 0};
#pragma unroll
        for (int d = 0; d < 4; d++)
            o[d >> 1] |= (scale_trunc(u2f(v[d] << 16), scale) | scale_trunc(u2f(v[d] & 0xffff0000u), scale) << 8) << (16 * (d & 1));
        if (c < cols) store_8_bytes(Wq + r * ldq, c, cols, o[0], o[1]);
    });
}

int launch_quantize_scale_trunc(const void* W, int64_t ldw, int rows, int cols_in, float scale, void* Wq, int64_t ldq, hipStream_t st) {
    int64_t cols = cols_in;
    one_row(ldw, ldq, rows, cols);
    const QuantWalk q = quantize_walk(rows, cols, 256, 2048, true);
    hipLaunchKernelGGL(q.by_rows ? quantize_scale_trunc_kernel<true> : quantize_scale_trunc_kernel<false>, q.grid, dim3(256), 0, st,
                       static_cast<const char*>(W), ldw, rows, cols, q.row_log2, scale, static_cast<char*>(Wq), ldq);
    return check_hip(hipGetLastError(), "quantize_scale_trunc_kernel launch");
}

// The same conversion and mmx_repack_b of its result in one pass over W [K, N]: every weight is read once and leaves as a byte of its
// fragment, where quantising to a matrix of bytes and packing that moved each byte twice more, in a launch of its own.  A wavefront
// takes 64 columns x 128 of k, the two 4 KiB units that repack_cols_kernel<1> makes of bytes: a lane reads 16 rows of 8 columns (a
// load covers 8 whole lines), converts, transposes its 16 x 8 bytes in registers, and the wavefront's slots leave through LDS as
// whole fragments.  Bound by memory (K x N, device time of the two launches -> of this one: 576 x 8640 8.1 + 3.9 -> 5.8 us, 800 x 9504
// 10.9 + 5.5 -> 9.9; 4096 x 11008 27.1, 5.0 TB/s).
__device__ __forceinline__ uint32_t scale_trunc_x4(uint32_t w01, uint32_t w23, float scale) {
    const float w[4] = {u2f(w01 << 16), u2f(w01 & 0xffff0000u), u2f(w23 << 16), u2f(w23 & 0xffff0000u)};
    uint32_t b[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        int i;  // (the instruction saturates and makes NaN 0, which the C++ conversion leaves undefined)
        asm("v_cvt_i32_f32 %0, %1" : "=v"(i) : "v"(from_bf16(to_bf16(w[e] * scale))));
        b[e] = (uint32_t)(i < -128 ? -128 : (i > 127 ? 127 : i)) & 0xffu;
    }
    return b[0] | b[1] << 8 | b[2] << 16 | b[3] << 24;
}

template <RowLength LEN>
__global__ __launch_bounds__(64) void scale_trunc_pack_kernel(const char* __restrict__ W, int64_t ldw, int K, int N, float scale,
                                                              char* __restrict__ out, int kunits, int npanels) {
    __shared__ __attribute__((aligned(16))) u32x4 slots[512];
    const int lane = threadIdx.x, ng = lane & 7, kg = lane >> 3;
    const int ku = blockIdx.x % kunits, pg = blockIdx.x / kunits;
    const int n = pg * 64 + ng * 8, k = ku * 128 + kg * 16;
    u32x4 row[16];
    if (pg * 64 + 64 <= N && ku * 128 + 128 <= K) {
#pragma unroll
        for (int e = 0; e < 16; e++) row[e] = load16<2>(W + (int64_t)(k + e) * ldw + (int64_t)n * 2);
    } else {
        load16_rows<2, LEN>(row, (int64_t)n * 2, (int64_t)N * 2, [&](int e) { return W + (int64_t)(k + e) * ldw; },
                            [&](int e) { return k + e < K; });
    }
    auto put = [&](int j, u32x4 slot) {  // the slot of column n + j
        const int col = ng * 8 + j;
        const int at = ((col >> 5) * 4 + (kg >> 1)) * 64 + (kg & 1) * 32 + (col & 31);
        slots[at ^ (((at >> 4) ^ (at >> 8)) & 15)] = slot;
    };
#pragma unroll
    for (int h = 0; h < 2; h++) {  // four columns at a time
        u32x4 s[4];
#pragma unroll
        for (int p = 0; p < 4; p++) {
            uint32_t q[4];
#pragma unroll
            for (int e = 0; e < 4; e++) q[e] = scale_trunc_x4(row[4 * p + e][2 * h], row[4 * p + e][2 * h + 1], scale);
            const uint32_t ab01 = __builtin_amdgcn_perm(q[1], q[0], 0x05010400u), ab23 = __builtin_amdgcn_perm(q[1], q[0], 0x07030602u);
            const uint32_t xy01 = __builtin_amdgcn_perm(q[3], q[2], 0x05010400u), xy23 = __builtin_amdgcn_perm(q[3], q[2], 0x07030602u);
            s[0][p] = __builtin_amdgcn_perm(xy01, ab01, 0x05040100u);
            s[1][p] = __builtin_amdgcn_perm(xy01, ab01, 0x07060302u);
            s[2][p] = __builtin_amdgcn_perm(xy23, ab23, 0x05040100u);
            s[3][p] = __builtin_amdgcn_perm(xy23, ab23, 0x07060302u);
        }
#pragma unroll
        for (int j = 0; j < 4; j++) put(4 * h + j, s[j]);
    }
    __syncthreads();
#pragma unroll
    for (int p = 0; p < 2; p++) {
        if (pg * 2 + p >= npanels) break;
        char* const o = out + ((int64_t)(pg * 2 + p) * kunits + ku) * 4096 + lane * 16;
#pragma unroll
        for (int f = 0; f < 4; f++) {
            const int at = (p * 4 + f) * 64 + lane;
            *reinterpret_cast<u32x4*>(o + f * 1024) = slots[at ^ (((at >> 4) ^ (at >> 8)) & 15)];
        }
    }
}

int launch_scale_trunc_pack(const void* W, int64_t ldw, int K, int N, float scale, void* packed, hipStream_t st) {
    const int kunits = (K + 127) / 128, npanels = (N + 31) / 32;
    const int64_t blocks = (int64_t)((npanels + 1) / 2) * kunits;
    if (blocks > 0x7fffffff) return set_error(MMX_E_INVALID, "weight matrix too large to pack in one launch");
    hipLaunchKernelGGL(N < 8 ? scale_trunc_pack_kernel<SHORT_ROW> : scale_trunc_pack_kernel<LONG_ROW>, dim3((unsigned)blocks), dim3(64), 0, st,
                       static_cast<const char*>(W), ldw, K, N, scale, static_cast<char*>(packed), kunits, npanels);
    return check_hip(hipGetLastError(), "scale_trunc_pack_kernel launch");
}

// ---- packed int8 -> packed bf16 (exact) -------------------------------------------------------------
// int8 slot (panel, f, lane): 16 consecutive k of column n -> bf16 fragments 2f and 2f+1 ... the
// 16 k's starting at 32f + 16g split into two runs of 8: run h goes to bf16 fragment 2f+g,
// lane (n%32) + 32*h.
__global__ void dequant_packed_kernel(const char* __restrict__ in, char* __restrict__ out, int nfrag8, int nfrag16,
                                      int64_t total_slots) {
    const int64_t slot = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (slot >= total_slots) return;
    const int lane = (int)(slot & 63);
    const int64_t pf = slot >> 6;
    const int f = (int)(pf % nfrag8);
    const int64_t panel = pf / nfrag8;
    const uint4 v = *reinterpret_cast<const uint4*>(in + slot * 16);
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
    const int g = lane >> 5, l32 = lane & 31;
#pragma unroll
    for (int h = 0; h < 2; h++) {
        alignas(16) uint16_t o[8];
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const int b = h * 8 + e;
            o[e] = to_bf16((float)(int8_t)((w[b >> 2] >> (8 * (b & 3))) & 0xff));
        }
        // the bf16 layout pads K to 64, the int8 one to 128: fragments past the bf16 padding hold only zeros
        if (2 * f + g < nfrag16) {
            const int64_t of = (panel * nfrag16 + 2 * f + g) * 64 + l32 + 32 * h;
            *reinterpret_cast<uint4*>(out + of * 16) = *reinterpret_cast<const uint4*>(o);
        }
    }
}

int launch_dequant_packed(const void* in, int K, int N, void* out, hipStream_t st) {
    const int nfrag8 = ((K + 127) / 128 * 128) / 32;
    const int nfrag16 = ((K + 63) / 64 * 64) / 16;
    const int64_t slots = (int64_t)((N + 31) / 32) * nfrag8 * 64;
    const int64_t blocks = (slots + 255) / 256;
    if (blocks > 0x7fffffff) return set_error(MMX_E_INVALID, "weight matrix too large");
    hipLaunchKernelGGL(dequant_packed_kernel, dim3((unsigned)blocks), dim3(256), 0, st, static_cast<const char*>(in),
                       static_cast<char*>(out), nfrag8, nfrag16, slots);
    return check_hip(hipGetLastError(), "dequant_packed_kernel launch");
}

// ---- c[M] = A[M,K] · b[K] ---------------------------------------------------------------------------
// amx_kernel::MatmulVector (include/kernels_amx.hpp:833-1043) and GemAvB (:1529-1618): one
// wavefront per row of A, lanes stride over K, wave reduction.
template <bool I8>
__global__ void matvec_kernel(const char* __restrict__ A, int64_t lda, const char* __restrict__ b, void* c, int M, int K) {
    const int row = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (row >= M) return;
    const char* a = A + (int64_t)row * lda;
    if (I8) {
        int acc = 0;
        for (int k = lane; k < K; k += 64) acc += (int)(int8_t)a[k] * (int)(int8_t)b[k];
        for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
        if (lane == 0) static_cast<int*>(c)[row] = acc;
    } else {
        float acc = 0.0f;
        for (int k = lane; k < K; k += 64)
            acc = __builtin_fmaf(from_bf16(reinterpret_cast<const uint16_t*>(a)[k]),
                                 from_bf16(reinterpret_cast<const uint16_t*>(b)[k]), acc);
        for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
        if (lane == 0) static_cast<float*>(c)[row] = acc;
    }
}

// The form for rows that are 16-byte aligned (the attention use: q against a cache of keys, one row per
// token, K = head size): LPR lanes share a row and fetch 16 bytes each, a wavefront covers 64/LPR rows at
// a time and UNR such groups per trip, so that every lane has UNR independent loads in flight.  Elements
// after the last whole 16 bytes of a row are added one by one.
template <bool I8, int LPR, int UNR>
__global__ void __launch_bounds__(256) matvec_rows_kernel(const char* __restrict__ A, int64_t lda, const char* __restrict__ b,
                                                          void* c, int M, int K) {
    constexpr int RPW = 64 / LPR, EPC = I8 ? 16 : 8;
    const int lane = threadIdx.x & 63, sub = lane % LPR, rsel = lane / LPR;
    const int64_t wave = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    const int64_t nwaves = (int64_t)gridDim.x * (blockDim.x >> 6);
    const int nchunks = K / EPC;
    const uint4* bq = reinterpret_cast<const uint4*>(b);
    for (int64_t row0 = wave * (RPW * UNR); row0 < M; row0 += nwaves * (RPW * UNR)) {
        const char* a[UNR];
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
            const int64_t r = row0 + u * RPW + rsel;
            a[u] = A + (r < M ? r : (int64_t)M - 1) * lda;
        }
        float facc[UNR];
        int iacc[UNR];
#pragma unroll
        for (int u = 0; u < UNR; ++u) facc[u] = 0.0f, iacc[u] = 0;
        for (int ch = sub; ch < nchunks; ch += LPR) {
            const uint4 bv = bq[ch];
            uint4 av[UNR];
#pragma unroll
            for (int u = 0; u < UNR; ++u) {  // read once: keep the rows out of the way of what the caches hold
                typedef unsigned v4u __attribute__((ext_vector_type(4)));
                const v4u t = __builtin_nontemporal_load(reinterpret_cast<const v4u*>(a[u]) + ch);
                av[u] = make_uint4(t.x, t.y, t.z, t.w);
            }
#pragma unroll
            for (int u = 0; u < UNR; ++u) {
                const uint32_t aw[4] = {av[u].x, av[u].y, av[u].z, av[u].w}, bw[4] = {bv.x, bv.y, bv.z, bv.w};
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (I8) {
                        iacc[u] = __builtin_amdgcn_sdot4((int)aw[i], (int)bw[i], iacc[u], false);
                    } else {
                        facc[u] = __builtin_fmaf(__uint_as_float(aw[i] << 16), __uint_as_float(bw[i] << 16), facc[u]);
                        facc[u] = __builtin_fmaf(__uint_as_float(aw[i] & 0xffff0000u), __uint_as_float(bw[i] & 0xffff0000u), facc[u]);
                    }
                }
            }
        }
        for (int k = nchunks * EPC + sub; k < K; k += LPR) {
#pragma unroll
            for (int u = 0; u < UNR; ++u) {
                if (I8)
                    iacc[u] += (int)(int8_t)a[u][k] * (int)(int8_t)b[k];
                else
                    facc[u] = __builtin_fmaf(from_bf16(reinterpret_cast<const uint16_t*>(a[u])[k]),
                                             from_bf16(reinterpret_cast<const uint16_t*>(b)[k]), facc[u]);
            }
        }
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
#pragma unroll
            for (int off = LPR / 2; off > 0; off >>= 1) {
                if (I8)
                    iacc[u] += __shfl_xor(iacc[u], off);
                else
                    facc[u] += __shfl_xor(facc[u], off);
            }
            const int64_t r = row0 + u * RPW + rsel;
            if (sub == 0 && r < M) {
                if (I8)
                    static_cast<int*>(c)[r] = iacc[u];
                else
                    static_cast<float*>(c)[r] = facc[u];
            }
        }
    }
}

template <bool I8, int LPR>
static void launch_matvec_rows(const void* A, int64_t lda, const void* b, void* c, int M, int K, hipStream_t st) {
    constexpr int UNR = 4, rows_per_block = 4 * (64 / LPR) * UNR;
    // one trip per wavefront: many short workgroups keep more requests in flight than a grid-stride loop does
    // (2^21 rows of 256 B: 6.9 TB/s against 6.4 with 4096 workgroups)
    const int64_t blocks = ((int64_t)M + rows_per_block - 1) / rows_per_block;
    hipLaunchKernelGGL((matvec_rows_kernel<I8, LPR, UNR>), dim3((unsigned)blocks), dim3(256), 0, st, static_cast<const char*>(A),
                       lda, static_cast<const char*>(b), c, M, K);
}

int launch_matvec(bool i8, const void* A, int64_t lda, const void* b, void* c, int M, int K, hipStream_t st) {
    if (M <= 0) return MMX_OK;
    const bool aligned = ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(b) | (uintptr_t)lda) & 15) == 0;
    const int nchunks = K / (i8 ? 16 : 8);
    if (aligned && nchunks > 0) {
        if (i8) {
            if (nchunks <= 4) launch_matvec_rows<true, 4>(A, lda, b, c, M, K, st);
            else if (nchunks <= 16) launch_matvec_rows<true, 16>(A, lda, b, c, M, K, st);
            else launch_matvec_rows<true, 64>(A, lda, b, c, M, K, st);
        } else {
            if (nchunks <= 4) launch_matvec_rows<false, 4>(A, lda, b, c, M, K, st);
            else if (nchunks <= 16) launch_matvec_rows<false, 16>(A, lda, b, c, M, K, st);
            else launch_matvec_rows<false, 64>(A, lda, b, c, M, K, st);
        }
        return check_hip(hipGetLastError(), "matvec_rows_kernel launch");
    }
    const int rows_per_block = 4;
    const int blocks = (M + rows_per_block - 1) / rows_per_block;
    if (i8)
        hipLaunchKernelGGL((matvec_kernel<true>), dim3(blocks), dim3(256), 0, st, static_cast<const char*>(A), lda,
                           static_cast<const char*>(b), c, M, K);
    else
        hipLaunchKernelGGL((matvec_kernel<false>), dim3(blocks), dim3(256), 0, st, static_cast<const char*>(A), lda,
                           static_cast<const char*>(b), c, M, K);
    return check_hip(hipGetLastError(), "matvec_kernel launch");
}

// ---- int4: per-column symmetric quantisation + packing, one workgroup per 32-column panel ----------------
// The maxima of the panel's columns come first, so its weights are read twice (the second time mostly from the caches); both
// passes move 16 bytes per lane, over whole lines, with the panel spread over 16 wavefronts.
//   [N, K]: a column is a row.  Pass 1: half a wavefront per column would leave lines half used, so a wavefront walks one
//   column at a time, 1 KiB per load.  Pass 2: a wavefront makes a fragment (32 columns x 64 of k) from 4 loads of 8 rows x
//   128 bytes; a lane's 8 weights are one dword of slot (k half g, column), dword i = chunk % 4: a store is two lines.
//   [K, N]: a row holds the panel's 32 columns in 64 bytes.  Pass 1: lane -> (row, 8 columns).  Pass 2: a lane reads 8 rows
//   of 8 columns and builds the dword of each column from its own 8 x 8 square.
// (4096 x 11008, [N, K] / [K, N]: two-byte loads by four wavefronts per panel took 261 / 360 us; now 45 / 70.)
constexpr int QUANT4_WAVES = 16;

__device__ __forceinline__ uint32_t int4_of(float w, float scale) {
    float q = rintf(w * scale);
    q = (q != q) ? 0.0f : q;  // a NaN weight, or an infinite one (its column's scale is then 0): quantised to 0
    q = fminf(fmaxf(q, -7.0f), 7.0f);
    return (uint32_t)(int)q & 0xfu;
}

// [N, K], 64 of k from k0 on: 4 loads of 8 rows x 128 bytes; and the fragment they make, scaled by qs.
__device__ __forceinline__ void load_fragment_rows(u32x4 (&v)[4], const char* W, int64_t ldw, int K, int N, int n0, int k0) {
    const int lane = threadIdx.x & 63, r8 = lane >> 3, k = k0 + 8 * (lane & 7);
    if (n0 + 32 <= N && k0 + 64 <= K) {
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = load16<2>(W + (int64_t)(n0 + 8 * i + r8) * ldw + (int64_t)k * 2);
    } else {
        load16_rows<2>(v, (int64_t)k * 2, (int64_t)K * 2, [&](int i) { return W + (int64_t)(n0 + 8 * i + r8) * ldw; },
                       [&](int i) { return n0 + 8 * i + r8 < N; });
    }
}
__device__ __forceinline__ void store_fragment_rows(const u32x4 (&v)[4], const float (&qs)[4], char* fragment) {
    const int lane = threadIdx.x & 63, r8 = lane >> 3, c = lane & 7;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        uint32_t d = 0;
#pragma unroll
        for (int e = 0; e < 4; e++)
            d |= (int4_of(u2f(v[i][e] << 16), qs[i]) | int4_of(u2f(v[i][e] & 0xffff0000u), qs[i]) << 4) << (8 * e);
        *reinterpret_cast<uint32_t*>(fragment + ((c >> 2) * 32 + 8 * i + r8) * 16 + (c & 3) * 4) = d;
    }
}

// [K, N], 128 of k from k0 on: a lane takes 8 columns of 8 rows, 16 chunks of k to a wavefront; and their two fragments.
__device__ __forceinline__ void load_fragments_cols(u32x4 (&v)[8], const char* W, int64_t ldw, int K, int N, int n0, int k0) {
    const int lane = threadIdx.x & 63, n = n0 + 8 * (lane & 3), k = k0 + 8 * (lane >> 2);
    if (n0 + 32 <= N && k0 + 128 <= K) {
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = load16<2>(W + (int64_t)(k + e) * ldw + (int64_t)n * 2);
    } else {
        load16_rows<2>(v, (int64_t)n * 2, (int64_t)N * 2, [&](int e) { return W + (int64_t)(k + e) * ldw; },
                       [&](int e) { return k + e < K; });
    }
}
__device__ __forceinline__ void store_fragments_cols(const u32x4 (&v)[8], const float (&qs)[8], char* fragments) {
    const int lane = threadIdx.x & 63, ng = lane & 3, kc = lane >> 2;
    char* const slot = fragments + (kc >> 3) * 1024 + (((kc >> 2) & 1) * 32 + 8 * ng) * 16 + (kc & 3) * 4;
#pragma unroll
    for (int n = 0; n < 8; n++) {
        uint32_t d = 0;
#pragma unroll
        for (int e = 0; e < 8; e++) d |= int4_of(n & 1 ? u2f(v[e][n >> 1] & 0xffff0000u) : u2f(v[e][n >> 1] << 16), qs[n]) << (4 * e);
        *reinterpret_cast<uint32_t*>(slot + n * 16) = d;
    }
}

// The scale of a column and what undoes it, from the column's largest |w|.
__device__ __forceinline__ float int4_scale(float amax, float* deq) {
    *deq = amax / 7.0f;
    return amax > 0.0f ? 7.0f / amax : 0.0f;
}

// K of at most 256 (the four fragments that every panel has): the panel stays in registers between the two passes, read once,
// by as many wavefronts as that takes - 4 of one fragment each from [N, K], 2 of two from [K, N].  (Sixteen wavefronts on a
// panel that short are mostly idle: [N, K] / [K, N], K = 32 x 1048576 296 / 314 -> 89 / 90 us, 64 x 262144 77 / 84 -> 24 / 27,
// 256 x 65536 22 / 29 -> 9 / 16.)
template <bool TRANSPOSED>
__global__ __launch_bounds__(TRANSPOSED ? 256 : 128) void quant4_pack_short_kernel(const char* __restrict__ W, int64_t ldw, int K, int N,
                                                                                   char* __restrict__ out, float* deq_out) {
    constexpr int WAVES = TRANSPOSED ? 4 : 2;
    __shared__ float smax[32][WAVES];
    __shared__ float sscale[32];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int n0 = blockIdx.x * 32;
    char* const o = out + (int64_t)blockIdx.x * 4096;
    u32x4 v[TRANSPOSED ? 4 : 8];
    if constexpr (TRANSPOSED) {
        load_fragment_rows(v, W, ldw, K, N, n0, 64 * wave);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float m = 0.0f;  // (fmaxf drops a NaN)
#pragma unroll
            for (int d = 0; d < 4; d++) m = fmaxf(fmaxf(m, fabsf(u2f(v[i][d] << 16))), fabsf(u2f(v[i][d] & 0xffff0000u)));
            for (int off = 1; off < 8; off <<= 1) m = fmaxf(m, __shfl_xor(m, off));
            if ((lane & 7) == 0) smax[8 * i + (lane >> 3)][wave] = m;
        }
    } else {
        load_fragments_cols(v, W, ldw, K, N, n0, 128 * wave);
#pragma unroll
        for (int n = 0; n < 8; n++) {
            float m = 0.0f;
#pragma unroll
            for (int e = 0; e < 8; e++) m = fmaxf(m, fabsf(n & 1 ? u2f(v[e][n >> 1] & 0xffff0000u) : u2f(v[e][n >> 1] << 16)));
            for (int off = 4; off < 64; off <<= 1) m = fmaxf(m, __shfl_xor(m, off));
            if (lane < 4) smax[8 * lane + n][wave] = m;
        }
    }
    __syncthreads();
    if (t < 32) {
        float a = 0.0f, deq;
#pragma unroll
        for (int w = 0; w < WAVES; w++) a = fmaxf(a, smax[t][w]);
        sscale[t] = int4_scale(a, &deq);
        if (n0 + t < N) deq_out[n0 + t] = deq;
    }
    __syncthreads();
    if constexpr (TRANSPOSED) {
        float qs[4];
#pragma unroll
        for (int i = 0; i < 4; i++) qs[i] = sscale[8 * i + (lane >> 3)];
        store_fragment_rows(v, qs, o + wave * 1024);
    } else {
        float qs[8];
#pragma unroll
        for (int e = 0; e < 8; e++) qs[e] = sscale[8 * (lane & 3) + e];
        store_fragments_cols(v, qs, o + wave * 2048);
    }
}

template <bool TRANSPOSED>
__global__ __launch_bounds__(QUANT4_WAVES * 64) void quant4_pack_kernel(const char* __restrict__ W, int64_t ldw, int K, int N,
                                                                        char* __restrict__ out, int nfrag, float* deq_out) {
    __shared__ float smax[32][QUANT4_WAVES];
    __shared__ float sscale[32];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int n0 = blockIdx.x * 32;
    constexpr int UNR = 4;
    // (fmaxf drops a NaN)
    if constexpr (TRANSPOSED) {
        for (int c = wave; c < 32; c += QUANT4_WAVES) {
            float m = 0.0f;
            if (n0 + c < N) {
                const char* const row = W + (int64_t)(n0 + c) * ldw;
                for (int k = lane * 8; k < K; k += 512 * UNR) {
                    // (past the end of the row its last 16 bytes, which a maximum may meet twice: one load instruction for the whole wavefront)
                    u32x4 v[UNR];
#pragma unroll
                    for (int u = 0; u < UNR; u++) {
                        const int from = k + 512 * u < K - 8 ? k + 512 * u : K - 8;
                        v[u] = load16<2>(row + (int64_t)from * 2);
                    }
#pragma unroll
                    for (int u = 0; u < UNR; u++)
#pragma unroll
                        for (int d = 0; d < 4; d++) m = fmaxf(fmaxf(m, fabsf(u2f(v[u][d] << 16))), fabsf(u2f(v[u][d] & 0xffff0000u)));
                }
            }
            for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
            if (lane < QUANT4_WAVES) smax[c][lane] = m;
        }
    } else {
        const int ng = lane & 3;  // columns 8 ng .. 8 ng + 7 of the panel
        float m[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        for (int k = wave * 16 + (lane >> 2); k < K; k += QUANT4_WAVES * 16 * UNR) {
            u32x4 v[UNR];
            auto ku = [&](int u) { return k + QUANT4_WAVES * 16 * u; };
            if (n0 + 32 <= N && ku(UNR - 1) < K) {
#pragma unroll
                for (int u = 0; u < UNR; u++) v[u] = load16<2>(W + (int64_t)ku(u) * ldw + (int64_t)(n0 + 8 * ng) * 2);
            } else {
                load16_rows<2>(v, (int64_t)(n0 + 8 * ng) * 2, (int64_t)N * 2, [&](int u) { return W + (int64_t)ku(u) * ldw; },
                               [&](int u) { return ku(u) < K; });
            }
#pragma unroll
            for (int u = 0; u < UNR; u++)
#pragma unroll
                for (int d = 0; d < 4; d++) {
                    m[2 * d] = fmaxf(m[2 * d], fabsf(u2f(v[u][d] << 16)));
                    m[2 * d + 1] = fmaxf(m[2 * d + 1], fabsf(u2f(v[u][d] & 0xffff0000u)));
                }
        }
#pragma unroll
        for (int e = 0; e < 8; e++) {
            for (int off = 4; off < 64; off <<= 1) m[e] = fmaxf(m[e], __shfl_xor(m[e], off));
            if (lane < 4) smax[8 * ng + e][wave] = m[e];
        }
    }
    __syncthreads();
    if (t < 32) {
        float a = 0.0f, deq;
#pragma unroll
        for (int r = 0; r < QUANT4_WAVES; r++) a = fmaxf(a, smax[t][r]);
        sscale[t] = int4_scale(a, &deq);
        if (n0 + t < N) deq_out[n0 + t] = deq;
    }
    __syncthreads();
    char* const o = out + (int64_t)blockIdx.x * nfrag * 1024;
    if constexpr (TRANSPOSED) {
        float qs[4];
#pragma unroll
        for (int i = 0; i < 4; i++) qs[i] = sscale[8 * i + (lane >> 3)];
        for (int f = wave; f < nfrag; f += QUANT4_WAVES) {
            u32x4 v[4];
            load_fragment_rows(v, W, ldw, K, N, n0, 64 * f);
            store_fragment_rows(v, qs, o + (int64_t)f * 1024);
        }
    } else {
        float qs[8];
#pragma unroll
        for (int e = 0; e < 8; e++) qs[e] = sscale[8 * (lane & 3) + e];
        for (int f2 = wave; f2 * 2 < nfrag; f2 += QUANT4_WAVES) {
            u32x4 v[8];
            load_fragments_cols(v, W, ldw, K, N, n0, 128 * f2);
            store_fragments_cols(v, qs, o + (int64_t)f2 * 2048);
        }
    }
}

// [N, K] with a K that 16 wavefronts hold in registers, F fragments' worth of 8 columns each: a workgroup takes 8 columns and reads them
// once, where the kernel above reads a panel for its maxima and again to quantise it, a workgroup to 32 columns.  Bound: memory.  us a
// call, before -> now: 4096 x 11008 44.9 -> 22.9 (113 MB, 4.9 TB/s), 11008 x 4096 44.6 -> 31.0, 2048 x 7072 12.3 -> 10.3, 3200 x 704
// 12.6 -> 5.2, 6400 x 2048 25.4 -> 9.8, 512 x 512 5.6 -> 5.1 (the launch).  12 fragments are what 1024 threads have registers for.
template <int F>
__global__ __launch_bounds__(QUANT4_WAVES * 64) void quant4_pack_once_kernel(const char* __restrict__ W, int64_t ldw, int K, int N,
                                                                             char* __restrict__ out, int nfrag, float* deq_out) {
    __shared__ float smax[8][QUANT4_WAVES];
    __shared__ float sscale[8];
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), r8 = lane >> 3, c = lane & 7;
    const int n0 = blockIdx.x * 8;
    const char* const row = W + (int64_t)(n0 + r8) * ldw;
    u32x4 v[F];
#pragma unroll
    for (int j = 0; j < F; j++) {
        const int k0 = 64 * (wave + QUANT4_WAVES * j), k = k0 + 8 * c;
        v[j] = u32x4{0u, 0u, 0u, 0u};
        if (n0 + 8 <= N && k0 + 64 <= K) {  // (scalar)
            v[j] = load16<2>(row + (int64_t)k * 2);
        } else if (k0 < K) {
            u32x4 w[1];
            load16_rows<2>(w, (int64_t)k * 2, (int64_t)K * 2, [&](int) { return row; }, [&](int) { return n0 + r8 < N; });
            v[j] = w[0];
        }
    }
    float m = 0.0f;  // (fmaxf drops a NaN)
#pragma unroll
    for (int j = 0; j < F; j++)
#pragma unroll
        for (int d = 0; d < 4; d++) m = fmaxf(fmaxf(m, fabsf(u2f(v[j][d] << 16))), fabsf(u2f(v[j][d] & 0xffff0000u)));
    for (int off = 1; off < 8; off <<= 1) m = fmaxf(m, __shfl_xor(m, off));
    if (c == 0) smax[r8][wave] = m;
    __syncthreads();
    if (t < 8) {
        float a = 0.0f, deq;
#pragma unroll
        for (int w = 0; w < QUANT4_WAVES; w++) a = fmaxf(a, smax[t][w]);
        sscale[t] = int4_scale(a, &deq);
        if (n0 + t < N) deq_out[n0 + t] = deq;
    }
    __syncthreads();
    const float q = sscale[r8];
    char* const o = out + (int64_t)(blockIdx.x >> 2) * nfrag * 1024 + ((c >> 2) * 32 + 8 * (blockIdx.x & 3) + r8) * 16 + (c & 3) * 4;
#pragma unroll
    for (int j = 0; j < F; j++) {
        const int f = wave + QUANT4_WAVES * j;
        uint32_t d = 0;
#pragma unroll
        for (int e = 0; e < 4; e++)
            d |= (int4_of(u2f(v[j][e] << 16), q) | int4_of(u2f(v[j][e] & 0xffff0000u), q) << 4) << (8 * e);
        if (f < nfrag) *reinterpret_cast<uint32_t*>(o + (int64_t)f * 1024) = d;
    }
}

int launch_quantize_pack_int4(const void* W, int64_t ldw, int K, int N, int transpose, void* packed, float* deq_out,
                              hipStream_t st) {
    const int nfrag = (K + 255) / 256 * 4;
    const int npanels = (N + 31) / 32;
    if (nfrag == 4) {
        hipLaunchKernelGGL(transpose ? quant4_pack_short_kernel<true> : quant4_pack_short_kernel<false>, dim3(npanels),
                           dim3(transpose ? 256 : 128), 0, st, static_cast<const char*>(W), ldw, K, N, static_cast<char*>(packed), deq_out);
        return check_hip(hipGetLastError(), "quant4_pack_short_kernel launch");
    }
    const dim3 threads(QUANT4_WAVES * 64);
    const int held = (nfrag + QUANT4_WAVES - 1) / QUANT4_WAVES;  // fragments per wavefront
    if (transpose && held <= 12) {
        const auto kern = held <= 2 ? quant4_pack_once_kernel<2> : (held <= 4 ? quant4_pack_once_kernel<4> : (held <= 8 ? quant4_pack_once_kernel<8> : quant4_pack_once_kernel<12>));
        hipLaunchKernelGGL(kern, dim3(4 * npanels), threads, 0, st, static_cast<const char*>(W), ldw, K, N, static_cast<char*>(packed), nfrag, deq_out);
        return check_hip(hipGetLastError(), "quant4_pack_once_kernel launch");
    }
    if (transpose)
        hipLaunchKernelGGL(quant4_pack_kernel<true>, dim3(npanels), threads, 0, st, static_cast<const char*>(W), ldw, K, N,
                           static_cast<char*>(packed), nfrag, deq_out);
    else
        hipLaunchKernelGGL(quant4_pack_kernel<false>, dim3(npanels), threads, 0, st, static_cast<const char*>(W), ldw, K, N,
                           static_cast<char*>(packed), nfrag, deq_out);
    return check_hip(hipGetLastError(), "quant4_pack_kernel launch");
}

}  // namespace mmx
