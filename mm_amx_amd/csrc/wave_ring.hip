// C[:, n0:n1] = PP(A · Bpacked[:, n0:n1]) on small tiles, for products whose 128-row tiles (gemm_tile.hpp) would leave CUs idle or
// hold few k-iterations each: bf16, int8, and bf16 over int8 weights.
//
// What bounds such a product is how fast a CU pulls its tile's operands through its vector memory path, and the fixed parts of
// a launch; the matrix cores are mostly idle.  A 128x64 tile of the workgroup-wide ring takes 640 cycles per 128 bytes of K
// (38 bytes per clock) even if it is alone on the chip, behind a barrier per half-stage, and 4 us with nothing to do.  So here
//   - tiles are small (32x32, 32x64 or 64x64), hence many, and a CU pulls few bytes;
//   - every wavefront holds the whole tile in its accumulators, and K goes round the wavefronts, 128 bytes at a time: each
//     has an LDS slot of its own, waits for its own loads only and meets the others once, when the sums are added;
//   - a stage's operands are read into registers, the slot goes to the next stage's loads, and then come the products;
//   - where tiles are few and K is long, K is also cut into 2 or 4 slices for as many workgroups (the protocol and workspace
//     layout of the tile kernels' split).
// us a launch, best of the tile kernels -> this: bf16 40 x 1024 x 1024 8.1 -> 4.0, 900 x 1600 x 256 9.2 -> 4.8, 512 x 1024 x 1024
// 8.3 -> 5.2, 256 x 4096 x 4096 17.9 -> 16.4, 40 x 8192 x 1024 (four slices) 15.8 -> 7.0; gate/up pairs 100 x 1024 x 2 x 2048
// 13.3 -> 6.0; int8 weights 256 x 1024 x 1024 10.7 -> 4.3; int8 256 x 2048 x 2048 8.5 -> 5.2.
#include <cmath>
#include <type_traits>

#include "common.hpp"

namespace mmx {

namespace {

constexpr int AUX_SC1 = 16;  // cache policy operand of the buffer instructions: device scope
constexpr int MAX_SLICES = 4;

struct WaveRingArgs {
    const char* A;
    int64_t lda;  // bytes
    const char* Bp;
    int64_t panel_stride;
    int M;
    int kbytes;  // of a row of A
    int stages;  // of 128 bytes of a row of A, the last one maybe not full
    int npanels, n0, n1;
    int tiles_fast, rows_fast;          // tiles along the direction that runs fastest, and whether that is the rows'
    int units, units_per_xcd;           // (tile, slice) units
    int slices, per_slice;              // stages per slice
    char* ws_part;
    uint32_t* ws_cnt;
    Epilogue ep;
};

enum { BF16 = 0, W8 = 1, I8 = 3 };  // operand types: bf16, bf16 over int8 weights, int8

// One 16-byte load per lane to 1 KiB of LDS, from a scalar base and a 32-bit lane offset.
__device__ __forceinline__ void load_lds(uint32_t lds, uint32_t off, const char* base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(lds), "v"(off), "s"(base) : "memory");
}

// MB x NP: 32x32 blocks of the tile; NW: wavefronts
template <int T, int MB, int NP, int NW>
__global__ __launch_bounds__(NW * 64, MB * NP == 1 ? 4 : 2) void wave_ring_kernel(const WaveRingArgs g) {
    constexpr int A_ST = MB * 4096, BP_ST = T == W8 ? 2048 : 4096, ST = A_ST + NP * BP_ST;
    using acc_t = typename std::conditional<T == I8, int, float>::type;
    using accv = typename std::conditional<T == I8, i32x16, f32x16>::type;
    typedef acc_t acc4 __attribute__((ext_vector_type(4)));
    extern __shared__ __attribute__((aligned(1024))) char smem[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, g32 = lane >> 5;
    // Workgroup ids go round the 8 XCDs, and each gets a contiguous run of units: the slices of a tile are neighbours, and so are
    // the tiles that share the larger operand, which then comes to one XCD's L2 only (the other one to all of them).
    const int L = (blockIdx.x & 7) * g.units_per_xcd + (blockIdx.x >> 3);
    if (L >= g.units) return;
    const int tile = L / g.slices, slice = L - tile * g.slices;
    const int slow = tile / g.tiles_fast, fast = tile - slow * g.tiles_fast;
    const int tn = g.rows_fast ? slow : fast, tm = g.rows_fast ? fast : slow;
    const int m0 = tm * 32 * MB, panel0 = (g.n0 >> 5) + tn * NP;
    const int s0 = slice * g.per_slice, s1 = s0 + g.per_slice < g.stages ? s0 + g.per_slice : g.stages;
    const Epilogue& ep = g.ep;

    // ---- the wavefront's stages: s0 + wave, s0 + wave + NW, ... through its slot ------------------------------------
    // A: rows of 128 bytes, 16-byte chunk c of row r at position c ^ ((r >> 1) & 7) (an operand read of 32 rows then spreads
    // over the banks); a load covers 8 rows, whole lines.  B: fragments as they are packed.
    uint32_t aoff[MB * 4];
#pragma unroll
    for (int i = 0; i < MB * 4; i++) {
        const int row = 8 * i + (lane >> 3), last = g.M - 1 - m0;
        aoff[i] = (uint32_t)(row < last ? row : last) * (uint32_t)g.lda + (uint32_t)(((lane & 7) ^ ((4 * i + (lane >> 4)) & 7)) * 16);
    }
    const char* const abase = g.A + (int64_t)m0 * g.lda;
    const char* bbase[NP];
#pragma unroll
    for (int p = 0; p < NP; p++) bbase[p] = g.Bp + (int64_t)(panel0 + p < g.npanels ? panel0 + p : g.npanels - 1) * g.panel_stride;
    char* const slot = smem + wave * ST;
    const uint32_t slot_lds = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)slot);
    const int tail = g.kbytes & 127;  // bytes of the last stage, if it is not full: 16, 32, ... 112
    auto issue = [&](int st) __attribute__((always_inline)) {
        const char* const a = abase + (int64_t)st * 128;
        if (__builtin_expect(tail && st == g.stages - 1, 0)) {  // (scalar) chunks behind the end of the row are zero and not touched
#pragma unroll
            for (int i = 0; i < MB * 4; i++) {
                if (((lane & 7) ^ ((4 * i + (lane >> 4)) & 7)) * 16 < tail) load_lds(slot_lds + i * 1024, aoff[i], a);
                else *reinterpret_cast<u32x4*>(slot + i * 1024 + lane * 16) = u32x4{0u, 0u, 0u, 0u};
            }
        } else {
#pragma unroll
            for (int i = 0; i < MB * 4; i++) load_lds(slot_lds + i * 1024, aoff[i], a);
        }
#pragma unroll
        for (int p = 0; p < NP; p++)
#pragma unroll
            for (int i = 0; i < BP_ST / 1024; i++)
                load_lds(slot_lds + A_ST + p * BP_ST + i * 1024, lane * 16, bbase[p] + (int64_t)st * BP_ST + i * 1024);
    };
    accv acc[MB][NP];
#pragma unroll
    for (int b = 0; b < MB; b++)
#pragma unroll
        for (int p = 0; p < NP; p++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[b][p][v] = 0;
    // A stage's operands are read from LDS into registers, the slot goes to the next stage's loads, and then come the products: the
    // next stage is on its way while this one is multiplied.
    constexpr int BR = BP_ST / 1024;  // fragments of a panel in a stage
    u32x4 ra[4][MB], rb[BR][NP];
    auto read = [&]() __attribute__((always_inline)) {
        const char* const sa = slot + l32 * 128;
        const char* const sb = slot + A_ST + lane * 16;
        const int swz = (l32 >> 1) & 7;
#pragma unroll
        for (int s = 0; s < 4; s++) {  // 32 bytes of K of a row of A at a time
            const int chunk = T == W8 ? 4 * (s >> 1) + 2 * g32 + (s & 1) : 2 * s + g32;
#pragma unroll
            for (int i = 0; i < MB; i++) ra[s][i] = *reinterpret_cast<const u32x4*>(sa + i * 4096 + ((chunk ^ swz) * 16));
            if (s < BR)
#pragma unroll
                for (int p = 0; p < NP; p++) rb[s][p] = *reinterpret_cast<const u32x4*>(sb + p * BP_ST + s * 1024);
        }
    };
    auto multiply = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < 4; s++) {
            u32x4 b[NP];
#pragma unroll
            for (int p = 0; p < NP; p++) {
                if constexpr (T == W8) {
                    const u32x4 raw = rb[s >> 1][p];
                    b[p] = __builtin_bit_cast(u32x4, (s & 1) ? s8x8_to_bf16(raw[2], raw[3]) : s8x8_to_bf16(raw[0], raw[1]));
                } else {
                    b[p] = rb[s][p];
                }
            }
#pragma unroll
            for (int i = 0; i < MB; i++)
#pragma unroll
                for (int p = 0; p < NP; p++) {
                    if constexpr (T == I8)
                        acc[i][p] = __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(i32x4, b[p]), __builtin_bit_cast(i32x4, ra[s][i]), acc[i][p], 0, 0, 0);
                    else
                        acc[i][p] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, b[p]), __builtin_bit_cast(bf16x8, ra[s][i]), acc[i][p], 0, 0, 0);
                }
        }
    };
    const int first = s0 + wave;
    const int count = first < s1 ? (s1 - first + NW - 1) / NW : 0;
    if (count > 0) issue(first);

    // the per-column operands of this thread's outputs (units of four columns of a row, the same columns in every unit of a
    // thread) travel behind the first stage; gate/up pairs: column q of gate in deq, of up in bias
    const bool pairs = NP == 2 && (ep.steps & MMX_PP_SILU_GATE);
    constexpr int UNITS = MB * 32 * 8 * NP, UT = (UNITS + NW * 64 - 1) / (NW * 64);
    const int q0 = tid & (pairs ? 7 : 8 * NP - 1);  // unit of the row
    const int n0u = panel0 * 32 + 4 * q0;           // its first column of B
    float deq[4], bias[4], qs[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int c = n0u + e < g.n1 ? n0u + e : g.n1 - 1;
        deq[e] = (ep.steps & MMX_PP_DEQUANT) && ep.deq_oc ? ep.deq_oc[c] : ep.deq;
        bias[e] = (ep.steps & MMX_PP_BIAS) ? ep.bias[c] : 0.0f;
        qs[e] = (ep.steps & MMX_PP_QUANT) && ep.q_oc ? ep.q_oc[c] : ep.q;
        if (pairs) bias[e] = (ep.steps & MMX_PP_DEQUANT) && ep.deq_oc ? ep.deq_oc[c + 32 < g.n1 ? c + 32 : g.n1 - 1] : ep.deq;
    }

    for (int i = 0; i < count; i++) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        read();
        if (i + 1 < count) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // every read of the slot is done
            issue(first + (i + 1) * NW);
        }
        multiply();
    }

    // ---- the wavefronts' sums meet in LDS, 4 registers (4 consecutive columns of a row) to a 16-byte piece ------------
    // piece (block, i, lane) sits at lane position l32 ^ (2 i + g32): units of one row are then read from different banks
    __syncthreads();
    const int live = s1 - s0 < NW ? s1 - s0 : NW;  // wavefronts that had a stage
    if (wave < live) {
#pragma unroll
        for (int b = 0; b < MB; b++)
#pragma unroll
            for (int p = 0; p < NP; p++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    acc4 v = {acc[b][p][4 * i], acc[b][p][4 * i + 1], acc[b][p][4 * i + 2], acc[b][p][4 * i + 3]};
                    *reinterpret_cast<acc4*>(smem + ((wave * MB + b) * NP + p) * 4096 + i * 1024 + ((l32 ^ (2 * i + g32)) + 32 * g32) * 16) = v;
                }
    }
    __syncthreads();
    auto sum_of = [&](int m, int p, int q) __attribute__((always_inline)) {  // row m, panel p, columns 4 q .. 4 q + 3 of it
        const char* at = smem + ((m >> 5) * NP + p) * 4096 + (q >> 1) * 1024 + (((m & 31) ^ q) + 32 * (q & 1)) * 16;
        acc4 r = *reinterpret_cast<const acc4*>(at);
        for (int w = 1; w < live; w++) r += *reinterpret_cast<const acc4*>(at + w * (MB * NP * 4096));
        return r;
    };
    acc4 sum[UT];
#pragma unroll
    for (int u = 0; u < UT; u++) {
        const int idx = tid + u * NW * 64, m = idx / (8 * NP), q = idx & (8 * NP - 1);
        if (idx < UNITS && !pairs) sum[u] = sum_of(m, q >> 3, q & 7);
    }
    if (g.slices > 1) {  // (never with pairs)
        constexpr int UNIT = MB * NP * 4096;  // bytes of a tile's sums
        __amdgpu_buffer_rsrc_t parts = __builtin_amdgcn_make_buffer_rsrc(g.ws_part + (int64_t)tile * g.slices * UNIT, 0, g.slices * UNIT, 0x00020000);
#pragma unroll
        for (int u = 0; u < UT; u++)
            if (tid + u * NW * 64 < UNITS)
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, sum[u]), parts, slice * UNIT + (tid + u * NW * 64) * 16, 0, AUX_SC1);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // every store of this wave has been acknowledged
        __syncthreads();                                  // ... and every read of the scratch is done
        volatile uint32_t* flag = reinterpret_cast<volatile uint32_t*>(smem);
        if (tid == 0) *flag = atomicInc(g.ws_cnt + tile, (uint32_t)g.slices - 1u);
        __syncthreads();
        if (*flag != (uint32_t)g.slices - 1u) return;  // (the last to arrive adds; nobody waits for anybody)
        asm volatile("" ::: "memory");
#pragma unroll
        for (int u = 0; u < UT; u++) {
            const int idx = tid + u * NW * 64;
            if (idx < UNITS) {
                u32x4 v[MAX_SLICES];
#pragma unroll
                for (int sl = 0; sl < MAX_SLICES; sl++)
                    if (sl < g.slices) v[sl] = __builtin_amdgcn_raw_buffer_load_b128(parts, sl * UNIT + idx * 16, 0, AUX_SC1);
                acc4 r = __builtin_bit_cast(acc4, v[0]);
#pragma unroll
                for (int sl = 1; sl < MAX_SLICES; sl++)
                    if (sl < g.slices) r += __builtin_bit_cast(acc4, v[sl]);  // in slice order, whoever came last
                sum[u] = r;
            }
        }
    }
    // ---- post-op and store, four columns of a row at a time --------------------------------------------------------
    const int out_n1 = pairs ? g.n1 >> 1 : g.n1;
#pragma unroll
    for (int u = 0; u < UT; u++) {
        const int idx = tid + u * NW * 64;
        const int m = idx / (pairs ? 8 : 8 * NP), q = q0;
        const int row = m0 + m;
        if (m >= MB * 32 || row >= g.M) continue;
        const int n = pairs ? (panel0 >> 1) * 32 + 4 * q : n0u;  // first column of the unit in C
        if (n >= out_n1) continue;
        float r[4];
        acc4 raw = {};
        if (pairs) {
            const char* at = smem + (m >> 5) * NP * 4096 + (q >> 1) * 1024 + (((m & 31) ^ q) + 32 * (q & 1)) * 16;
            acc4 gt = *reinterpret_cast<const acc4*>(at), up = *reinterpret_cast<const acc4*>(at + 4096);
            for (int w = 1; w < live; w++) {
                gt += *reinterpret_cast<const acc4*>(at + w * (MB * NP * 4096));
                up += *reinterpret_cast<const acc4*>(at + w * (MB * NP * 4096) + 4096);
            }
#pragma unroll
            for (int e = 0; e < 4; e++) {
                float a = (float)gt[e], b = (float)up[e];
                if (ep.steps & MMX_PP_DEQUANT) {  // compressed weights: gate and up each by the scale of its own column
                    a = a * deq[e];
                    b = b * bias[e];
                }
                r[e] = silu(a) * b;
            }
        } else {
            raw = sum[u];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                r[e] = (float)raw[e];  // (int32: vcvtdq2ps, round to nearest even)
                if (ep.steps & MMX_PP_DEQUANT) r[e] = r[e] * deq[e];
                if (ep.steps & MMX_PP_BIAS) r[e] = r[e] + bias[e];
                if (ep.steps & MMX_PP_GELU) r[e] = gelu_erf_minimax(r[e]);
                if (ep.steps & MMX_PP_QUANT) r[e] = r[e] * qs[e];
            }
        }
        char* const crow = ep.C + (int64_t)row * ep.ldc;
        auto put = [&](auto bytes_c, const uint32_t (&w)[4]) __attribute__((always_inline)) {  // 4 elements of SZ bytes, packed in w
            constexpr int SZ = decltype(bytes_c)::value;
            char* const dst = crow + (int64_t)n * SZ;
            if (n + 4 <= out_n1) {  // (the hardware takes such stores whole, whatever the alignment)
                __builtin_memcpy(__builtin_assume_aligned(dst, SZ), w, 4 * SZ);
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (n + e < out_n1) {
                        const uint32_t x = w[e * SZ / 4] >> (8 * ((e * SZ) & 3));
                        __builtin_memcpy(dst + e * SZ, &x, SZ);
                    }
            }
        };
        using std::integral_constant;
        if (ep.out_dtype == MMX_BF16) {
            const uint32_t w[4] = {(uint32_t)to_bf16(r[0]) | (uint32_t)to_bf16(r[1]) << 16, (uint32_t)to_bf16(r[2]) | (uint32_t)to_bf16(r[3]) << 16, 0, 0};
            put(integral_constant<int, 2>{}, w);
        } else if (ep.out_dtype == MMX_I8) {
            const uint32_t w[4] = {to_s8_sat_x4(r[0], r[1], r[2], r[3]), 0, 0, 0};
            put(integral_constant<int, 1>{}, w);
        } else {
            uint32_t w[4];
#pragma unroll
            for (int e = 0; e < 4; e++) w[e] = T == I8 && ep.out_dtype == MMX_I32 ? (uint32_t)(int)raw[e] : f2u(r[e]);
            put(integral_constant<int, 4>{}, w);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}


typedef void (*WaveRingKernel)(const WaveRingArgs);
template <int T, int MB, int NP, int NW>
int launch_cfg(const WaveRingArgs& g, hipStream_t st) {
    constexpr int slots = NW * (MB * 4096 + NP * (T == W8 ? 2048 : 4096)), red = NW * MB * NP * 4096, lds = slots > red ? slots : red;
    static_assert(lds <= 160 * 1024, "LDS of a CU");
    static std::atomic<uint64_t> attr_done{0};
    const WaveRingKernel kern = wave_ring_kernel<T, MB, NP, NW>;
    const int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(kern), lds, attr_done);
    if (rc) return rc;
    char name[96], split[16] = "";
    if (g.slices > 1) snprintf(split, sizeof split, "_ksplit%d", g.slices);
    snprintf(name, sizeof name, "gemm_%s_%dx%d_wave_ring%s_out_%s%s", T == I8 ? "i8" : (T == W8 ? "w8" : "bf16"), 32 * MB, 32 * NP, NW == 4 ? "4w" : "",
             g.ep.out_dtype == MMX_F32 ? "f32" : (g.ep.out_dtype == MMX_BF16 ? "bf16" : (g.ep.out_dtype == MMX_I8 ? "i8" : "i32")), split);
    note_kernel(name);
    hipLaunchKernelGGL(kern, dim3(g.units_per_xcd * 8), dim3(NW * 64), lds, st, g);
    return check_hip(hipGetLastError(), "wave_ring_kernel launch");
}
}  // namespace

namespace {

// The four forms, and the model that chooses between them and the tile kernels (us, fitted to 9000 timings over 840 shapes: M 33
// to 2048, K 256 to 11008, N 256 to 16384, the three types and gate/up pairs; 12 % rms): a fixed part, the larger of what the
// busiest CU pulls and what all of them read from memory plus 0.3 of the smaller, another round of workgroups, the slices'
// meeting, and the blocks a CU finishes.  On 387 shapes drawn from the same ranges small tiles are taken on 250, at 0.62 of the time
// of the best forced tile on average (0.32 to 1.04; profiles/small_tiles_against_tile_kernels.txt).  (A 64x32 tile, and four
// wavefronts on a 32x64 one, gained 0.2 % more.  128x64 and 64x128 tiles, four wavefronts with the whole tile each, are behind the
// tile kernels' 128x64 where those are used: 512 x 4096 x 4096 int8 19.8 / 19.0 us against 17.6 with a slot per wavefront,
// 22.7 / 20.4 with one ring for the workgroup and half the LDS reads; what a CU pulls from L2 bounds both.)
struct Form {
    int mb, np, nw, per_cu;  // per_cu: workgroups that a CU holds
    float us_per_kib;        // pulled by one CU
    // Over int8 weights (stages of fewer bytes, and the conversion) the chosen form's estimate is held against the tile kernels' times
    // e^x, x = w8[0] + w8[1] ln(stages of a slice / 64) + w8[2] ln(workgroups on the busiest CU) + w8[3] ln(MB of A x MB of B / 400)
    // + w8[4] with slices: fitted to 307 shapes near the line, on which the estimate was 7 to 16 % off, and is 4 to 9 so.
    float w8[5];
};
constexpr Form FORMS[4] = {{1, 1, 8, 2, 0.0079f, {0.81f, -0.19f, -0.22f, 0.18f, 0.0f}},
                           {1, 2, 8, 1, 0.0093f, {0.50f, -0.15f, -0.185f, 0.135f, -0.10f}},
                           {2, 2, 8, 1, 0.0105f, {0.39f, -0.255f, -0.10f, 0.115f, -0.045f}},
                           {2, 2, 4, 2, 0.0109f, {0.46f, -0.245f, -0.27f, 0.12f, -0.095f}}};

// The form is taken where its estimate is below this share of the tile kernels'.  Over 800 shapes whose two estimates are within 0.6 to
// 1.35 of each other small tiles are taken on 594, at 0.77 of the tile kernels' time on average, 10 of them more than 3 % slower (at most
// 14 %).  Without the corrections for int8 weights, here and in the tile kernels' estimate, and a share of 0.93, 119 of 700 such shapes
// stayed with the tile kernels though small tiles were more than 3 % faster (up to 1.5 times), 52 with them; with the margin that a K split has
// to win by counted in the tile kernels' estimate, int8 weights 895 x 9760 x 1792 went from 51 to 63 us.
constexpr float WIN = 0.95f;

struct WaveRingPlan {
    int form, slices;
    float us;
    int on_cu;  // workgroups on the busiest CU
};

WaveRingPlan choose_form(int type, int M, int K, int Ncols, bool pairs, int k_splits, size_t ws_bytes) {
    const int cus = num_cus(), es = type == I8 ? 1 : 2, bs = type == BF16 ? 2 : 1;
    const int stages = (int)(((int64_t)K * es + 127) / 128), panels = (Ncols + 31) / 32;
    const float mb_a = (float)M * K * es * 1e-6f, mb_b = (float)K * Ncols * bs * 1e-6f, mb_read = mb_a + mb_b;
    WaveRingPlan best = {-1, 1, 1e30f, 0};
    for (int f = 0; f < 4; f++) {
        const Form& c = FORMS[f];
        if (pairs && c.np != 2) continue;
        if (f == 3 && type != W8 && !pairs) continue;  // (elsewhere the tile kernels are ahead wherever it would be)
        const int64_t tiles = (int64_t)((M + 32 * c.mb - 1) / (32 * c.mb)) * ((panels + c.np - 1) / c.np);
        if (tiles > (1 << 24)) continue;
        for (int S = 1; S <= MAX_SLICES; S *= 2) {
            const int per_slice = (stages + S - 1) / S;
            if (S > 1 && (pairs || k_splits == 1 || tiles * S > 2 * cus || tiles > WS_MAX_TILES || (S - 1) * per_slice >= stages ||
                          WS_COUNTER_BYTES + (size_t)tiles * S * c.mb * c.np * 4096 > ws_bytes)) continue;
            const int on_cu = (int)((tiles * S + cus - 1) / cus), rounds = (int)((tiles * S + cus * c.per_cu - 1) / (cus * c.per_cu));
            const float kib = (float)per_slice * (c.mb * 4.0f + c.np * (type == W8 ? 2.0f : 4.0f));
            const float pull = on_cu * kib * c.us_per_kib, memory = 0.134f * mb_read;
            const float us = 2.5f + (pull > memory ? pull + 0.3f * memory : memory + 0.3f * pull) + 1.4f * (rounds - 1) +
                             (S > 1 ? 1.8f : 0.0f) + 0.43f * c.mb * c.np * on_cu;
            if (us < best.us) best = {f, S, us, on_cu};
        }
    }
    if (type == W8 && best.form >= 0) {
        const float* const w = FORMS[best.form].w8;
        best.us *= expf(w[0] + w[1] * logf((stages + best.slices - 1) / best.slices * (1.0f / 64)) + w[2] * logf((float)best.on_cu) +
                        w[3] * logf(mb_a * mb_b * (1.0f / 400)) + (best.slices > 1 ? w[4] : 0.0f));
    }
    return best;
}

}  // namespace

static bool wave_ring_can(int type, int K, bool aligned) {
    const int64_t kbytes = (int64_t)K * (type == I8 ? 1 : 2);
    return aligned && kbytes % 16 == 0 && kbytes >= 128 && K <= (1 << 24);
}

// Takes the call (returns MMX_OK or an error) or leaves it to the tile kernels (returns 1), whose own model says tiles_us.
// type: 0 bf16, 1 bf16 over int8 weights, 3 int8.  The choice depends on the shape and on the workspace: what it holds bounds the
// slices, and a call without one has k_splits = 1.
int launch_wave_ring(int type, const void* A, int64_t lda, const void* Bp, int M, int K, int N, int n0, int n1, const Epilogue& ep,
                     const SplitRequest& rq, float tiles_us, hipStream_t st) {
    const bool pairs = (ep.steps & MMX_PP_SILU_GATE) != 0;
    // (32-bit offsets within a tile's rows)
    if (!wave_ring_can(type, K, ((reinterpret_cast<uintptr_t>(A) | (uintptr_t)lda) & 15) == 0) || lda >= (1 << 24)) return 1;
    const WaveRingPlan p = choose_form(type, M, K, n1 - n0, pairs, rq.ws ? rq.k_splits : 1, rq.ws_bytes);
    if (p.form < 0 || p.us >= WIN * tiles_us) return 1;
    const Form& c = FORMS[p.form];
    const int es = type == I8 ? 1 : 2;
    const int panels = ((n1 + 31) >> 5) - (n0 >> 5), tiles_m = (M + 32 * c.mb - 1) / (32 * c.mb), tiles_n = (panels + c.np - 1) / c.np;
    WaveRingArgs g;
    g.A = static_cast<const char*>(A);
    g.lda = lda;
    g.Bp = static_cast<const char*>(Bp);
    g.M = M;
    g.kbytes = K * es;
    g.stages = (g.kbytes + 127) / 128;
    g.panel_stride = (type == BF16 ? (int64_t)g.stages : (int64_t)((K + 127) / 128)) * 4096;
    g.npanels = (N + 31) / 32;
    g.n0 = n0;
    g.n1 = n1;
    g.rows_fast = (int64_t)M * es <= (int64_t)(n1 - n0) * (type == BF16 ? 2 : 1);
    g.tiles_fast = g.rows_fast ? tiles_m : tiles_n;
    g.slices = p.slices;
    g.per_slice = (g.stages + p.slices - 1) / p.slices;
    g.units = tiles_m * tiles_n * p.slices;
    g.units_per_xcd = (g.units + 7) / 8;
    g.ws_cnt = reinterpret_cast<uint32_t*>(rq.ws);
    g.ws_part = rq.ws ? rq.ws + WS_COUNTER_BYTES : nullptr;
    g.ep = ep;
    auto launch = [&](auto type_c) {
        constexpr int T = decltype(type_c)::value;
        switch (p.form) {
        case 0: return launch_cfg<T, 1, 1, 8>(g, st);
        case 1: return launch_cfg<T, 1, 2, 8>(g, st);
        case 2: return launch_cfg<T, 2, 2, 8>(g, st);
        }
        if constexpr (T != I8) return launch_cfg<T, 2, 2, 4>(g, st);
        return set_error(MMX_E_UNSUPPORTED, "no such form for int8");
    };
    using std::integral_constant;
    return type == I8 ? launch(integral_constant<int, I8>{}) : (type == W8 ? launch(integral_constant<int, W8>{}) : launch(integral_constant<int, BF16>{}));
}

// Bytes of workspace the call above can use (0: no slices), or -1 if it would leave the call to the tile kernels.  Rows are counted in
// whole 64s: an upper bound, and one answer for counts of rows in the same 64 that get the same form and slices.  (Rows of A that
// are not aligned go to the masked pipeline there, which takes no slices.)
int64_t wave_ring_workspace_bytes(int type, int M, int K, int Ncols, bool pairs, int k_splits, size_t most, float tiles_us) {
    if (!wave_ring_can(type, K, true)) return -1;
    const WaveRingPlan p = choose_form(type, M, K, Ncols, pairs, k_splits, most);
    if (p.form < 0 || p.us >= WIN * tiles_us) return -1;
    const Form& c = FORMS[p.form];
    if (p.slices == 1) return 0;
    return (int64_t)(WS_COUNTER_BYTES + (size_t)((M + 63) / 64 * 2 / c.mb) * (((Ncols + 31) / 32 + c.np - 1) / c.np) * p.slices * c.mb * c.np * 4096);
}

}  // namespace mmx
