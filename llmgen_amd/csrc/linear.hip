// linear.hip -- y [M, N] = x [M, K] * w [N, K]^T in the reference CPU backend's order (hip_linear).
//
// The reference (src/backend/cpu/linear.zig:7-28) forms every output as one f32 sum over k = 0 .. K-1, a rounded
// multiply and a rounded add per term.  The product of two bf16 values has at most 16 significant bits, so f32 holds
// it exactly unless it leaves the exponent range; then multiply-and-add is a fused multiply-add, and
// v_mfma_f32_16x16x4_f32 is exactly that: four fused multiply-adds per output, k ascending, each rounded to nearest
// even, denormals kept (the bf16 matrix instructions are not: they add several products before they round).  The
// K sum cannot be split and its order cannot change, so the work is spread over outputs only.
//
// Exactness is checked, not assumed: each staged value must be zero or lie in a window of 128 exponents
// (x: [2^-63, 2^65), w: [2^-67, 2^61)), so that a product is below 2^126 and a multiple of 2^-144.  The check is an
// add and an AND per pair of values (adding 64 or 68 to the exponent field sets its top bit exactly inside the
// window); zeros fail it and are sorted out in a second look at the rows that were staged.  A tile that holds any
// other value (infinities and NaN among them) is computed again with the products of the chunks that hold one rounded
// before they are added.  If one of the first two chunks holds one, the first pass ends there.  631 x 1024 x 3072: 46 us
// with none, 86 with one column of x outside, 190 with one value in every 16 of k (the plain multiply-add kernel that
// these replace: 368 with any input); 2048 x 6144 x 2048: 371, 502 and 1084 us (1704); 32 x 151936 x 1024: 96, 136 and
// 241 us (431).
//
// What bounds it.  f32 matrix instructions run at 155 TFLOP/s (1/16 of bf16) and share their issue slots with the
// VALU: measured, every VALU instruction beside them adds its full 4 cycles.  So operands are widened to f32 once per
// tile on their way into LDS (bf16 rows -> registers -> f32 rows in LDS, laid out so that one ds_read_b128 gives a
// lane its operand of four instructions) and the product loop holds nothing but LDS reads and matrix instructions.
// Loads run PF chunks ahead of the staging, staging two chunks ahead of the products and the LDS reads one chunk
// ahead, so that one barrier per chunk is all a wave waits for.
//
// Small steps (decode) are bound by the chain of one output instead: 8 cycles per k, 3.4 us at K = 1024.  There a
// wave owns a single 16 x 16 tile and staging is left to producer waves of the same workgroup, which sit on the other
// SIMDs, so the chain's SIMD does nothing else (K = 3072, N = 1024, 32 rows: 16.3 us; with the staging in the same wave
// 26 us; one output per lane with 256-column workgroups, as multiplies and adds: 343 us).
#include "hip_common.h"

#include <algorithm>
#include <type_traits>
#include <utility>

#pragma clang fp contract(off)

namespace {

// Added to a pair of bf16 values, sets bit 14 of each half exactly where the exponent field lies in the window.
constexpr uint32_t LIN_X_BIAS = 0x20002000u;  // exponent field 64..191: [2^-63, 2^65)
constexpr uint32_t LIN_W_BIAS = 0x22002200u;  // exponent field 60..187: [2^-67, 2^61)
constexpr uint32_t LIN_IN = 0x40004000u;

// One value: zero, or inside the window of its operand.
__device__ __forceinline__ bool lin_half_ok(uint32_t h, uint32_t bias) {
    return (h & 0x7fffu) == 0 || (((h & 0x7fffu) + (bias & 0x7fffu)) & 0xC000u) == 0x4000u;
}

// One launch computes up to three products of the same x (q, k and v; gate and up): their column tiles follow each
// other in the grid, a tile lies in one of them.  With `res`, y = res + (the product rounded to bf16), rounded again:
// what a separate add of the stored product gives.
struct LinOut {
    void *y;
    const bf16_t *w;
    int N;
};
struct LinArgs {
    LinOut out[3];
    const bf16_t *x, *res;
    int M, K, y_f32, vec_out, tiles_m;
};
// The product that column tile `tn` (tiles of TN columns) belongs to, and its first column there.
__device__ __forceinline__ LinOut lin_out(const LinArgs &a, int tn, int TN, int &n0) {
    LinOut o = a.out[0];
    int first = (o.N + TN - 1) / TN;
    if (tn >= first) {
        tn -= first;
        o = a.out[1];
        first = (o.N + TN - 1) / TN;
        if (tn >= first) {
            tn -= first;
            o = a.out[2];
        }
    }
    n0 = tn * TN;
    return o;
}
long lin_cols(const LinArgs &a, int TN) {
    long t = 0;
    for (const LinOut &o : a.out) t += (o.N + TN - 1) / TN;
    return t;
}
__device__ __forceinline__ float lin_bf16(bf16_t b) { return __builtin_bit_cast(float, (uint32_t)b << 16); }
__device__ __forceinline__ float lin_round(float f) {
    return lin_bf16(__builtin_bit_cast(bf16_t, (__bf16)f));
}
__device__ __forceinline__ void lin_put(const LinArgs &a, const LinOut &out, int m, int n, float v) {
    const long o = (long)m * out.N + n;
    if (a.res) v = lin_bf16(a.res[o]) + lin_round(v);
    if (a.y_f32)
        static_cast<float *>(out.y)[o] = v;
    else
        static_cast<bf16_t *>(out.y)[o] = __builtin_bit_cast(bf16_t, (__bf16)v);
}

// The order of one step's instructions: the LDS reads spread between the matrix instructions, then the staging's VALU
// work in one piece, then its LDS writes spread likewise.  A wave issues in order and its LDS queue is short, so reads
// or writes issued together hold up the matrix instructions behind them, and every change between VALU and matrix
// instructions costs 8 cycles (as the compiler orders a step by itself: 997 x 1024 x 3072 70.9 us, so 56.5 us).
template <int READS, int WRITES, int PRODUCTS>
__device__ __forceinline__ void lin_interleave() {
    constexpr int PER = PRODUCTS / (READS + WRITES) > 0 ? PRODUCTS / (READS + WRITES) : 1;
#pragma unroll
    for (int i = 0; i < READS; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, PER, 0);  // matrix instructions
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);    // LDS read
    }
    if (WRITES) __builtin_amdgcn_sched_group_barrier(0x002, 64, 0);  // VALU
#pragma unroll
    for (int i = 0; i < WRITES; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, PER, 0);
        __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);  // LDS write
    }
    __builtin_amdgcn_sched_group_barrier(0x008, PRODUCTS, 0);
}

// A workgroup's tile: WM x WN waves of MT x NT blocks of 16 x 16 outputs, PW extra waves that only stage (0: every
// wave stages), KC values of k per LDS chunk.
template <int MT, int NT, int WM, int WN, int PW, int KC>
struct LinTile {
    static constexpr int TM = WM * MT * 16, TN = WN * NT * 16, ROWS = TM + TN;
    static constexpr int WAVES = WM * WN, THREADS = (WAVES + PW) * 64, STAGERS = (PW ? PW : WAVES) * 64;
    static constexpr int UNITS = KC / 16;  // 16 consecutive k of a row: one staging slot
    static constexpr int WORK = ROWS * UNITS, SLOTS = (WORK + STAGERS - 1) / STAGERS;
    static constexpr int STRIDE = KC + 4;  // f32 per staged row
    // whether slot s of a staging thread has work (whole waves drop out of the last slot)
    static __device__ __forceinline__ bool has(int id, int s) {
        return (s + 1) * STAGERS <= WORK || id + s * STAGERS < WORK;
    }
};

// "At least two waves a SIMD" keeps the sums in ordinary registers, where the VALU adds to them without moves.  Not so in
// the kernels with producer waves, which are 2 % faster without it (32 x 1024 x 3072: 15.9 and 16.3 us; with values outside
// the window throughout 83 and 58 us).  32 x 32 tiles, many to a CU, fit four waves a SIMD, as many as the LDS holds
// (100 x 9001 x 200: 12.4 us, 13.4 with three).
template <int MT, int NT, int WM, int WN, int PW, int KC, int PF>
__global__ void __launch_bounds__((WM * WN + PW) * 64, PW ? 1 : WM * WN * MT * NT == 4 ? 4 : 2)
    linear_kernel(const LinArgs a) {
    using T = LinTile<MT, NT, WM, WN, PW, KC>;
    static_assert(PF % 2 == 0, "chunk parity names the LDS buffer");
    __shared__ __attribute__((aligned(16))) float lds[2][T::ROWS * T::STRIDE];
    __shared__ int flag[3];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (tid < 2) flag[tid] = 0;
    // tiles in order of columns, each XCD (block index mod 8) a contiguous range of them
    const int tiles = gridDim.x;
    const int per = tiles >> 3, rem = tiles & 7, xcd = blockIdx.x & 7, at = blockIdx.x >> 3;
    const int tile = xcd * per + min(xcd, rem) + at;
    int n0;
    const LinOut out = lin_out(a, tile / a.tiles_m, T::TN, n0);
    const int m0 = tile % a.tiles_m * T::TM;
    const int K = a.K, full = K / KC, tail = K - full * KC;

    // ---- staging: raw bf16 rows -> f32 in LDS, each 16 k of a row as [k % 4][k / 4]
    const int sid = PW ? tid - T::WAVES * 64 : tid;
    const bf16_t *src[T::SLOTS];
    int dst[T::SLOTS], koff[T::SLOTS];
    bool is_w[T::SLOTS];
    u32x4_t raw[PF][T::SLOTS][2];
    int ahead = 0;  // next chunk to load
    bool bad = false;
    auto begin = [&]() __attribute__((always_inline)) {
        ahead = 0;
#pragma unroll
        for (int s = 0; s < T::SLOTS; ++s) {
            const int i = sid + s * T::STAGERS, row = min(i / T::UNITS, T::ROWS - 1), u = i % T::UNITS;
            is_w[s] = row < T::TN;
            const long r = is_w[s] ? min(n0 + row, out.N - 1) : min(m0 + row - T::TN, a.M - 1);
            koff[s] = u * 16;
            src[s] = (is_w[s] ? out.w : a.x) + r * K + u * 16;
            dst[s] = row * T::STRIDE + u * 16;
        }
    };
    auto load = [&](u32x4_t (&r)[T::SLOTS][2]) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < T::SLOTS; ++s)
            if (T::has(sid, s))
#pragma unroll
                for (int h = 0; h < 2; ++h) r[s][h] = ld16(src[s] + h * 8);
        const int step = ++ahead < full ? KC : 0;  // past the last full chunk: that chunk again
#pragma unroll
        for (int s = 0; s < T::SLOTS; ++s) src[s] += step;
    };
    // the last K % KC values of each row, zeros beyond them; the pointers stand at the last full chunk (or at k 0)
    auto load_tail = [&](u32x4_t (&r)[T::SLOTS][2]) {
        const int base = full > 0 ? KC : 0;
#pragma unroll
        for (int s = 0; s < T::SLOTS; ++s)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                r[s][h] = u32x4_t{0u, 0u, 0u, 0u};
                if (T::has(sid, s) && koff[s] + h * 8 < tail) r[s][h] = ld16(src[s] + base + h * 8);
            }
    };
    auto stage_put = [&](const u32x4_t (&r)[T::SLOTS][2], int buf) __attribute__((always_inline)) {
        uint32_t in = LIN_IN;
#pragma unroll
        for (int s = 0; s < T::SLOTS; ++s) {
            if (!T::has(sid, s)) continue;
            const uint32_t bias = is_w[s] ? LIN_W_BIAS : LIN_X_BIAS;
            float f[16];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
#pragma unroll
                for (int i = 0; i < 4; ++i) in &= r[s][h][i] + bias;
                unpack_bf16x8(r[s][h], f + 8 * h);
            }
#pragma unroll
            for (int q = 0; q < 4; ++q)
                *reinterpret_cast<f32x4_t *>(&lds[buf][dst[s] + q * 4]) = f32x4_t{f[q], f[4 + q], f[8 + q], f[12 + q]};
        }
        return in;
    };
    auto stage_check = [&](const u32x4_t (&r)[T::SLOTS][2], uint32_t in) __attribute__((always_inline)) {
        if (__builtin_expect(__ballot(in != LIN_IN) != 0, 0)) {
#pragma unroll
            for (int s = 0; s < T::SLOTS; ++s) {
                if (!T::has(sid, s)) continue;
                const uint32_t bias = is_w[s] ? LIN_W_BIAS : LIN_X_BIAS;
                for (int h = 0; h < 2; ++h)
                    for (int i = 0; i < 4; ++i) {
                        const uint32_t d = r[s][h][i];
                        bad |= !(lin_half_ok(d & 0xffffu, bias) && lin_half_ok(d >> 16, bias));
                    }
            }
        }
    };
    auto stage = [&](const u32x4_t (&r)[T::SLOTS][2], int buf) { stage_check(r, stage_put(r, buf)); };

    // ---- products
    const int wm = wave % WM, wn = wave / WM;
    const int frag = (lane & 15) * T::STRIDE + (lane >> 4) * 4;
    const int wbase = wn * NT * 16 * T::STRIDE + frag, xbase = (T::TN + wm * MT * 16) * T::STRIDE + frag;
    f32x4_t acc[MT][NT];
    auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int n = 0; n < NT; ++n) acc[m][n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    };
    f32x4_t wf[2][T::UNITS][NT], xf[2][T::UNITS][MT];
    auto fetch = [&](int set) __attribute__((always_inline)) {
        const float *b = lds[set];
#pragma unroll
        for (int s = 0; s < T::UNITS; ++s) {
#pragma unroll
            for (int n = 0; n < NT; ++n)
                wf[set][s][n] = *reinterpret_cast<const f32x4_t *>(b + wbase + n * 16 * T::STRIDE + s * 16);
#pragma unroll
            for (int m = 0; m < MT; ++m)
                xf[set][s][m] = *reinterpret_cast<const f32x4_t *>(b + xbase + m * 16 * T::STRIDE + s * 16);
        }
    };
    auto compute = [&](int set) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < T::UNITS; ++s)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int m = 0; m < MT; ++m)
#pragma unroll
                    for (int n = 0; n < NT; ++n)
                        acc[m][n] =
                            __builtin_amdgcn_mfma_f32_16x16x4f32(wf[set][s][n][j], xf[set][s][m][j], acc[m][n], 0, 0, 0);
    };

    // The first `units` units of a staged chunk; `apart`: with separate multiplies and adds, as the reference does.
    // v_mfma_f32_16x16x1 takes the same operands and gives the products of its four k apart, each fma(x, w, +0) and so
    // rounded once; the VALU adds them k by k.  (A product of -0 may come out as +0, but no sum is ever -0, so that does
    // not show.)  96 cycles for 16 x 16 x 4 products on one SIMD, against 32 fused and 128 as VALU multiplies and adds.
    auto products = [&](const float *b, int units, bool apart) __attribute__((always_inline)) {
#pragma unroll 1
        for (int s = 0; s < units; ++s) {
            f32x4_t w4[NT], x4[MT];
#pragma unroll
            for (int n = 0; n < NT; ++n)
                w4[n] = *reinterpret_cast<const f32x4_t *>(b + wbase + n * 16 * T::STRIDE + s * 16);
#pragma unroll
            for (int m = 0; m < MT; ++m)
                x4[m] = *reinterpret_cast<const f32x4_t *>(b + xbase + m * 16 * T::STRIDE + s * 16);
            if (apart) {
                f32x16_t p[2];  // one block's products form while the other's are added
                constexpr int ALL = 4 * MT * NT;
#pragma unroll
                for (int t = 0; t <= ALL; ++t) {
                    if (t < ALL)
                        p[t & 1] = __builtin_amdgcn_mfma_f32_16x16x1f32(w4[t % NT][t / (MT * NT)],
                                                                        x4[t / NT % MT][t / (MT * NT)], f32x16_t{}, 0, 0, 0);
                    if (t > 0) {
                        f32x4_t &sum = acc[(t - 1) / NT % MT][(t - 1) % NT];
#pragma unroll
                        for (int i = 0; i < 16; ++i) sum[i & 3] = sum[i & 3] + p[(t - 1) & 1][i];
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int m = 0; m < MT; ++m)
#pragma unroll
                        for (int n = 0; n < NT; ++n)
                            acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(w4[n][j], x4[m][j], acc[m][n], 0, 0, 0);
            }
        }
    };
    // Step i: the products of chunk i, the fragments of chunk i + 1, the staging of chunk i + 2, the loads of chunk
    // i + 2 + PF.  Returns whether a value lies outside its window (then the sums are of no use): asked after the first
    // two chunks (flag[0]) and at the end (flag[1]: with a short K a fast wave is at the last steps, and sets its flag, while
    // a slow one has yet to read the first, and both must take the same way past the barriers).
    const int chunks = full + (tail > 0);
    auto flagged = [&](int i) { return __builtin_amdgcn_readfirstlane(flag[i]) != 0; };
    auto run = [&](auto stager, auto multiplier) {
        constexpr bool S = decltype(stager)::value, C = decltype(multiplier)::value;
        if constexpr (S) {
            begin();
            if (full > 0) {
#pragma unroll
                for (int p = 0; p < PF; ++p) load(raw[p]);
            }
            if (full == 0) load_tail(raw[0]);
            stage(raw[0], 0);
            if (full > 0) load(raw[0]);
        }
        if constexpr (C) clear();
        __syncthreads();
        if constexpr (C) fetch(0);
        if constexpr (S) {
            if (full == 1 && tail) load_tail(raw[1]);
            if (chunks > 1) stage(raw[1], 1);
            if (full > 0) load(raw[1]);
            if (bad) flag[0] = 1;
        }
        __syncthreads();
        if (__builtin_expect(flagged(0), 0)) return true;
        int i = 0;
        for (; i + PF + 2 <= full; i += PF) {
#pragma unroll
            for (int p = 0; p < PF; ++p) {
                uint32_t in = LIN_IN;
                if constexpr (C) fetch((p + 1) & 1);
                if constexpr (S) in = stage_put(raw[(p + 2) % PF], p & 1);
                if constexpr (C) {
                    compute(p & 1);
                    // (a last slot of only some waves is a branch, and its own scheduling region)
                    if constexpr (!S || T::WORK % T::STAGERS == 0)
                        lin_interleave<T::UNITS *(MT + NT), S ? T::SLOTS * 4 : 0, T::UNITS * 4 * MT * NT>();
                }
                if constexpr (S) {
                    stage_check(raw[(p + 2) % PF], in);
                    load(raw[(p + 2) % PF]);
                }
                __syncthreads();
            }
        }
        // at most PF + 2 chunks are left, the last of them perhaps partial
        if constexpr (S) {
#pragma unroll
            for (int r = 2; r < PF + 2; ++r)
                if (tail && i + r == full) load_tail(raw[r % PF]);
        }
#pragma unroll
        for (int p = 0; p < PF + 2; ++p)
            if (i + p < chunks) {
                if constexpr (C)
                    if (i + p + 1 < chunks) fetch((p + 1) & 1);
                if constexpr (S)
                    if (i + p + 2 < chunks) stage(raw[(p + 2) % PF], p & 1);
                if constexpr (C) compute(p & 1);
                if constexpr (S)
                    if (bad) flag[1] = 1;
                __syncthreads();
            }
        return flagged(1);
    };
    const bool multiplier = !PW || __builtin_amdgcn_readfirstlane(wave) < T::WAVES, stager = !PW || !multiplier;
    bool again;
    if constexpr (PW == 0) {
        again = run(std::true_type{}, std::true_type{});
    } else {
        if (multiplier)
            again = run(std::false_type{}, std::true_type{});
        else
            again = run(std::true_type{}, std::false_type{});
    }
    if (__builtin_expect(again, 0)) {  // a value outside its window: the tile again, chunks that hold one apart
        clear();
        if (chunks <= 2) {  // they are both in LDS still
            if (multiplier)
                for (int c = 0; c < chunks; ++c) products(lds[c], c < full ? T::UNITS : (tail + 15) / 16, true);
        } else {
            // Step c: the products of chunk c, the staging of chunk c + 1, the load of chunk c + 2; flag[c % 3]: chunk c
            // is to be kept apart.
            auto next = [&](int c) {
                if (c < full)
                    load(raw[0]);
                else if (c < chunks)
                    load_tail(raw[0]);
            };
            auto put = [&](int c) {
                bad = false;
                stage(raw[0], c & 1);
                if (bad) flag[c % 3] = 1;
                next(c + 1);
            };
            if (stager) {
                begin();
                next(0);
            }
            __syncthreads();
            if (tid < 3) flag[tid] = 0;
            __syncthreads();
            if (stager) put(0);
            __syncthreads();
            for (int c = 0; c < chunks; ++c) {
                if (stager && c + 1 < chunks) put(c + 1);
                if (multiplier) products(lds[c & 1], c < full ? T::UNITS : (tail + 15) / 16, flagged(c % 3));
                if (tid == 0) flag[(c + 2) % 3] = 0;
                __syncthreads();
            }
        }
    }
    if (!multiplier) return;
    // D of the instruction: its columns are rows of x, a lane's four values are consecutive columns of y
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int row = m0 + (wm * MT + m) * 16 + (lane & 15);
        if (row >= a.M) continue;
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            const int col = n0 + (wn * NT + n) * 16 + (lane >> 4) * 4;
            f32x4_t v = acc[m][n];
            if (a.vec_out && col < out.N) {
                const long o = (long)row * out.N + col;
                if (a.y_f32) {
                    *reinterpret_cast<f32x4_t *>(static_cast<float *>(out.y) + o) = v;
                    continue;
                }
                if (a.res) {
                    const u32x2_t r = *reinterpret_cast<const u32x2_t *>(a.res + o);
                    v = f32x4_t{bf16lo_to_f32(r[0]) + lin_round(v[0]), bf16hi_to_f32(r[0]) + lin_round(v[1]),
                                bf16lo_to_f32(r[1]) + lin_round(v[2]), bf16hi_to_f32(r[1]) + lin_round(v[3])};
                }
                *reinterpret_cast<u32x2_t *>(static_cast<bf16_t *>(out.y) + o) =
                    u32x2_t{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
            } else {
                for (int r = 0; r < 4; ++r)
                    if (col + r < out.N) lin_put(a, out, row, col + r, v[r]);
            }
        }
    }
}

template <int MT, int NT, int WM, int WN, int PW, int KC, int PF>
void linear_launch(LinArgs a) {
    using T = LinTile<MT, NT, WM, WN, PW, KC>;
    a.tiles_m = (a.M + T::TM - 1) / T::TM;
    linear_kernel<MT, NT, WM, WN, PW, KC, PF>
        <<<(unsigned)(a.tiles_m * lin_cols(a, T::TN)), T::THREADS, 0, g_llmgen_stream>>>(a);
}

// Up to eight rows and many columns (the LM head of a small decode step): bound by the read of w.  No LDS and no
// barriers: a wave owns 32 columns and all rows, a lane reads 16-byte pieces of its own row of w straight into
// registers (both halves of the wave hold the same 32 columns at alternate pieces), three stages of 64 k ahead, and
// v_mfma_f32_4x4x1_f32 takes them as they lie: BLGP picks the half that holds k, CBSZ / ABID the four-row block of x
// that does, so that nothing is moved between lanes.  8 x 151936 x 1024: 78 -> 63.5 us, one row 75 -> 57.5 us (5.4 TB/s);
// at 16 rows the tiles below are as fast (79 us).
constexpr int STREAM_ROWS = 8, STREAM_COLS = 128, STREAM_KC = 64, STREAM_PF = 3;

template <int... Ks>
__device__ __forceinline__ f32x4_t stream_products(f32x4_t acc, const float (&wf)[4][8], const float (&xf)[8],
                                                   std::integer_sequence<int, Ks...>) {
    // k of the stage, ascending: piece k / 8 of the row of w (wave half k / 8 % 2), block k / 8 of x, value k % 8
    ((acc = __builtin_amdgcn_mfma_f32_4x4x1f32(xf[Ks % 8], wf[Ks / 16][Ks % 8], acc, 3, Ks / 8, 1 + (Ks / 8 & 1))), ...);
    return acc;
}

// The same with the products rounded before they are added, four k at a time (see `products` above).
template <int... Qs>
__device__ __forceinline__ f32x4_t stream_apart(f32x4_t acc, const float (&wf)[4][8], const float (&xf)[8],
                                                std::integer_sequence<int, Qs...>) {
    auto four = [&](auto q) __attribute__((always_inline)) {
        constexpr int K0 = decltype(q)::value * 4;
        const f32x4_t p[4] = {stream_products(f32x4_t{}, wf, xf, std::integer_sequence<int, K0>{}),
                              stream_products(f32x4_t{}, wf, xf, std::integer_sequence<int, K0 + 1>{}),
                              stream_products(f32x4_t{}, wf, xf, std::integer_sequence<int, K0 + 2>{}),
                              stream_products(f32x4_t{}, wf, xf, std::integer_sequence<int, K0 + 3>{})};
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[r] = acc[r] + p[i][r];
    };
    (four(std::integral_constant<int, Qs>{}), ...);
    return acc;
}

__global__ void __launch_bounds__(256, 2) linear_stream_kernel(const LinArgs a) {
    constexpr int KC = STREAM_KC, PF = STREAM_PF;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int b0;
    const LinOut out = lin_out(a, blockIdx.x, STREAM_COLS, b0);
    const int n0 = b0 + wave * 32, K = a.K, full = K / KC, tail = K - full * KC;
    const int half = lane >> 5, xpiece = (lane >> 2) & 7;
    const bf16_t *wp = out.w + (long)min(n0 + (lane & 31), out.N - 1) * K + half * 8;
    const bf16_t *xp = a.x + (long)min(half * 4 + (lane & 3), a.M - 1) * K + xpiece * 8;
    u32x4_t wr[PF][4], xr[PF];
    auto load = [&](int set, int c) {  // past the last full stage: that stage again
        const long o = (long)min(c, full - 1) * KC;
#pragma unroll
        for (int i = 0; i < 4; ++i) wr[set][i] = ld16(wp + o + i * 16);
        xr[set] = ld16(xp + o);
    };
    auto load_tail = [&](int set) {
        const long o = (long)full * KC;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            wr[set][i] = u32x4_t{0u, 0u, 0u, 0u};
            if (i * 16 + half * 8 < tail) wr[set][i] = ld16(wp + o + i * 16);
        }
        xr[set] = u32x4_t{0u, 0u, 0u, 0u};
        if (xpiece * 8 < tail) xr[set] = ld16(xp + o);
    };
    f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
    auto use = [&](int set) {
        float wf[4][8], xf[8];
        uint32_t in = LIN_IN;
        bool bad = false;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            unpack_bf16x8(wr[set][i], wf[i]);
#pragma unroll
            for (int d = 0; d < 4; ++d) in &= wr[set][i][d] + LIN_W_BIAS;
        }
        unpack_bf16x8(xr[set], xf);
#pragma unroll
        for (int d = 0; d < 4; ++d) in &= xr[set][d] + LIN_X_BIAS;
        if (__builtin_expect(__ballot(in != LIN_IN) != 0, 0)) {
#pragma unroll
            for (int d = 0; d < 4; ++d) {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    bad |= !(lin_half_ok(wr[set][i][d] & 0xffffu, LIN_W_BIAS) &&
                             lin_half_ok(wr[set][i][d] >> 16, LIN_W_BIAS));
                bad |= !(lin_half_ok(xr[set][d] & 0xffffu, LIN_X_BIAS) && lin_half_ok(xr[set][d] >> 16, LIN_X_BIAS));
            }
        }
        if (__builtin_expect(__ballot(bad) != 0, 0)) {  // a value outside its window: products and sums apart
            acc = stream_apart(acc, wf, xf, std::make_integer_sequence<int, KC / 4>{});
            return;
        }
        // the VALU work stays in one piece: each change between it and the matrix cores costs 8 cycles
        __builtin_amdgcn_sched_barrier(0);
        acc = stream_products(acc, wf, xf, std::make_integer_sequence<int, KC>{});
        __builtin_amdgcn_sched_barrier(0);
    };
    int c = 0;
    if (full > 0) {
#pragma unroll
        for (int p = 0; p < PF; ++p) load(p, p);
        for (; c + PF <= full; c += PF)
#pragma unroll
            for (int p = 0; p < PF; ++p) {
                use(p);
                load(p, c + p + PF);
            }
    }
#pragma unroll
    for (int p = 0; p < PF; ++p) {
        if (c + p == full && tail) load_tail(p);
        if (c + p < full + (tail > 0)) use(p);
    }
    const int n = n0 + (lane & 31);
    if (n >= out.N) return;
#pragma unroll
    for (int r = 0; r < 4; ++r)
        if (half * 4 + r < a.M) lin_put(a, out, half * 4 + r, n, acc[r]);
}

// K of 8 and 16 (a low-rank update): nothing to pipeline, and the tiles would stage and multiply mostly zeros.  Bound by
// latencies and the store of y: a lane owns a column, its row of w and SHORT_ROWS rows of x are loaded at once, then
// multiplies and adds as the reference's.  1 x 1000 x 8: 1.8 us (tiles 4.0, the multiply-add kernel before them 3.0),
// 300 x 4096 x 16 3.9 (6.9, 6.0), 2051 x 4096 x 8 10.0 (17.0, 13.3); from K = 24 on the tiles are the faster.
constexpr int SHORT_ROWS = 8, SHORT_COLS = 256;
template <int K>
__global__ void __launch_bounds__(SHORT_COLS) linear_short_kernel(const LinArgs a) {
    int n0;
    const LinOut out = lin_out(a, blockIdx.x / a.tiles_m, SHORT_COLS, n0);
    const int n = n0 + threadIdx.x, m0 = blockIdx.x % a.tiles_m * SHORT_ROWS;
    if (n >= out.N) return;
    u32x4_t wr[K / 8], xr[SHORT_ROWS][K / 8];
#pragma unroll
    for (int i = 0; i < K / 8; ++i) {
        wr[i] = ld16(out.w + (long)n * K + i * 8);
#pragma unroll
        for (int r = 0; r < SHORT_ROWS; ++r) xr[r][i] = ld16(a.x + (long)min(m0 + r, a.M - 1) * K + i * 8);
    }
    float w[K], x[K];
#pragma unroll
    for (int i = 0; i < K / 8; ++i) unpack_bf16x8(wr[i], w + i * 8);
#pragma unroll
    for (int r = 0; r < SHORT_ROWS; ++r) {
        if (m0 + r >= a.M) return;
#pragma unroll
        for (int i = 0; i < K / 8; ++i) unpack_bf16x8(xr[r][i], x + i * 8);
        float sum = 0.f;
#pragma unroll
        for (int k = 0; k < K; ++k) sum = sum + x[k] * w[k];
        lin_put(a, out, m0 + r, n, sum);
    }
}
template <int K>
void linear_short_launch(LinArgs a) {
    a.tiles_m = (a.M + SHORT_ROWS - 1) / SHORT_ROWS;
    linear_short_kernel<K><<<(unsigned)(a.tiles_m * lin_cols(a, SHORT_COLS)), SHORT_COLS, 0, g_llmgen_stream>>>(a);
}

// Tiles of the throughput-bound sizes.  A launch takes about as long as the CU with the most tiles:
// ceil(tiles / CUs) * blocks of a tile / rate, where `rate` is the share of the matrix cores' peak that the tile
// reached on sizes it fits (launch time taken off): 0.68 for 32 x 32 (350 x 1024 x 3072: 34 us), 0.76 for 32 x 96 (2051 x
// 1024 x 1024: 43 to 48 us, by how warm the chip is), 0.80 for 64 x 64 (997 x 1024 x 3072: 57 to 66 us), 0.83 for 64 x 192
// (997 x 3072 x 1024: 54 to 63 us) and 0.85 for 128 x 128 (2048 x 6144 x 2048: 371 to 385 us = 134 to 139 TFLOP/s).  Larger
// tiles stage less per product but quantise coarser.  Of 92 sizes spread over M 17..3066, N 768..11480 and K 256..8192 the
// chosen tile is 1.4 % slower than the best of the five on average, 7.8 % at most.  All five stage in whole slots per wave
// (a slot that only some waves have splits the step's schedule: 96 x 32 with a 64-value chunk 10 % slower).
struct LinChoice {
    int tm, tn;
    float rate;
    void (*launch)(LinArgs);
};
const LinChoice LIN_CHOICES[] = {{32, 32, 0.68f, linear_launch<1, 1, 2, 2, 0, 64, 2>},
                                 {32, 96, 0.76f, linear_launch<1, 3, 2, 2, 0, 32, 2>},
                                 {64, 64, 0.80f, linear_launch<2, 2, 2, 2, 0, 32, 2>},
                                 {64, 192, 0.83f, linear_launch<2, 3, 2, 4, 0, 32, 2>},
                                 {128, 128, 0.85f, linear_launch<4, 2, 2, 4, 0, 32, 2>}};

void linear_dispatch(const LinArgs &a) {
    const long blocks = (long)((a.M + 15) / 16) * lin_cols(a, 16);
    const int cus = llmgen_num_cus();
    if (a.K == 8) return linear_short_launch<8>(a);
    if (a.K == 16) return linear_short_launch<16>(a);
    // At most one 16 x 16 block per CU: one block and three staging waves a workgroup (7.8 us at 1 x 1024 x 1024,
    // 17.3 us at 32 x 1024 x 3072; 32 x 32 tiles 9.5 and 26 us).
    if (blocks <= cus) return linear_launch<1, 1, 1, 1, 3, 128, 2>(a);
    // At most two: two blocks and two staging waves (11.2 us at 32 x 3072 x 1024, 12 us as single blocks; 32 x 32 tiles
    // take 10.8 us back to back, but 0.5 us more between other kernels: an MLP of 32 tokens 48.2 us, so 46.8 us).
    if (blocks <= 2 * cus) return linear_launch<1, 1, 1, 2, 2, 64, 4>(a);
    // Up to 16 rows and more blocks: bound by the read of w.  To 8 rows the stream above, to 16 small
    // workgroups, eight of them a CU (16 x 151936 x 1024: 79 us; 32 x 32 tiles, half of them empty, 107 us).
    if (a.M <= 16) {
        if (a.M > STREAM_ROWS) return linear_launch<1, 1, 1, 2, 0, 64, 2>(a);
        linear_stream_kernel<<<(unsigned)lin_cols(a, STREAM_COLS), 256, 0, g_llmgen_stream>>>(a);
        return;
    }
    const LinChoice *best = nullptr;
    float cost = 0.f;
    for (const LinChoice &c : LIN_CHOICES) {
        const long tiles = (long)((a.M + c.tm - 1) / c.tm) * lin_cols(a, c.tn);
        const float t = (float)((tiles + cus - 1) / cus) * (float)(c.tm * c.tn) / c.rate;
        if (!best || t < cost) best = &c, cost = t;
    }
    best->launch(a);
}

bool lin_reject(const char *what) {
    fprintf(stderr, "llmgen: %s: K must be a positive multiple of 8\n", what);
    return true;
}
// whether four outputs of a row can be moved as one word
bool lin_words(const void *p, int N, int bytes) { return N % 4 == 0 && (uintptr_t)p % (4 * bytes) == 0; }

}  // namespace

extern "C" {

void hip_linear(void *y, int y_f32, const uint16_t *x, const uint16_t *w, int M, int N, int K) {
    if (M <= 0 || N <= 0) return;
    if ((K <= 0 || K % 8 != 0) && lin_reject("hip_linear")) return;
    linear_dispatch(LinArgs{{{y, w, N}, {}, {}}, x, nullptr, M, K, y_f32, lin_words(y, N, y_f32 ? 4 : 2), 0});
}

void hip_linear_add(uint16_t *y, const uint16_t *res, const uint16_t *x, const uint16_t *w, int M, int N, int K) {
    if (M <= 0 || N <= 0) return;
    if ((K <= 0 || K % 8 != 0) && lin_reject("hip_linear_add")) return;
    const int vec = lin_words(y, N, 2) && lin_words(res, N, 2);
    linear_dispatch(LinArgs{{{y, w, N}, {}, {}}, x, res, M, K, 0, vec, 0});
}

void hip_linear3(uint16_t *y0, const uint16_t *w0, int N0, uint16_t *y1, const uint16_t *w1, int N1, uint16_t *y2,
                 const uint16_t *w2, int N2, const uint16_t *x, int M, int K) {
    N0 = std::max(N0, 0), N1 = std::max(N1, 0), N2 = std::max(N2, 0);
    if (M <= 0 || (N0 | N1 | N2) == 0) return;
    if ((K <= 0 || K % 8 != 0) && lin_reject("hip_linear3")) return;
    const int vec = lin_words(y0, N0, 2) && lin_words(y1, N1, 2) && lin_words(y2, N2, 2);
    linear_dispatch(LinArgs{{{y0, w0, N0}, {y1, w1, N1}, {y2, w2, N2}}, x, nullptr, M, K, 0, vec, 0});
}

}  // extern "C"
