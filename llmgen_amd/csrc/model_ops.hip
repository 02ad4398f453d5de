// model_ops.hip -- the non-attention ops of the Qwen3 forward except linear (embedding, RMSNorm, NEOX RoPE, SiLU,
// add, mul, gather_last, sampling), and the fused q/k norm + RoPE + KV write that replaces five of them before
// attention.
//
// Order and roundings come first, speed within them: every output is computed in the order the reference CPU
// backend uses (src/backend/cpu/*.zig), with one IEEE rounding per f32 multiply / add / divide / sqrt and one
// RNE rounding to bf16 per stored value, so a forward built from them matches the CPU backend bit for bit
// outside attention.  Contraction into FMAs is switched off for the whole file for that reason.
#include "hip_common.h"

#include <math.h>

#include <algorithm>

#pragma clang fp contract(off)

namespace {

__device__ __forceinline__ float bf2f(bf16_t b) { return __builtin_bit_cast(float, (uint32_t)b << 16); }
__device__ __forceinline__ bf16_t f2bf(float f) { return __builtin_bit_cast(bf16_t, (__bf16)f); }

// ---------------------------------------------------------------------------------------------- embedding
__global__ void embedding_kernel(bf16_t *out, const int *ids, const bf16_t *w, int T, int H) {
    const int chunks = H >> 3;
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long)T * chunks) return;
    const int t = (int)(i / chunks), c = (int)(i % chunks);
    const long row = ids[t];
    *reinterpret_cast<u32x4_t *>(out + (long)t * H + c * 8) = ld16(w + row * H + c * 8);
}

// ---------------------------------------------------------------------------------------------- RMSNorm
// The sum of squares is one f32 chain per row in index order (the reference's order), D dependent adds of about 4.5
// cycles each, and nothing can shorten it: at D = 1024 it is 2 us of the launch.  Everything else is kept off it: all
// lanes square the row's values (exactly what the reference adds, one rounded multiply each) and leave them in LDS,
// and the chain is a run of adds fed by 16-byte LDS reads.  A wave owns R rows, 64 / R lanes each; every lane runs its
// row's chain (the reads of a row's lanes are one broadcast address), so the sum needs no exchange afterwards.
// Measured, D = 1024: 32 rows 14.7 -> 5.2 us, 2051 rows 36 -> 7.4 us (before: one lane of a wave formed each square and
// sum).
constexpr int NORM_MAX_D = 8192;
// The output and the gains may lie at any value's address (x is 16-byte aligned), which these types tell the compiler; it
// moves them as whole vectors all the same.
typedef u32x4_t u32x4_any_t __attribute__((aligned(2)));
typedef f32x4_t f32x4_any_t __attribute__((aligned(4)));
template <int R>
__global__ void __launch_bounds__(64) rmsnorm_kernel(bf16_t *out, const bf16_t *x, const float *w, long rows, int D,
                                                      float eps) {
    extern __shared__ __attribute__((aligned(16))) float sq[];
    constexpr int L = 64 / R;  // lanes per row
    const int sub = threadIdx.x % L, chunks = D >> 3;
    const long r = min((long)blockIdx.x * R + threadIdx.x / L, rows - 1);  // surplus lanes repeat the last row
    const bool valid = (long)blockIdx.x * R + threadIdx.x / L < rows;
    const bf16_t *xr = x + r * D;
    float *sr = sq + threadIdx.x / L * (D + 4);  // rows start in different banks
    // Few rows (one a wave) are bound by latencies: up to KEEP pieces of a row stay in registers, with their gains loaded
    // before the chain, and the chain reads ahead (32 rows of 1024: 5.7 us without, 5.2 us with).  Many rows need the
    // waves instead of the registers (8195 x 128 in this form 7.0 us, not 5.2).
    constexpr int KEEP = R == 1 ? 4 : 1, AHEAD = R == 1 ? 2 : 1;
    const bool kept = R == 1 && chunks <= KEEP * L;
    u32x4_t raw[KEEP];
    f32x4_t gain[KEEP][2];
    auto square = [&](u32x4_t v, int c) {
        float f[8];
        unpack_bf16x8(v, f);
#pragma unroll
        for (int h = 0; h < 2; ++h)
            *reinterpret_cast<f32x4_t *>(sr + c * 8 + h * 4) =
                f32x4_t{f[4 * h] * f[4 * h], f[4 * h + 1] * f[4 * h + 1], f[4 * h + 2] * f[4 * h + 2],
                        f[4 * h + 3] * f[4 * h + 3]};
    };
    if (kept) {
#pragma unroll
        for (int i = 0; i < KEEP; ++i)
            if (sub + i * L < chunks) raw[i] = ld16(xr + (sub + i * L) * 8);
#pragma unroll
        for (int i = 0; i < KEEP; ++i)
            if (sub + i * L < chunks) {
                gain[i][0] = *reinterpret_cast<const f32x4_any_t *>(w + (sub + i * L) * 8);
                gain[i][1] = *reinterpret_cast<const f32x4_any_t *>(w + (sub + i * L) * 8 + 4);
            }
#pragma unroll
        for (int i = 0; i < KEEP; ++i)
            if (sub + i * L < chunks) square(raw[i], sub + i * L);
    } else {
#pragma unroll 4
        for (int c = sub; c < chunks; c += L) square(ld16(xr + c * 8), c);
    }
    __syncthreads();
    // the chain, 64 terms at a time
    float ss = 0.0f;
    const int blocks = D / 64;
    f32x4_t v[AHEAD][16];
    auto fetch = [&](int set, int blk) {
#pragma unroll
        for (int i = 0; i < 16; ++i) v[set][i] = *reinterpret_cast<const f32x4_t *>(sr + blk * 64 + i * 4);
    };
    auto add = [&](int set) {
#pragma unroll
        for (int i = 0; i < 16; ++i) ss = ss + v[set][i][0] + v[set][i][1] + v[set][i][2] + v[set][i][3];
    };
    if constexpr (AHEAD == 2) {
        if (blocks > 0) fetch(0, 0);
        for (int b = 0; b + 1 < blocks; b += 2) {
            fetch(1, b + 1);
            add(0);
            fetch(0, min(b + 2, blocks - 1));
            add(1);
        }
        if (blocks & 1) add(0);
    } else {
        for (int b = 0; b < blocks; ++b) {
            fetch(0, b);
            add(0);
        }
    }
    for (int d = blocks * 64; d < D; d += 8) {
        const f32x4_t u = *reinterpret_cast<const f32x4_t *>(sr + d), t = *reinterpret_cast<const f32x4_t *>(sr + d + 4);
        ss = ss + u[0] + u[1] + u[2] + u[3] + t[0] + t[1] + t[2] + t[3];
    }
    const float scale = 1.0f / sqrtf(ss / (float)D + eps);
    if (!valid) return;
    auto finish = [&](u32x4_t x8, f32x4_t g0, f32x4_t g1, int c) {
        float f[8];
        unpack_bf16x8(x8, f);
        const float g[8] = {g0[0], g0[1], g0[2], g0[3], g1[0], g1[1], g1[2], g1[3]};
        u32x4_t o;
#pragma unroll
        for (int h = 0; h < 4; ++h)
            o[h] = pack_bf16x2(bf2f(f2bf(f[2 * h] * scale)) * g[2 * h], bf2f(f2bf(f[2 * h + 1] * scale)) * g[2 * h + 1]);
        *reinterpret_cast<u32x4_any_t *>(out + r * D + c * 8) = o;
    };
    if (kept) {
#pragma unroll
        for (int i = 0; i < KEEP; ++i)
            if (sub + i * L < chunks) finish(raw[i], gain[i][0], gain[i][1], sub + i * L);
    } else {
#pragma unroll 4
        for (int c = sub; c < chunks; c += L)
            finish(ld16(xr + c * 8), *reinterpret_cast<const f32x4_any_t *>(w + c * 8),
                   *reinterpret_cast<const f32x4_any_t *>(w + c * 8 + 4), c);
    }
}

// ---------------------------------------------------------------------------------------------- RoPE
__global__ void rope_kernel(bf16_t *out, const bf16_t *x, const float *cos_t, const float *sin_t, const int *pos,
                            int T, int n_head, int hd) {
    const int half = hd >> 1;
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long)T * n_head * half) return;
    const int d = (int)(i % half);
    const long th = i / half;  // t * n_head + h
    const int t = (int)(th / n_head);
    const long b = th * hd;
    const long p = pos[t];
    const float c = cos_t[p * hd + d], s = sin_t[p * hd + d];
    const float x0 = bf2f(x[b + d]), x1 = bf2f(x[b + d + half]);
    out[b + d] = f2bf(x0 * c - x1 * s);
    out[b + d + half] = f2bf(x1 * c + x0 * s);
}

// ---------------------------------------------------------------------------------------------- elementwise
// Long streams of bf16: eight values per lane and 16-byte accesses where every pointer allows them, the last n % 8 one by
// one; else a value per lane in a kernel of its own, which has none of the split's arithmetic (2^24 values, add: 25.5 us, 26.8
// as the vector kernel's tail).
struct SiluOp {
    __device__ __forceinline__ float operator()(float v, float) const { return v / (1.0f + expf(-v)); }
};
struct AddOp {
    __device__ __forceinline__ float operator()(float a, float b) const { return a + b; }
};
struct SiluMulOp {  // SiLU's result is rounded to bf16 before the product, as when it is stored in between
    __device__ __forceinline__ float operator()(float v, float u) const { return bf2f(f2bf(SiluOp{}(v, 0.f))) * u; }
};
struct MulOp {
    __device__ __forceinline__ float operator()(float a, float b) const { return a * b; }
};

template <class Op>
__global__ void __launch_bounds__(256) elementwise_kernel(bf16_t *out, const bf16_t *a, const bf16_t *b, size_t vecs,
                                                          size_t n, Op op) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < vecs) {
        float x[8], y[8];
        unpack_bf16x8(ld16(a + i * 8), x);
        unpack_bf16x8(ld16(b + i * 8), y);
        u32x4_t o;
#pragma unroll
        for (int h = 0; h < 4; ++h) o[h] = pack_bf16x2(op(x[2 * h], y[2 * h]), op(x[2 * h + 1], y[2 * h + 1]));
        *reinterpret_cast<u32x4_t *>(out + i * 8) = o;
    } else {
        const size_t e = vecs * 8 + (i - vecs);
        if (e < n) out[e] = f2bf(op(bf2f(a[e]), bf2f(b[e])));
    }
}

template <class Op>
__global__ void __launch_bounds__(256) elementwise_single_kernel(bf16_t *out, const bf16_t *a, const bf16_t *b, size_t n,
                                                                 Op op) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = f2bf(op(bf2f(a[i]), bf2f(b[i])));
}

__global__ void gather_rows_kernel(bf16_t *out, const bf16_t *x, const int *idx, int S, int H) {
    const int chunks = H >> 3;
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long)S * chunks) return;
    const int s = (int)(i / chunks), c = (int)(i % chunks);
    *reinterpret_cast<u32x4_t *>(out + (long)s * H + c * 8) = ld16(x + (long)idx[s] * H + c * 8);
}

// ---------------------------------------------------------------------------------------------- sampling
// Greedy / Gumbel-max token choice (cpu/sample.zig:17-45 semantics).
// Every candidate (value v, index i) becomes one 64-bit key: the high word is v's bits mapped so that unsigned
// order is float order, the low word is ~i.  The largest key is then the largest value and, among equal values,
// the smallest index -- exactly what the reference's strictly-greater scan keeps -- so the reduction is a plain
// unsigned max with no tie logic.  NaN and -inf never win that scan (no comparison with them is true), so they
// are not candidates; key 0 means "no candidate" and yields index 0, the scan's starting index.
// What bit parity with the CPU backend fixes is kept as it is: the splitmix64 stream per (seed, row, index), the
// uniform from its top 24 bits and the Gumbel value v / t - log(-log u), each f32 operation rounded once.
//
// A workgroup scans a row, or a slice of a long one: drawing the noise of a 151936-wide row (two logarithms and two
// 64-bit products per value) takes one CU 70 us.  Slices of one row meet in out[row] itself: the key of the index that it
// holds can be formed again from the logits, so a workgroup that found a better candidate replaces it with a
// compare-and-swap (retried while others do the same; every retry means the row got better).  An index left there by an
// earlier call is one more candidate of this row, anything else is no candidate, so nothing has to be cleared first.  No
// scratch, and the result does not depend on the order: the largest key wins.
// Measured, rows of 151936, one workgroup a row -> slices: one row greedy 16.2 -> 4.2 us, with noise 69 -> 5.2 us; 32 rows
// 17.0 -> 4.4 and 70 -> 12.3 us, a third of them with noise 70 -> 9.2 us.
__device__ __forceinline__ uint64_t mix64(uint64_t x) {  // SplitMix64 finaliser, as cpu/sample.zig:7-12
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}

__device__ __forceinline__ uint64_t cand_key(float v, int i) {
    if (!(v > -INFINITY)) return 0;  // NaN, -inf
    if (v == 0.f) v = 0.f;           // -0 == +0 for the scan: equal keys, so the smaller index wins
    const uint32_t u = __builtin_bit_cast(uint32_t, v);
    const uint32_t ord = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
    return ((uint64_t)ord << 32) | (uint32_t)~(uint32_t)i;
}

__device__ __forceinline__ uint64_t shfl_xor64(uint64_t x, int m) {
    const int lane = __lane_id();
    const int lo = __builtin_amdgcn_ds_bpermute((lane ^ m) << 2, (int)(uint32_t)x);
    const int hi = __builtin_amdgcn_ds_bpermute((lane ^ m) << 2, (int)(uint32_t)(x >> 32));
    return ((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo;
}

// The key of candidate i with logit x: greedy, or the Gumbel value under the row's noise stream.
template <bool GUMBEL>
__device__ __forceinline__ uint64_t key_of(float x, int i, float temp, uint64_t rs) {
    if (GUMBEL) {
        const uint64_t r = mix64(rs + (uint32_t)i);
        const float u = ((float)(r >> 40) + 0.5f) * (1.0f / 16777216.0f);
        x = x / temp - logf(-logf(u));
    }
    return cand_key(x, i);
}

// The best key of one slice of a row for this lane.  The row is read in 16-byte vectors from its first aligned value on
// (greedy four per lane in flight; with noise the arithmetic hides the read); the first slice also takes the values before
// that, the last one those left at the end.
template <bool GUMBEL, int THREADS>
__device__ __forceinline__ uint64_t scan_slice(const bf16_t *row, int V, int slice, int slices, float temp,
                                               uint64_t rs) {
    constexpr int U = GUMBEL ? 1 : 4;
    const int head = min(V, (int)((16 - ((uintptr_t)row & 15)) & 15) / 2), vecs = (V - head) / 8;
    const int per = slices == 1 ? vecs : (vecs + slices - 1) / slices;
    const int v0 = slice * per, v1 = min(vecs, v0 + per);
    uint64_t best = 0;
    auto take = [&](float x, int i) {
        const uint64_t k = key_of<GUMBEL>(x, i, temp, rs);
        best = k > best ? k : best;
    };
    float top = -INFINITY;  // greedy: the value and index of this lane's best candidate
    int at = 0;
    for (int v = v0 + threadIdx.x; v < v1; v += THREADS * U) {
        u32x4_t raw[U];
#pragma unroll
        for (int u = 0; u < U; ++u) raw[u] = ld16(row + head + (long)min(v + u * THREADS, v1 - 1) * 8);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int vi = v + u * THREADS;
            if (vi >= v1) break;
            float f[8];
            unpack_bf16x8(raw[u], f);
            if (GUMBEL) {
#pragma unroll
                for (int e = 0; e < 8; ++e) take(f[e], head + vi * 8 + e);
                continue;
            }
            // a lane scans upwards, so only a larger value can displace its best (and NaN is never larger)
            float m = f[0];
#pragma unroll
            for (int e = 1; e < 8; ++e) m = fmaxf(m, f[e]);
            if (m > top) {
                top = m;
#pragma unroll
                for (int e = 7; e >= 0; --e) at = f[e] == m ? head + vi * 8 + e : at;
            }
        }
    }
    if (!GUMBEL) best = cand_key(top, at);
    const int rest = head + vecs * 8 + threadIdx.x;
    if (slice == 0 && (int)threadIdx.x < head) take(bf2f(row[threadIdx.x]), threadIdx.x);
    if (slice == slices - 1 && rest < V) take(bf2f(row[rest]), rest);
    return best;
}

// CUT: S rows cut into noise_slices workgroups, of which greedy rows use the first greedy_slices; else a workgroup a row.
// All first slices come first, then all second ones, each time one row further on: workgroups go to the XCDs in turn, and
// so the slices in use, and those of one row, lie on all of them (slice by slice of a row, two slices of which greedy rows
// use one left every other XCD idle: 256 greedy rows of 65536 9.4 us, so 5.8).
template <int THREADS, bool CUT>
__global__ void __launch_bounds__(THREADS) sample_rows_kernel(int *out, const bf16_t *logits, const float *temps,
                                                               const uint64_t *seed, int V, int noise_slices,
                                                               int greedy_slices, int S) {
    const int slice = CUT ? blockIdx.x / S : 0, s = CUT ? (blockIdx.x + slice) % S : blockIdx.x;
    const float temp = temps[s];
    const bool gumbel = temp > 0.0f;
    const int slices = !CUT ? 1 : gumbel ? noise_slices : greedy_slices;
    if (slice >= slices) return;
    const bf16_t *row = logits + (long)s * V;
    const uint64_t rs = gumbel ? mix64(*seed ^ ((uint64_t)s << 40)) : 0;
    uint64_t best = gumbel ? scan_slice<true, THREADS>(row, V, slice, slices, temp, rs)
                           : scan_slice<false, THREADS>(row, V, slice, slices, temp, 0);
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) {
        const uint64_t o = shfl_xor64(best, m);
        best = o > best ? o : best;
    }
    __shared__ uint64_t wave_best[THREADS / 64];
    if ((threadIdx.x & 63) == 0) wave_best[threadIdx.x >> 6] = best;
    __syncthreads();
    if (threadIdx.x != 0) return;
    for (int w = 1; w < THREADS / 64; ++w) best = wave_best[w] > best ? wave_best[w] : best;
    const int mine = best == 0 ? 0 : (int)~(uint32_t)best;  // 0: the scan's starting index, if no value is a candidate
    if (slices == 1) {
        out[s] = mine;
        return;
    }
    int cur = __hip_atomic_load(out + s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (;;) {
        uint64_t k = 0;
        if ((unsigned)cur < (unsigned)V) {
            const float x = bf2f(row[cur]);
            k = gumbel ? key_of<true>(x, cur, temp, rs) : key_of<false>(x, cur, temp, 0);
        }
        if (best < k || (best == k && cur == mine) ||
            __hip_atomic_compare_exchange_strong(out + s, &cur, mine, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT))
            return;
    }
}

bool reject(const char *what) {
    fprintf(stderr, "llmgen: %s\n", what);
    return true;
}

unsigned blocks_for(size_t n, unsigned per) { return (unsigned)((n + per - 1) / per); }

// Whether p is memory of the current device, where a compare-and-swap needs nothing from the bus (host memory: PCIe
// atomics, which not every machine routes).  A query only, allowed while a stream is captured.
bool on_this_device(const void *p) {
    const hipError_t before = hipPeekAtLastError();
    int dev = 0;
    hipPointerAttribute_t at{};
    if (hipGetDevice(&dev) == hipSuccess && hipPointerGetAttributes(&at, p) == hipSuccess)
        return at.type == hipMemoryTypeDevice && at.device == dev;
    (void)hipGetLastError();  // this query's own error; an earlier one stays known
    if (before != hipSuccess) llmgen_record_error(before);
    return false;
}

template <class Op>
void elementwise(bf16_t *out, const bf16_t *a, const bf16_t *b, size_t n, Op op) {
    if (n == 0) return;
    // Short streams are bound by the latency of one lane's work, and a value per lane is the least of it (SiLU of 16385 values
    // 1.91 us, 1.97 in vectors, of 2^17 1.92 and 2.03, add 1.95 either way; of 2^20 2.77 and 2.61, add 2.69 and 2.17).
    if (n <= 131072 || (((uintptr_t)out | (uintptr_t)a | (uintptr_t)b) & 15)) {
        elementwise_single_kernel<<<blocks_for(n, 256), 256, 0, g_llmgen_stream>>>(out, a, b, n, op);
        return;
    }
    const size_t vecs = n / 8;
    elementwise_kernel<<<blocks_for(vecs + (n - vecs * 8), 256), 256, 0, g_llmgen_stream>>>(out, a, b, vecs, n, op);
}

}  // namespace

extern "C" {

void hip_embedding(uint16_t *out, const int32_t *ids, const uint16_t *weight, int T, int H) {
    if (T <= 0) return;
    if (H <= 0 || H % 8 != 0) {
        reject("hip_embedding: H must be a positive multiple of 8");
        return;
    }
    const size_t n = (size_t)T * (H / 8);
    embedding_kernel<<<blocks_for(n, 256), 256, 0, g_llmgen_stream>>>(out, ids, weight, T, H);
}

void hip_rmsnorm(uint16_t *out, const uint16_t *x, const float *w, long rows, int D, float eps) {
    if (rows <= 0) return;
    if (D <= 0 || D % 8 != 0 || D > NORM_MAX_D) {
        reject("hip_rmsnorm: D must be a positive multiple of 8, at most 8192");
        return;
    }
    // Rows per wave: as many as leave a wave for every SIMD (a SIMD runs two chains no faster than one after the
    // other) while the rows of 7 or 8 waves still fit a CU's LDS (8193 x 1024: 4 rows a wave 13.2 us, 8 rows 20.0 us; 3000 x
    // 2048: 2 rows 13.6 us, 1 row 20.4 us; 8193 x 2560: 47 and 57 us; 8193 x 4096, where 2 rows a wave leave room for 4
    // waves: 100 and 88 us).
    const long simds = 4L * llmgen_num_cus();
    auto launch = [&](auto kernel, int R) {
        kernel<<<(unsigned)((rows + R - 1) / R), 64, (size_t)R * (D + 4) * 4, g_llmgen_stream>>>(out, x, w, rows, D, eps);
    };
    if (rows >= 8 * simds && D <= 512)
        launch(rmsnorm_kernel<8>, 8);
    else if (rows >= 4 * simds && D <= 1024)
        launch(rmsnorm_kernel<4>, 4);
    else if (rows >= 2 * simds && D <= 2560)
        launch(rmsnorm_kernel<2>, 2);
    else
        launch(rmsnorm_kernel<1>, 1);
}

void hip_rope(uint16_t *out, const uint16_t *x, const float *cos_tab, const float *sin_tab, const int32_t *positions,
              int T, int n_head, int hd) {
    if (T <= 0 || n_head <= 0) return;
    if (hd <= 0 || hd % 2 != 0) {
        reject("hip_rope: hd must be positive and even");
        return;
    }
    const size_t n = (size_t)T * n_head * (hd / 2);
    rope_kernel<<<blocks_for(n, 256), 256, 0, g_llmgen_stream>>>(out, x, cos_tab, sin_tab, positions, T, n_head, hd);
}

void hip_silu(uint16_t *out, const uint16_t *x, size_t n) { elementwise(out, x, x, n, SiluOp{}); }

void hip_add(uint16_t *out, const uint16_t *a, const uint16_t *b, size_t n) { elementwise(out, a, b, n, AddOp{}); }

void hip_mul(uint16_t *out, const uint16_t *a, const uint16_t *b, size_t n) { elementwise(out, a, b, n, MulOp{}); }

void hip_silu_mul(uint16_t *out, const uint16_t *gate, const uint16_t *up, size_t n) {
    elementwise(out, gate, up, n, SiluMulOp{});
}

void hip_gather_rows(uint16_t *out, const uint16_t *x, const int32_t *idx, int S, int H) {
    if (S <= 0) return;
    if (H <= 0 || H % 8 != 0) {
        reject("hip_gather_rows: H must be a positive multiple of 8");
        return;
    }
    const size_t n = (size_t)S * (H / 8);
    gather_rows_kernel<<<blocks_for(n, 256), 256, 0, g_llmgen_stream>>>(out, x, idx, S, H);
}

// No scratch is needed (the argument stays for the reference's argument list, sample.zig:4-14, and may be null).
size_t hip_sample_scratch_bytes(int max_S) {
    (void)max_S;
    return 0;
}

void hip_sample(int32_t *out_ids, const uint16_t *logits, const float *temps, const uint64_t *seed, int S, int V,
                void *scratch) {
    (void)scratch;
    if (S <= 0) return;
    if (V <= 0) {
        reject("hip_sample: V must be positive");
        return;
    }
    // Slices of rows with noise: 2048 values in one at least, four vectors a lane of 512, and 8 to 16 slices, few rows 32.
    // The host does not know which rows have noise: a third of them fills the chip evenly only in small slices (200 rows
    // of 151936, a third with noise: 31 us in 16 slices, 67 in two of 1024 lanes, 72 whole; all of them: 55, 68 and 73 us).  Whole rows
    // where many rows fill it anyway, and where slices would be short (256 rows of 12000 with noise: 8.0 us whole, 8.9 in
    // four; 256 rows of 16384: 10.1 and 10.5 us, but a third of them 9.8 and 7.1).
    // Greedy rows are a plain read, and their slices queue at the compare-and-swaps, since the words of all rows are
    // neighbours: one, or a few of 16384 values at least (32 rows of 151936: 9.9 us in one, 6.3 in two, 4.6 in four; 200 rows
    // of 65536: 6.1, 5.9, 6.0).
    const int cus = llmgen_num_cus();
    int n = std::min(V / 2048, S <= cus / 8 ? 32 : std::max(8, std::min(16, V / 4096)));
    n = V <= 8192 || (V < 16384 && S > cus / 2) ? 1 : std::max(1, std::min(n, (V < 24576 ? 4 : 16) * cus / S));
    if (n > 1 && !on_this_device(out_ids)) n = 1;  // one workgroup a row, which writes its id with a plain store
    const int g = std::min(n, V < 65536 ? 1 : S <= cus * 5 / 8 ? 4 : 2);
    auto launch = [&](auto kernel, int grid, int threads) {
        kernel<<<grid, threads, 0, g_llmgen_stream>>>(out_ids, logits, temps, seed, V, n, g, S);
    };
    // Whole rows: lanes for a vector each; where a CU holds several rows, at most 512 of them (700 rows of 12000, a third
    // with noise: 9.3 us, with 1024 lanes 14.0, all with noise 18.2 and 17.6).
    if (n > 1)
        launch(sample_rows_kernel<512, true>, n * S, 512);
    else if (V <= 2048)
        launch(sample_rows_kernel<256, false>, S, 256);
    else if (V <= 4096 || S > cus)
        launch(sample_rows_kernel<512, false>, S, 512);
    else
        launch(sample_rows_kernel<1024, false>, S, 1024);
}

}  // extern "C"

// ------------------------------------------------------------------------------------------------------------
// Fused per-head q/k RMSNorm + NEOX RoPE + paged KV write (one launch for what the unfused graph does in five:
// rmsnorm(q), rmsnorm(k), rope(q), rope(k), store_kv).  Eight lanes own one 128-wide head row, 16 elements each
// (two 16-byte loads, coalesced), and the row stays in registers from load to store.  Every value is rounded
// exactly where the unfused ops round it, and the sum of squares is formed in index order: lane j of the row
// continues the running sum it receives from lane j-1 (a DPP shift per step, eight steps), so the outputs are
// bit-identical to the unfused sequence.  RoPE partners (i, i + 64) sit in lanes j and j ^ 4.  Rows
// [0, T*nq) are q rows (written to q_out, which may alias q); rows [T*nq, T*(nq+nkv)) are k rows, written into
// the paged cache together with the v row of the same (token, KV head).  Slot < 0 skips the cache write.
namespace {
constexpr int QK_HD = 128;
constexpr int QK_LPR = 8;  // lanes per row

__global__ void __launch_bounds__(256) qk_norm_rope_store_kernel(
    bf16_t *q_out, bf16_t *k_cache, bf16_t *v_cache, const bf16_t *q, const bf16_t *k, const bf16_t *v,
    const float *q_w, const float *k_w, float eps, const float *cos_t, const float *sin_t, const int *pos,
    const int *slots, int T, int nq, int nkv, int block_size) {
    const long gt = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int sub = threadIdx.x & (QK_LPR - 1);
    const long rows_q = (long)T * nq, rows = rows_q + (long)T * nkv;
    const bool valid = gt / QK_LPR < rows;
    const long r = valid ? gt / QK_LPR : rows - 1;  // out-of-range lanes still take part in the exchanges
    const bool is_q = r < rows_q;
    const long rk = r - rows_q;
    const int t = is_q ? (int)(r / nq) : (int)(rk / nkv);
    const int h = is_q ? 0 : (int)(rk % nkv);
    const bf16_t *src = (is_q ? q + r * QK_HD : k + rk * QK_HD) + sub * 16;
    const float *w = (is_q ? q_w : k_w) + sub * 16;

    u32x4_t xv[2] = {ld16(src), ld16(src + 8)};
    float x[16];
    unpack_bf16x8(xv[0], x);
    unpack_bf16x8(xv[1], x + 8);
    // running sum of squares in index order across the row's eight lanes
    float in = 0.0f, cand = 0.0f;
#pragma unroll
    for (int step = 0; step < QK_LPR; ++step) {
        cand = in;
#pragma unroll
        for (int e = 0; e < 16; ++e) cand += x[e] * x[e];
        // row_shr:1 -- lane j receives lane j-1's running sum (lane 0 of each row starts from 0)
        const float prev = __builtin_bit_cast(
            float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, cand), 0x111, 0xF, 0xF, false));
        in = sub ? prev : 0.0f;
    }
    // the last lane of the row holds the complete sum
    const int last_lane = (__lane_id() & ~(QK_LPR - 1)) | (QK_LPR - 1);
    const float ss = __builtin_bit_cast(
        float, __builtin_amdgcn_ds_bpermute(last_lane << 2, __builtin_bit_cast(int, cand)));
    const float scale = 1.0f / sqrtf(ss / (float)QK_HD + eps);
    float n[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) n[e] = bf2f(f2bf(bf2f(f2bf(x[e] * scale)) * w[e]));
    // RoPE: lanes 0-3 hold dims i < 64 (x0), lanes 4-7 their partners i + 64 (x1); cos/sin rows repeat per half
    float other[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) other[e] = lane_xor(n[e], 4);
    const int dim0 = sub * 16;
    const float *cr = cos_t + (long)pos[t] * QK_HD + dim0;
    const float *sr = sin_t + (long)pos[t] * QK_HD + dim0;
    const bool low = sub < 4;
    u32x4_t ov[2];
#pragma unroll
    for (int e = 0; e < 16; e += 2) {
        float o2[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const float c = cr[e + u], s = sr[e + u];
            o2[u] = low ? n[e + u] * c - other[e + u] * s : n[e + u] * c + other[e + u] * s;
        }
        ov[e >> 3][(e & 7) >> 1] = pack_bf16x2(o2[0], o2[1]);
    }
    if (!valid) return;
    if (is_q) {
        bf16_t *dst = q_out + r * QK_HD + dim0;
        *reinterpret_cast<u32x4_t *>(dst) = ov[0];
        *reinterpret_cast<u32x4_t *>(dst + 8) = ov[1];
        return;
    }
    const int slot = slots[t];
    if (slot < 0) return;
    const long off = (((long)(slot / block_size) * nkv + h) * block_size + slot % block_size) * QK_HD + dim0;
    const bf16_t *vsrc = v + rk * QK_HD + dim0;
    const u32x4_t v0 = ld16(vsrc), v1 = ld16(vsrc + 8);
    *reinterpret_cast<u32x4_t *>(k_cache + off) = ov[0];
    *reinterpret_cast<u32x4_t *>(k_cache + off + 8) = ov[1];
    *reinterpret_cast<u32x4_t *>(v_cache + off) = v0;
    *reinterpret_cast<u32x4_t *>(v_cache + off + 8) = v1;
}
}  // namespace

extern "C" void hip_qk_norm_rope_store_kv(uint16_t *q_out, uint16_t *k_cache, uint16_t *v_cache, const uint16_t *q,
                                          const uint16_t *k, const uint16_t *v, const float *q_norm_w,
                                          const float *k_norm_w, float eps, const float *cos_tab,
                                          const float *sin_tab, const int32_t *positions,
                                          const int32_t *slot_mapping, int T, int nq, int nkv, int hd,
                                          int block_size) {
    if (T <= 0) return;
    if (hd != QK_HD || nq <= 0 || nkv <= 0 || block_size <= 0) {
        reject("hip_qk_norm_rope_store_kv: needs hd == 128 and positive nq, nkv, block_size");
        return;
    }
    const size_t threads = (size_t)T * (nq + nkv) * QK_LPR;
    qk_norm_rope_store_kernel<<<blocks_for(threads, 256), 256, 0, g_llmgen_stream>>>(
        q_out, k_cache, v_cache, q, k, v, q_norm_w, k_norm_w, eps, cos_tab, sin_tab, positions, slot_mapping, T, nq,
        nkv, block_size);
}
