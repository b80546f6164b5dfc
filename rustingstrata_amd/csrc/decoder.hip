// The decoder stack around the quantized matmuls: per-head RMS norm with NEOX rope and the f16 KV-cache store
// (Backend::rms_norm_rope_kv / rms_norm_rope_qk / rope_pairs / kv_store, src/backend.rs:250-277,380), argmax over
// logit rows (Backend::argmax_rows, :246), x += y and SwiGLU (:282-284), float-weight matmuls (the router's F32
// weights through gemv / gemm_dense), embedding rows (Model::embed, src/model.rs:334-339, on the device) and seeded
// synthetic GGUF blocks.
#include <cmath>

#include "decoder.h"
#include "formats.h"
#include "xlane.h"

namespace strata {

__device__ __forceinline__ uint16_t f32_to_f16_bits(float v) {
    _Float16 h = (_Float16)v;  // round to nearest even, as __float2half_rn
    uint16_t b;
    __builtin_memcpy(&b, &h, 2);
    return b;
}


// CUs of the device (256 where that cannot be told).
static int cu_count() {
    static const int ncu = [] {
        int dev = 0, v = 0;
        return hipGetDevice(&dev) == hipSuccess && hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0 ? v : 256;
    }();
    return ncu;
}

// ---- rms_norm + rope (+ KV store) ----
// One wave per head, n <= 512, the head staged in LDS. The sum of squares runs in index order on one lane (n adds per
// head, a small part of the launch), and out = x * (1 / sqrt(ss / n + eps)) * w in the reference's operation order,
// so the normed head has the CPU's bits (src/ops.rs:3-7; kernel
// src/cuda/kernels.cu:2196-2227). The rope turns pair (i, i + n_rot / 2) by theta = pos * base^(-2 i / n_rot), theta
// in f64 and its sine and cosine rounded to f32 as ops::rope_neox does (src/ops.rs:36-45).
constexpr int NR_WAVES = 4;

// Head gb (query heads first, then key heads) of a launch: its source row, norm weights, output row and whether it
// stores to the KV cache.
struct NrHead {
    const float* xr;
    const float* w;
    float* o;
    const float* vr;  // value row (key heads of a storing launch), else null
    int b, per;
};
__device__ __forceinline__ NrHead nr_head(const NormRope& a, int gb) {
    NrHead h;
    if (gb < a.qrows) {
        h.b = gb; h.per = a.qper;
        h.xr = a.qx + (uint64_t)(gb / a.qper) * a.q_tstride + (uint64_t)(gb % a.qper) * a.q_stride;
        h.w = a.qw; h.o = a.qo + (uint64_t)gb * a.n; h.vr = nullptr;
    } else {
        const int b = gb - a.qrows, tk = b / a.per, hh = b - tk * a.per;
        h.b = b; h.per = a.per;
        h.xr = a.x + (uint64_t)tk * a.x_tstride + (uint64_t)hh * a.x_stride; h.w = a.w; h.o = a.out + (uint64_t)b * a.n;
        h.vr = a.kc ? a.v + (uint64_t)tk * a.v_tstride + (uint64_t)hh * a.n : nullptr;
    }
    return h;
}

// One head by one wave: out = x * (1 / sqrt(ss / n + eps)) * w, rope, and (key heads of a storing launch) the f16
// KV store. s: the wave's 512-float LDS stage. HAVE_SS: ss is given (else lane 0 sums the head from the stage).
template <bool HAVE_SS>
__device__ __forceinline__ void nr_run(const NormRope& a, const NrHead& h, float* s, int lane, float ss) {
    const int n = a.n, half = a.n_rot / 2;
    const bool store = h.vr != nullptr;
    // every load of the wave first (the head, its norm weights, the value row), then the rope angles while they land
    constexpr int NV = 512 / 64;
    float xv[NV], wv[NV], vv[NV];
#pragma unroll
    for (int j = 0; j < NV; j++) {
        const int i = lane + 64 * j;
        if (i < n) {
            xv[j] = h.xr[i];
            wv[j] = h.w[i];
            if (store) vv[j] = h.vr[i];
        }
    }
    const int pos = a.step[0] + h.b / h.per;
    float sn[NV / 2], cs[NV / 2];
#pragma unroll
    for (int j = 0; j < NV / 2; j++) {
        const int i = lane + 64 * j;
        if (i < half) {
            const double f = i < a.nfreq ? a.freq[i] : pow((double)a.base, -2.0 * (double)i / (double)a.n_rot);
            double sd, cd;
            sincos((double)pos * f, &sd, &cd);
            sn[j] = (float)sd;
            cs[j] = (float)cd;
        }
    }
    if constexpr (!HAVE_SS) {
#pragma unroll
        for (int j = 0; j < NV; j++)
            if (lane + 64 * j < n) s[lane + 64 * j] = xv[j];
        __builtin_amdgcn_wave_barrier();
        if (lane == 0)
            ss = nr_sumsq(n, [&](int i0, float4 (&r)[8]) {
#pragma unroll
                for (int c = 0; c < 8; c++) r[c] = *(const float4*)&s[i0 + 4 * c];
            });
        ss = __shfl(ss, 0, 64);
        __builtin_amdgcn_wave_barrier();  // lane 0's reads are done before the normed values overwrite the stage
    }
    const float sc = 1.0f / sqrtf(ss / (float)n + a.eps);
#pragma unroll
    for (int j = 0; j < NV; j++)
        if (lane + 64 * j < n) s[lane + 64 * j] = xv[j] * sc * wv[j];
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int j = 0; j < NV / 2; j++) {
        const int i = lane + 64 * j;
        if (i < half) {
            const float p = s[i], q = s[i + half];
            s[i] = p * cs[j] - q * sn[j];
            s[i + half] = p * sn[j] + q * cs[j];
        }
    }
    __builtin_amdgcn_wave_barrier();
    const uint64_t e = ((uint64_t)pos * h.per + h.b % h.per) * n;
#pragma unroll
    for (int j = 0; j < NV; j++) {
        const int i = lane + 64 * j;
        if (i < n) {
            const float r = s[i];
            h.o[i] = r;
            if (store) {
                a.kc[e + i] = f32_to_f16_bits(r);
                a.vc[e + i] = f32_to_f16_bits(vv[j]);
            }
        }
    }
    __builtin_amdgcn_wave_barrier();  // the stage is reused by the wave's next head
}

// A wave per head (decode: few heads, each wave's latency is the launch's).
__global__ __launch_bounds__(64 * NR_WAVES) void norm_rope_kernel(NormRope a) {
    __shared__ __align__(16) float sh[NR_WAVES][512];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int gb = (int)blockIdx.x * NR_WAVES + wave;
    if (gb >= a.qrows + a.rows) return;
    nr_run<false>(a, nr_head(a, gb), sh[wave], lane, 0.0f);
}

// Many heads of 128 values, all rotated (a prefill chunk): a block takes NR_MANY heads. Its threads stage the heads
// in LDS with every load issued at once; wave 0 then sums the squares a lane
// per head (the heads' sequential chains run side by side); each wave then takes 16 consecutive heads, a lane per
// rope pair (i, i + 64), recomputing the pair's angle only when the position changes. The arithmetic is
// norm_rope_kernel's, so both kernels give the same bits. STAGED: the value rows of stored key heads are requested with
// the heads and wait in LDS (66 KB a block, two a CU), else they are read where they are stored (33 KB, four a CU).
constexpr int NR_MANY = 64, NR_P = 129;  // heads a block; LDS pitch of a staged head (bank spread for the sums)
template <bool STAGED>
__global__ __launch_bounds__(64 * NR_WAVES) void norm_rope_many_kernel(NormRope a) {
    __shared__ float xs[NR_MANY][NR_P], vs[STAGED ? NR_MANY : 1][NR_P];
    __shared__ float ssq[NR_MANY];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int total = a.qrows + a.rows, g0 = (int)blockIdx.x * NR_MANY;
    const float qw0 = a.qrows ? a.qw[lane] : 0.0f, qw1 = a.qrows ? a.qw[lane + 64] : 0.0f;
    const float kw0 = a.rows ? a.w[lane] : 0.0f, kw1 = a.rows ? a.w[lane + 64] : 0.0f;
    // 16-byte chunk c = tid + 256 u of the block: head c / 32, values 4 (c % 32) ..
    float4 xv[8], vv[STAGED ? 8 : 1];
#pragma unroll
    for (int u = 0; u < 8; u++) {
        const int c = tid + 256 * u, j = c >> 5, g = g0 + j;
        if (g < total) {
            const NrHead h = nr_head(a, g);
            xv[u] = *(const float4*)(h.xr + 4 * (c & 31));
            if constexpr (STAGED)
                if (h.vr) vv[u] = *(const float4*)(h.vr + 4 * (c & 31));
        }
    }
#pragma unroll
    for (int u = 0; u < 8; u++) {
        const int c = tid + 256 * u, j = c >> 5, g = g0 + j, i = 4 * (c & 31);
        if (g < total) {
            xs[j][i] = xv[u].x; xs[j][i + 1] = xv[u].y; xs[j][i + 2] = xv[u].z; xs[j][i + 3] = xv[u].w;
            if constexpr (STAGED)
                if (g >= a.qrows && a.kc) {
                    vs[j][i] = vv[u].x; vs[j][i + 1] = vv[u].y; vs[j][i + 2] = vv[u].z; vs[j][i + 3] = vv[u].w;
                }
        }
    }
    __syncthreads();
    if (wave == 0) {
        float ss = 0.0f;
        if (g0 + lane < total) {
            const float* xr = xs[lane];
            ss = nr_sumsq(128, [&](int i0, float4 (&r)[8]) {
#pragma unroll
                for (int c = 0; c < 8; c++) r[c] = make_float4(xr[i0 + 4 * c], xr[i0 + 4 * c + 1], xr[i0 + 4 * c + 2], xr[i0 + 4 * c + 3]);
            });
        }
        ssq[lane] = ss;
    }
    __syncthreads();
    int cur = -1;  // position of the pair angle held
    float sn = 0.0f, cs = 1.0f;
    for (int jj = 0; jj < NR_MANY / NR_WAVES; jj++) {
        const int j = (NR_MANY / NR_WAVES) * wave + jj, g = g0 + j;
        if (g >= total) break;
        const NrHead h = nr_head(a, g);
        const int pos = a.step[0] + h.b / h.per;
        if (pos != cur) {
            cur = pos;
            const double f = lane < a.nfreq ? a.freq[lane] : pow((double)a.base, -2.0 * (double)lane / 128.0);
            double sd, cd;
            sincos((double)pos * f, &sd, &cd);
            sn = (float)sd;
            cs = (float)cd;
        }
        const bool q = g < a.qrows;
        const float sc = 1.0f / sqrtf(ssq[j] / 128.0f + a.eps);
        const float p = xs[j][lane] * sc * (q ? qw0 : kw0), r = xs[j][lane + 64] * sc * (q ? qw1 : kw1);
        const float o0 = p * cs - r * sn, o1 = p * sn + r * cs;
        h.o[lane] = o0;
        h.o[lane + 64] = o1;
        if (h.vr) {
            const uint64_t e = ((uint64_t)pos * h.per + h.b % h.per) * 128;
            a.kc[e + lane] = f32_to_f16_bits(o0);
            a.kc[e + lane + 64] = f32_to_f16_bits(o1);
            const float* vr = STAGED ? vs[j] : h.vr;
            a.vc[e + lane] = f32_to_f16_bits(vr[lane]);
            a.vc[e + lane + 64] = f32_to_f16_bits(vr[lane + 64]);
        }
    }
}

// rope_neox of pairs lo .. hi - 1 only (Backend::rope_pairs, src/backend.rs:254; kernel src/cuda/kernels.cu:1596-1610),
// in place on `heads` rows `stride` floats apart, head b of token b / per at position step[0] + b / per.
__global__ __launch_bounds__(64 * NR_WAVES) void rope_pairs_kernel(float* x, uint64_t stride, int heads, int per,
                                                                   int n_rot, const int* step, float base, int lo, int hi) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int b = (int)blockIdx.x * NR_WAVES + wave;
    if (b >= heads) return;
    const int pos = step[0] + b / per, half = n_rot / 2;
    float* h = x + (uint64_t)b * stride;
    for (int i = lane; i < half; i += 64) {
        if (i < lo || i >= hi) continue;
        const double theta = (double)pos * pow((double)base, -2.0 * (double)i / (double)n_rot);
        const float sn = (float)sin(theta), c = (float)cos(theta);
        const float p = h[i], q = h[i + half];
        h[i] = p * c - q * sn;
        h[i + half] = p * sn + q * c;
    }
}

// Whether the many-heads form stages the value rows: while its blocks all fit at two a CU, where a launch is one block's chain
// and the rows' latency part of it (128 tokens x 40 heads 13.6 us, 14.8 not staged; 1000 x 32 18.2, 20.9); with more blocks
// four a CU are faster (1501 x 36 29.0 staged, 26.5 not, 4096 x 36 59.2, 44.4; 1501 x 32 28.0, 23.9).
bool nr_staged(int heads, int ncu) { return (heads + NR_MANY - 1) / NR_MANY <= 2 * ncu; }

hipError_t launch_norm_rope(const NormRope& a0, hipStream_t s) {
    const int total = a0.qrows + a0.rows;
    if (total <= 0) return hipSuccess;
    // the rope frequencies depend only on the pair index: the host's pow (the one the CPU reference calls) fills
    // them once per launch, so the kernel's f64 work is the sine and cosine
    NormRope a = a0;
    if (!a.q_tstride) a.q_tstride = (uint64_t)a.qper * a.q_stride;
    if (!a.x_tstride) a.x_tstride = (uint64_t)a.per * a.x_stride;
    if (!a.v_tstride) a.v_tstride = (uint64_t)a.per * a.n;
    a.nfreq = a.n_rot / 2 <= NormRope::NFREQ ? a.n_rot / 2 : 0;
    for (int i = 0; i < a.nfreq; i++) a.freq[i] = std::pow((double)a.base, -2.0 * (double)i / (double)a.n_rot);
    const bool vec = ((uintptr_t)a.qx | (uintptr_t)a.x | (uintptr_t)a.v) % 16 == 0 && a.q_stride % 4 == 0 &&
                     a.x_stride % 4 == 0 && a.q_tstride % 4 == 0 && a.x_tstride % 4 == 0 && a.v_tstride % 4 == 0;
    const unsigned many = (unsigned)((total + NR_MANY - 1) / NR_MANY);
    if (total >= 4 * NR_MANY && vec && a.n == 128 && a.n_rot == 128) {  // the many-heads form: 16-byte chunks, heads of 128
        if (!nr_staged(total, cu_count())) norm_rope_many_kernel<false><<<dim3(many), dim3(64 * NR_WAVES), 0, s>>>(a);
        else norm_rope_many_kernel<true><<<dim3(many), dim3(64 * NR_WAVES), 0, s>>>(a);
    } else
        norm_rope_kernel<<<dim3((unsigned)((total + NR_WAVES - 1) / NR_WAVES)), dim3(64 * NR_WAVES), 0, s>>>(a);
    return hipGetLastError();
}

hipError_t launch_rope_pairs(float* x, uint64_t stride, int heads, int per, int n_rot, const int* step, float base,
                             int lo, int hi, hipStream_t s) {
    if (heads <= 0 || hi <= lo) return hipSuccess;
    rope_pairs_kernel<<<dim3((unsigned)((heads + NR_WAVES - 1) / NR_WAVES)), dim3(64 * NR_WAVES), 0, s>>>(
        x, stride, heads, per, n_rot, step, base, lo, hi);
    return hipGetLastError();
}

// kv_store (src/cuda/kernels.cu:2181-2186): value i of the t tokens' rows of n goes to cache element step[0] n + i.
__global__ __launch_bounds__(256) void kv_store_kernel(const float* k, const float* v, uint16_t* kc, uint16_t* vc,
                                                       uint64_t n, uint64_t total, const int* step) {
    const uint64_t base = (uint64_t)step[0] * n;
    for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (uint64_t)gridDim.x * 256) {
        kc[base + i] = f32_to_f16_bits(k[i]);
        vc[base + i] = f32_to_f16_bits(v[i]);
    }
}

hipError_t launch_kv_store(const float* k, const float* v, uint16_t* kc, uint16_t* vc, int n, int t, const int* step,
                           hipStream_t s) {
    const uint64_t total = (uint64_t)n * t;
    if (!total) return hipSuccess;
    const uint64_t blocks = std::min<uint64_t>((total + 255) / 256, 4096);
    kv_store_kernel<<<dim3((unsigned)blocks), dim3(256), 0, s>>>(k, v, kc, vc, (uint64_t)n, total, step);
    return hipGetLastError();
}

// ---- argmax ----
// ops::argmax's order (src/ops.rs:110-112): the largest value under f32::total_cmp, the first index on ties. A value
// and its index pack into one 64-bit key whose unsigned maximum is that choice: the total-order image of the bits
// above, ~index below.
constexpr int AMAX_PARTS = 64;

__device__ __forceinline__ uint64_t amax_key(float v, int i) {
    const int32_t b = __float_as_int(v);
    const uint32_t u = (uint32_t)(b ^ (int32_t)((uint32_t)(b >> 31) >> 1)) ^ 0x80000000u;
    return ((uint64_t)u << 32) | (uint32_t)(0xFFFFFFFFu - (uint32_t)i);
}
__device__ __forceinline__ uint64_t wave_max_u64(uint64_t k) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        const uint32_t lo = __shfl_xor((uint32_t)k, o, 64), hi = __shfl_xor((uint32_t)(k >> 32), o, 64);
        const uint64_t other = ((uint64_t)hi << 32) | lo;
        k = other > k ? other : k;
    }
    return k;
}

__global__ __launch_bounds__(256) void argmax_part_kernel(const float* x, int n, uint64_t* part) {
    __shared__ uint64_t sk[4];
    const float* xr = x + (uint64_t)blockIdx.y * n;
    uint64_t best = 0;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += AMAX_PARTS * 256) {
        const uint64_t k = amax_key(xr[i], i);
        best = k > best ? k : best;
    }
    best = wave_max_u64(best);
    if ((threadIdx.x & 63) == 0) sk[threadIdx.x >> 6] = best;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint64_t b = sk[0];
        for (int w = 1; w < 4; w++) b = sk[w] > b ? sk[w] : b;
        part[(uint64_t)blockIdx.y * AMAX_PARTS + blockIdx.x] = b;
    }
}

__global__ __launch_bounds__(64) void argmax_final_kernel(const uint64_t* part, int* out) {
    const uint64_t k = wave_max_u64(part[(uint64_t)blockIdx.x * AMAX_PARTS + threadIdx.x]);
    if (threadIdx.x == 0) out[blockIdx.x] = (int)(0xFFFFFFFFu - (uint32_t)k);
}

uint64_t argmax_part_bytes(int rows) { return (uint64_t)rows * AMAX_PARTS * 8; }

hipError_t launch_argmax_rows(const float* x, int n, int rows, uint64_t* part, int* out, hipStream_t s) {
    if (rows <= 0) return hipSuccess;
    argmax_part_kernel<<<dim3(AMAX_PARTS, (unsigned)rows), dim3(256), 0, s>>>(x, n, part);
    argmax_final_kernel<<<dim3((unsigned)rows), dim3(64), 0, s>>>(part, out);
    return hipGetLastError();
}

// ---- elementwise ----
__global__ __launch_bounds__(256) void add_kernel(float* x, const float* y, uint64_t n) {
    for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (uint64_t)gridDim.x * 256) x[i] = x[i] + y[i];
}
__global__ __launch_bounds__(256) void swiglu_kernel(float* g, const float* u, uint64_t n) {
    for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (uint64_t)gridDim.x * 256)
        g[i] = silu_f32(g[i]) * u[i];
}
static unsigned ew_blocks(uint64_t n) { return (unsigned)std::min<uint64_t>((n + 255) / 256, 8192); }

hipError_t launch_add(float* x, const float* y, uint64_t n, hipStream_t s) {
    if (!n) return hipSuccess;
    add_kernel<<<dim3(ew_blocks(n)), dim3(256), 0, s>>>(x, y, n);
    return hipGetLastError();
}
hipError_t launch_swiglu(float* g, const float* u, uint64_t n, hipStream_t s) {
    if (!n) return hipSuccess;
    swiglu_kernel<<<dim3(ew_blocks(n)), dim3(256), 0, s>>>(g, u, n);
    return hipGetLastError();
}

// ---- embedding rows: out[i] = dequant(row min(ids[i], rows - 1)) (Model::embed, src/model.rs:334-339) ----
template <int T>
__global__ __launch_bounds__(256) void get_rows_kernel(const uint8_t* __restrict__ w, uint64_t rb, uint64_t rows,
                                                       int cols, const int* ids, uint64_t groups, float* __restrict__ out) {
    const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= groups) return;
    const int gpr = cols / 32;
    const uint64_t r = i / gpr;
    const int g = (int)(i % gpr);
    const int id = ids[r];
    const uint64_t src = id < 0 ? 0 : (uint64_t)id >= rows ? rows - 1 : (uint64_t)id;
    const uint8_t* sb = w + src * rb + (uint64_t)(g / 8) * sb_bytes(T);
    float v[32];
    dequant32<T>(sb, g % 8, v);
    float4* o = (float4*)(out + r * cols + 32 * g);
#pragma unroll
    for (int j = 0; j < 8; j++) o[j] = make_float4(v[4 * j], v[4 * j + 1], v[4 * j + 2], v[4 * j + 3]);
}

template <int T>
static hipError_t get_rows_t(const uint8_t* w, uint64_t rows, uint64_t cols, const int* ids, int n, float* out,
                             hipStream_t s) {
    const uint64_t groups = (uint64_t)n * (cols / 32);
    if (!groups) return hipSuccess;
    get_rows_kernel<T><<<dim3((unsigned)((groups + 255) / 256)), dim3(256), 0, s>>>(w, row_bytes(T, cols), rows,
                                                                                   (int)cols, ids, groups, out);
    return hipGetLastError();
}

hipError_t launch_get_rows(int ty, const uint8_t* w, uint64_t rows, uint64_t cols, const int* ids, int n, float* out,
                           hipStream_t s) {
    switch (ty) {
    case Q8_0: return get_rows_t<Q8_0>(w, rows, cols, ids, n, out, s);
    case Q2_K: return get_rows_t<Q2_K>(w, rows, cols, ids, n, out, s);
    case Q3_K: return get_rows_t<Q3_K>(w, rows, cols, ids, n, out, s);
    case Q4_K: return get_rows_t<Q4_K>(w, rows, cols, ids, n, out, s);
    case Q5_K: return get_rows_t<Q5_K>(w, rows, cols, ids, n, out, s);
    case Q6_K: return get_rows_t<Q6_K>(w, rows, cols, ids, n, out, s);
    case IQ2_XXS: return get_rows_t<IQ2_XXS>(w, rows, cols, ids, n, out, s);
    case IQ3_S: return get_rows_t<IQ3_S>(w, rows, cols, ids, n, out, s);
    case IQ4_XS: return get_rows_t<IQ4_XS>(w, rows, cols, ids, n, out, s);
    }
    return hipErrorInvalidValue;
}

// ---- f32-weight GEMV: one wave per weight row, every input of the launch on that row ----
constexpr int GF_NT = 4;
__global__ __launch_bounds__(256) void gemv_f32_kernel(const float* __restrict__ w, int rows, int cols,
                                                       const float* __restrict__ x, uint64_t x_stride, float* y,
                                                       uint64_t y_stride, int nt, int act) {
    const int r = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (r >= rows) return;
    const float4* wr = (const float4*)(w + (uint64_t)r * cols);
    float acc[GF_NT] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int c = lane; c < cols / 4; c += 64) {
        const float4 wv = wr[c];
#pragma unroll
        for (int t = 0; t < GF_NT; t++) {
            if (t < nt) {
                const float4 xv = ((const float4*)(x + t * x_stride))[c];
                acc[t] += wv.x * xv.x + wv.y * xv.y + wv.z * xv.z + wv.w * xv.w;
            }
        }
    }
#pragma unroll
    for (int t = 0; t < GF_NT; t++) {
        if (t < nt) {
            const float v = wave_sum_xor(acc[t]);
            if (lane == 0) {
                float* yo = y + t * y_stride + r;
                *yo = act == 2 ? *yo + v : v;
            }
        }
    }
}

// One input (a decode step): a wave per row, a block per wave; each pass loads GF1_U 16-byte chunks of the row and of
// x per lane before using any, so a 2048-value row takes one memory round trip. A lane sums the same chunks in the
// same order as gemv_f32_kernel, so both kernels give the same bits.
constexpr int GF1_U = 8;
__global__ __launch_bounds__(64) void gemv_f32_1_kernel(const float* __restrict__ w, int rows, int cols,
                                                        const float* __restrict__ x, float* y, int act) {
    const int r = blockIdx.x, lane = threadIdx.x, n4 = cols / 4;
    const float4* wr = (const float4*)(w + (uint64_t)r * cols);
    const float4* xr = (const float4*)x;
    float acc = 0.0f;
    for (int c0 = 0; c0 < n4; c0 += 64 * GF1_U) {
        float4 wv[GF1_U], xv[GF1_U];
#pragma unroll
        for (int u = 0; u < GF1_U; u++) {
            const int c = c0 + lane + 64 * u;
            wv[u] = c < n4 ? wr[c] : make_float4(0.f, 0.f, 0.f, 0.f);
            xv[u] = c < n4 ? xr[c] : make_float4(0.f, 0.f, 0.f, 0.f);
        }
#pragma unroll
        for (int u = 0; u < GF1_U; u++)
            if (c0 + lane + 64 * u < n4) acc += wv[u].x * xv[u].x + wv[u].y * xv[u].y + wv[u].z * xv[u].z + wv[u].w * xv[u].w;
    }
    const float v = wave_sum_xor(acc);
    if (lane == 0) y[r] = act == 2 ? y[r] + v : v;
}

hipError_t launch_gemv_f32(const float* w, int rows, int cols, const float* x, uint64_t x_stride, float* y,
                           uint64_t y_stride, int nt, int act, hipStream_t s) {
    if (!rows || !nt) return hipSuccess;
    if (nt == 1) {
        gemv_f32_1_kernel<<<dim3((unsigned)rows), dim3(64), 0, s>>>(w, rows, cols, x, y, act);
        return hipGetLastError();
    }
    for (int t0 = 0; t0 < nt; t0 += GF_NT) {
        const int n = std::min(GF_NT, nt - t0);
        gemv_f32_kernel<<<dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, s>>>(w, rows, cols, x + t0 * x_stride, x_stride,
                                                                                y + t0 * y_stride, y_stride, n, act);
    }
    return hipGetLastError();
}

// ---- f32-weight GEMM (gemm_dense of a float matrix): each output's dot runs over k in index order with a multiply
// then an add, as Tensor::matvec's f32 iterator sum (src/weights.rs:29-37): the CPU's bits. That makes every output
// one dependent chain of 2 cols instructions (a lone wave issues one in 5-6 cycles), so few outputs are bound by the
// chain and many by the VALU (62 us for 4096 x 128 x 2048 at two instructions a term). Four forms by the work they leave a
// CU (gemm_f32_form); router of 128 x 2048, us a call, before (one form: 4 chains a lane, x and weights
// through one LDS buffer whose loads each step waited for) and now: 27 tokens 72 -> 18, 512 72 -> 29, 1501 72 -> 39,
// 4096 77 -> 66. ----

// A block of 4 waves takes 64 positions (a lane each) x 4 RW weight rows (RW chains a lane). x and the weight rows come
// by direct global-to-LDS loads into a ring of gf_nb steps of 32 k (three or four steps in flight: one step's work is
// shorter than a trip to memory), the registers of a group are read from it one group ahead. x sits as [position][32 k]
// with 16-byte chunk c of position p at c ^ ((p / 2) & 7): the 16 lanes of a 16-byte read touch every bank once.
constexpr int GF_M = 64, GF_K = 32;  // positions a block; k of a step
// Steps in the LDS ring: as many as leave three blocks a CU (512 x 2048, 1501 positions: six steps, two blocks a CU 119 us,
// five steps, three blocks 90).
constexpr int gf_nb(int rw) { return rw == 1 ? 6 : 5; }
constexpr int gf_lds(int rw) { return gf_nb(rw) * (GF_M + 4 * rw) * GF_K * 4; }
static_assert(3 * gf_lds(1) <= 160 * 1024 && 3 * gf_lds(2) <= 160 * 1024 && 3 * gf_lds(4) <= 160 * 1024, "three blocks a CU");
template <int RW>
__global__ __launch_bounds__(256) void gemm_f32_kernel(const float* __restrict__ w, int rows, int cols,
                                                       const float* __restrict__ x, uint64_t x_stride, float* y,
                                                       uint64_t y_stride, int n, int act) {
    constexpr int GK = 32 / RW, GS = GF_K / GK;  // k of a register group; groups a step
    constexpr int NL = GF_M * GF_K * 4 / 1024 / 4;          // load instructions a wave and step
    constexpr int GF_NB = gf_nb(RW);
    __shared__ __align__(16) float xs[GF_NB][GF_M * GF_K];
    __shared__ __align__(16) float ws[GF_NB][4 * RW * GF_K];
    const int m0 = blockIdx.x * GF_M, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r0 = blockIdx.y * 4 * RW + RW * wave;
    const int nst = (cols + GF_K - 1) / GF_K;
    // load instruction i of this wave: x rows 8 (NL wave + i) + lane / 8, LDS chunk lane % 8 of the row holding its
    // chunk (lane % 8) ^ (row / 2 % 8); rows past n read the last row, columns past the end the row's last ones (unused)
    const float* xr[NL];
    int xc[NL];
#pragma unroll
    for (int i = 0; i < NL; i++) {
        const int r = 8 * (NL * wave + i) + (lane >> 3);
        xr[i] = x + (uint64_t)min(m0 + r, n - 1) * x_stride;
        xc[i] = 4 * ((lane & 7) ^ ((r >> 1) & 7));
    }
    const float* wr = w + (uint64_t)min(r0 + (lane >> 3), rows - 1) * cols;
    auto issue = [&](int st, int b) __attribute__((always_inline)) {
        const int k0 = min(st, nst - 1) * GF_K;
#pragma unroll
        for (int i = 0; i < NL; i++) load_lds16((uint64_t)(xr[i] + min(k0 + xc[i], cols - 4)), &xs[b][256 * (NL * wave + i)]);
        if (lane < 8 * RW) load_lds16((uint64_t)(wr + min(k0 + 4 * (lane & 7), cols - 4)), &ws[b][RW * GF_K * wave]);
    };
    float acc[RW] = {};
    float4 xa[2][GK / 4];
    float4 wa[2][RW][GK / 4];
    // the registers of group gi (k = GK gi ..): x and the weights (one address a wave: a broadcast) from the step's buffers
    auto fetch = [&](int gi, int b, float4 (&xg)[GK / 4], float4 (&ww)[RW][GK / 4]) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < GK / 4; q++) xg[q] = *(const float4*)&xs[b][lane * GF_K + 4 * (((gi % GS) * (GK / 4) + q) ^ ((lane >> 1) & 7))];
#pragma unroll
        for (int j = 0; j < RW; j++)
#pragma unroll
            for (int q = 0; q < GK / 4; q++) ww[j][q] = *(const float4*)&ws[b][(RW * wave + j) * GF_K + (gi % GS) * GK + 4 * q];
    };
    auto run = [&](const float4 (&xg)[GK / 4], const float4 (&ww)[RW][GK / 4]) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < GK / 4; q++) {
            const float a[4] = {xg[q].x, xg[q].y, xg[q].z, xg[q].w};
            float p[4][RW];
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int j = 0; j < RW; j++) {
                    const float4 wq = ww[j][q];
                    p[e][j] = a[e] * (e == 0 ? wq.x : e == 1 ? wq.y : e == 2 ? wq.z : wq.w);
                    if constexpr (RW == 1) asm volatile("" : "+v"(p[e][j]));
                }
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int j = 0; j < RW; j++) acc[j] += p[e][j];
        }
    };
    const int ng = cols / GK;
#pragma unroll
    for (int b = 0; b < GF_NB - 1; b++) issue(b, b);
    wait_vm<(NL + 1) * (GF_NB - 2)>();
    lds_barrier();
    if (ng > 0) fetch(0, 0, xa[0], wa[0]);
    int b = 0;
    // one step; PAR: its first group's register set
    auto step = [&](int st, auto PAR) __attribute__((always_inline)) {
        constexpr int par = decltype(PAR)::value;
        const int b1 = b + 1 == GF_NB ? 0 : b + 1, bp = b == 0 ? GF_NB - 1 : b - 1;
        wait_vm<(NL + 1) * (GF_NB - 3)>();  // this wave's loads of step st + 1
        lds_barrier();                // everybody's; and buffer bp (step st - 1) has been read
        issue(st + GF_NB - 1, bp);
#pragma unroll
        for (int u = 0; u < GS; u++) {
            const int gi = st * GS + u;
            if (gi >= ng) break;
            wait_lds();  // this group's registers, all at once: the next group's reads then run under all of its products
                         // (4 rows a wave: 70.3 us at 512 x 2048, 1024 positions, with the compiler's waits one by one, 67.4 so)
            // (past the last group the last one again, unused)
            fetch(gi + 1 < ng ? gi + 1 : gi, u + 1 < GS || gi + 1 >= ng ? b : b1, xa[(par + u + 1) & 1], wa[(par + u + 1) & 1]);
            run(xa[(par + u) & 1], wa[(par + u) & 1]);
#pragma unroll
            for (int j = 0; j < RW; j++) asm volatile("" : "+v"(acc[j]));  // (keeps this group's work ahead of the next wait)
        }
        if (st + 1 == nst)  // the last columns, less than a group
            for (int k = ng * GK; k < cols; k++)
#pragma unroll
                for (int j = 0; j < RW; j++)
                    acc[j] += xs[b][lane * GF_K + 4 * (((k - st * GF_K) >> 2) ^ ((lane >> 1) & 7)) + (k & 3)] * ws[b][(RW * wave + j) * GF_K + k - st * GF_K];
        b = b1;
    };
    for (int st = 0; st < nst; st += 2) {
        step(st, std::integral_constant<int, 0>{});
        if (st + 1 < nst) step(st + 1, std::integral_constant<int, GS & 1>{});
    }
    wait_loads();  // (the ring's loads past the last step)
    const int m = m0 + lane;
    if (m < n) {
#pragma unroll
        for (int j = 0; j < RW; j++) {
            const int r = r0 + j;
            if (r >= rows) continue;
            float* yo = y + (uint64_t)m * y_stride + r;
            const float v = acc[j];
            *yo = act == 0 ? v : act == 1 ? silu_f32(*yo) * v : *yo + v;
        }
    }
}

// Few outputs: four lanes share an output's products (lane e of a quad holds terms 4 e .. 4 e + 3 of each 16, one
// multiply for four terms) and each of them runs the whole chain, taking the products by quad permutes that fold into
// the adds; a wave takes 16 rows x P positions, whose chains interleave (an add may not follow its predecessor within
// two issues), U groups of 16 terms loaded ahead.
template <int P, int U>
__global__ __launch_bounds__(256) void gemm_f32_quad_kernel(const float* __restrict__ w, int rows, int cols,
                                                            const float* __restrict__ x, uint64_t x_stride, float* y,
                                                            uint64_t y_stride, int n, int act) {
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, e = lane & 3;
    const int m = (blockIdx.x * 4 + wave) * P, r = blockIdx.y * 16 + (lane >> 2);
    if (m >= n) return;
    const float* xr[P];
#pragma unroll
    for (int j = 0; j < P; j++) xr[j] = x + (uint64_t)min(m + j, n - 1) * x_stride + 4 * e;
    const float* wr = w + (uint64_t)min(r, rows - 1) * cols + 4 * e;
    float4 xv[2][P][U], wv[2][U];
    auto load = [&](int k0, float4 (&xx)[P][U], float4 (&ww)[U]) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int k = min(k0 + 16 * u + 4 * e, cols - 4) - 4 * e;
            ww[u] = *(const float4*)(wr + k);
#pragma unroll
            for (int j = 0; j < P; j++) xx[j][u] = *(const float4*)(xr[j] + k);
        }
    };
    float acc[P] = {};
    auto run = [&](int k0, const float4 (&xx)[P][U], const float4 (&ww)[U], auto TAIL) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (decltype(TAIL)::value && k0 + 16 * u >= cols) break;
            float p[P][4];
            const bool live = !decltype(TAIL)::value || k0 + 16 * u + 4 * e < cols;
#pragma unroll
            for (int j = 0; j < P; j++) {
                p[j][0] = live ? ww[u].x * xx[j][u].x : 0.0f; p[j][1] = live ? ww[u].y * xx[j][u].y : 0.0f;
                p[j][2] = live ? ww[u].z * xx[j][u].z : 0.0f; p[j][3] = live ? ww[u].w * xx[j][u].w : 0.0f;
            }
            static_for<0, 16>([&](auto I) {
                constexpr int i = decltype(I)::value;
#pragma unroll
                for (int j = 0; j < P; j++) acc[j] += quad_bcast<(i >> 2)>(p[j][i & 3]);
            });
        }
    };
    constexpr int KP = 16 * U;
    load(0, xv[0], wv[0]);
    int k0 = 0;
    for (; k0 + 2 * KP <= cols; k0 += 2 * KP) {
        load(k0 + KP, xv[1], wv[1]);
        run(k0, xv[0], wv[0], std::false_type{});
        load(k0 + 2 * KP, xv[0], wv[0]);
        run(k0 + KP, xv[1], wv[1], std::false_type{});
    }
    for (; k0 < cols; k0 += KP) {
        run(k0, xv[0], wv[0], std::true_type{});
        load(k0 + KP, xv[0], wv[0]);
    }
    if (e == 0 && r < rows) {
#pragma unroll
        for (int j = 0; j < P; j++)
            if (m + j < n) {
                float* yo = y + (uint64_t)(m + j) * y_stride + r;
                *yo = act == 0 ? acc[j] : act == 1 ? silu_f32(*yo) * acc[j] : *yo + acc[j];
            }
    }
}
template <int RW>
static void gemm_f32_t(const float* w, int rows, int cols, const float* x, uint64_t x_stride, float* y, uint64_t y_stride,
                       int n, int act, hipStream_t s) {
    const dim3 grid((unsigned)((n + GF_M - 1) / GF_M), (unsigned)((rows + 4 * RW - 1) / (4 * RW)));
    gemm_f32_kernel<RW><<<grid, dim3(256), 0, s>>>(w, rows, cols, x, x_stride, y, y_stride, n, act);
}

// The form of an F32 GEMM: 0 the quad form, else the ring form of that many rows a wave (1, 2, 4). Each form's cost in us
// for 2048 columns, from what it leaves the fullest CU: the quad form by its waves a SIMD (2 positions x 16 rows each: 18 us
// for one, 28-31 for two, 39 / 51 / 133 / 196 for 3 / 4 / 9 / 16), a ring form by its blocks of 64 positions x 4 RW rows, three
// of them a CU at a time (RW 1: 29 / 31 / 40 us for 1 / 2 / 3 blocks, 57 / 72 / 96 for 4 / 6 / 8; RW 2: 41 / 46, 85 / 109 /
// 142; RW 4: 59 / 68 / 90, 128 for 4, 213 for 8). Counting outputs alone gave a tall matrix of few positions to the ring
// form with most lanes idle: 5 positions of 16384 x 2048 176 us, in the quad form 56.
int gemm_f32_form(int n, int rows, int ncu) {
    auto cdiv = [](long long a, long long b) { return (a + b - 1) / b; };
    const long long r = cdiv(cdiv(n, 2) * cdiv(rows, 16), 4ll * ncu);
    long long best = r == 1 ? 18 : r == 2 ? 29 : 13 * r + 4;
    int form = 0;
    constexpr int RW[3] = {1, 2, 4};
    constexpr int COST[3][5] = {{29, 31, 36, 21, 26}, {41, 46, 54, 31, 38}, {59, 68, 88, 32, 40}};
    for (int i = 0; i < 3; i++) {
        const long long b = cdiv(cdiv(n, GF_M) * cdiv(rows, 4 * RW[i]), ncu);
        const long long cost = b < 3 ? COST[i][b - 1] : COST[i][2] * (b / 3) + (b % 3 ? COST[i][2 + b % 3] : 0);
        if (cost < best) {
            best = cost;
            form = RW[i];
        }
    }
    return form;
}

hipError_t launch_gemm_f32(const float* w, int rows, int cols, const float* x, uint64_t x_stride, float* y,
                           uint64_t y_stride, int n, int act, hipStream_t s) {
    if (!rows || !n) return hipSuccess;
    // (the ring's loads into LDS take 16-byte aligned weight rows, the quad form any float's address)
    switch ((uintptr_t)w % 16 ? 0 : gemm_f32_form(n, rows, cu_count())) {
    case 0: {
        constexpr int P = 2, U = 8;
        const dim3 grid((unsigned)((n + 4 * P - 1) / (4 * P)), (unsigned)((rows + 15) / 16));
        gemm_f32_quad_kernel<P, U><<<grid, dim3(256), 0, s>>>(w, rows, cols, x, x_stride, y, y_stride, n, act);
        break;
    }
    case 1: gemm_f32_t<1>(w, rows, cols, x, x_stride, y, y_stride, n, act, s); break;
    case 2: gemm_f32_t<2>(w, rows, cols, x, x_stride, y, y_stride, n, act, s); break;
    default: gemm_f32_t<4>(w, rows, cols, x, x_stride, y, y_stride, n, act, s); break;
    }
    return hipGetLastError();
}

// ---- synthetic weights: random block bytes with every f16 scale field in [lo, hi) (the reference's random_tensor
// design, tests/kernels.rs:1473-1550), from a counter-based hash of (seed, position) ----
__device__ __forceinline__ uint64_t mix64(uint64_t z) {
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

__global__ __launch_bounds__(256) void fill_bytes_kernel(uint8_t* w, uint64_t bytes, uint64_t seed) {
    const uint64_t words = bytes / 4;
    for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < (bytes + 3) / 4; i += (uint64_t)gridDim.x * 256) {
        const uint32_t r = (uint32_t)mix64(seed * 0x9E3779B97F4A7C15ull + i);
        if (i < words) {
            ((uint32_t*)w)[i] = r;
        } else {
            for (uint64_t b = 4 * i; b < bytes; b++) w[b] = (uint8_t)(r >> (8 * (b - 4 * i)));
        }
    }
}

__global__ __launch_bounds__(256) void fill_scales_kernel(uint8_t* w, uint64_t n_blocks, int bb, int f0, int f1,
                                                          uint64_t seed, float lo, float hi) {
    for (uint64_t b = (uint64_t)blockIdx.x * 256 + threadIdx.x; b < n_blocks; b += (uint64_t)gridDim.x * 256) {
        const uint64_t r = mix64(~seed * 0xD1B54A32D192ED03ull + b);
        const float u0 = (float)(uint32_t)r * 2.3283064365386963e-10f, u1 = (float)(uint32_t)(r >> 32) * 2.3283064365386963e-10f;
        *(uint16_t*)(w + b * bb + f0) = f32_to_f16_bits(lo + (hi - lo) * u0);
        if (f1 >= 0) *(uint16_t*)(w + b * bb + f1) = f32_to_f16_bits(lo + (hi - lo) * u1);
    }
}

hipError_t launch_fill_blocks(int ty, uint8_t* w, uint64_t n_blocks, uint64_t seed, float lo, float hi, hipStream_t s) {
    if (!n_blocks) return hipSuccess;
    const int bb = block_bytes(ty);
    int f0 = 0, f1 = -1;  // offsets of the f16 scale fields in a block (d, and dmin where the type has one)
    switch (ty) {
    case Q2_K: f0 = 80; f1 = 82; break;
    case Q3_K: f0 = 108; break;
    case Q4_K: case Q5_K: f0 = 0; f1 = 2; break;
    case Q6_K: f0 = 208; break;
    default: f0 = 0; break;
    }
    const uint64_t bytes = n_blocks * (uint64_t)bb;
    fill_bytes_kernel<<<dim3(ew_blocks((bytes + 3) / 4)), dim3(256), 0, s>>>(w, bytes, seed);
    fill_scales_kernel<<<dim3(ew_blocks(n_blocks)), dim3(256), 0, s>>>(w, n_blocks, bb, f0, f1, seed, lo, hi);
    return hipGetLastError();
}

}  // namespace strata
