// The banded KV cache's codec on the GPU (gfx950): a filled segment of keys or values, (heads, seq, dim) activations, becomes
// ids of a fixed width per head with one (min, step) per channel, and banded segments become the id layout attention reads.
//
//   range   per channel the smallest and largest value, as partial results per chunk of rows; joined by a launch of its own
//   check   per head the width that certifies tau (or the width the caller asks for), and how far the decoder's values would
//           lie from the input: nothing is written but those figures
//   pack    ids = round((x - min) / step) at the heads' final widths, bit-packed LSB first
//   unpack  packed heads -> one byte (or 16 bits) per id at their places in the layout, constants in centre form
//
// All four are bound by memory: x is read once per kernel (8 MB per 4096-key segment of 4 heads x 256 channels stay in the
// caches after the first), everything else is smaller.  Measured on such a segment, keys and values and their layout:
// 2868 us as ~100 torch launches with 64-bit temporaries per bit; 193 us with a launch for each of range, join, check and pack and the
// check's thousand figures written to the host; 146 us with the join in the check, three figures a head, and the ids packed at the
// width asked for while those are on their way; 126 us with several rows' loads on their way at once and the heads' counters apart.
// What is left is launches: the kernels take 58 of them, 250 keys of 2 x 64 channels take 95 (153 before).
//
// Arithmetic is the codec's own expression by expression: fp32 differences, one IEEE division, rounding to nearest even,
// products and sums rounded separately (contraction is off in this file).
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <algorithm>

#include "../../include/qvb8_amd.h"
#include "qvb8_device.h"
#include "qvb8_host.h"

#pragma clang fp contract(off)

namespace qvb8 {
namespace {

constexpr int kKvThreads = 256;
constexpr int kKvMaxDim = 2048;                // channels per head: the constants of a head lie in LDS
constexpr float kKvStepFloor = 1e-12f;

__device__ __forceinline__ float finite_or_zero(float v) { return __builtin_fabsf(v) < __builtin_inff() ? v : 0.f; }   // NaN compares false

// V neighbouring values of a row as they are stored, and as fp32 (NaN and infinities read as 0).  Loading and converting are apart, so
// that the loads of several rows are on their way together.
template <int DT, int V>
struct Values {
    static constexpr int kWords = V == 8 ? (DT == QVB8_F32 ? 8 : 4) : 1;
    uint32_t w[kWords];
    __device__ __forceinline__ void load(const void* x, int64_t at) {
        if constexpr (V == 8) {
            const uint4* p = reinterpret_cast<const uint4*>(reinterpret_cast<const uint8_t*>(x) + at * (DT == QVB8_F32 ? 4 : 2));
#pragma unroll
            for (int k = 0; k < kWords / 4; ++k) {
                const uint4 q = p[k];
                w[4 * k] = q.x; w[4 * k + 1] = q.y; w[4 * k + 2] = q.z; w[4 * k + 3] = q.w;
            }
        } else {
            w[0] = DT == QVB8_F32 ? reinterpret_cast<const uint32_t*>(x)[at] : reinterpret_cast<const uint16_t*>(x)[at];
        }
    }
    __device__ __forceinline__ float operator[](int k) const {
        if constexpr (DT == QVB8_F32) return finite_or_zero(__builtin_bit_cast(float, w[k]));
        const uint32_t h = (w[k / 2] >> (16 * (k % 2))) & 0xFFFFu;
        return finite_or_zero(DT == QVB8_F16 ? f16_bits_to_f32(h) : bf16_bits_to_f32(h));
    }
};
template <int DT, int V>
__device__ __forceinline__ void load_values(const void* x, int64_t at, float (&v)[V]) {
    Values<DT, V> raw;
    raw.load(x, at);
#pragma unroll
    for (int k = 0; k < V; ++k) v[k] = raw[k];
}
// Rows in flight per thread (range: twice as many).  One row after the other, a trip to memory each, the range of 4 x 4096 x 256 bf16
// values took 9.1 us; 5.4 this way.
constexpr int kKvRows = 4;

// grid (chunks, heads).  partial[head][chunk][2][dim]: minima, maxima of the chunk's rows.  A thread owns V neighbouring
// channels and every `groups`-th row; the row groups meet in LDS.  `clear` (or null): two words per head, zeroed for the launch that follows.
// Words that many workgroups add to lie this far apart: atomics on one cache line wait for each other (128 workgroups of four heads on one
// line: the check takes 20.2 us, 11.5 this way).
constexpr int kStateApart = 64;
constexpr int kRangeThreads = 512;            // there are few chunks: every workgroup that follows reads all their results
template <int DT, int V>
__global__ void __launch_bounds__(kRangeThreads) kv_range_kernel(const void* x, int seq, int dim, int rows_per_chunk, float* partial, uint32_t* clear) {
    extern __shared__ float s_red[];                                   // [groups][dim] x 2
    const int head = blockIdx.y, chunk = blockIdx.x;
    if (clear && chunk == 0 && threadIdx.x < 2) clear[(2 * head + threadIdx.x) * kStateApart] = 0u;
    const int nv = dim / V, across = min(nv, kRangeThreads), groups = kRangeThreads / across;
    const int cv0 = threadIdx.x % across, group = threadIdx.x / across;
    const int r0 = chunk * rows_per_chunk, r1 = min(seq, r0 + rows_per_chunk);
    float* s_hi = s_red + groups * dim;
    if (group < groups) {
        for (int cv = cv0; cv < nv; cv += across) {
            float lo[V], hi[V];
#pragma unroll
            for (int k = 0; k < V; ++k) { lo[k] = __builtin_inff(); hi[k] = -__builtin_inff(); }
            for (int r = r0 + group; r < r1; r += groups * 2 * kKvRows) {
                Values<DT, V> v[2 * kKvRows];                          // (a row past the end: the last one again)
#pragma unroll
                for (int j = 0; j < 2 * kKvRows; ++j) v[j].load(x, ((int64_t)head * seq + min(r + j * groups, r1 - 1)) * dim + cv * V);
#pragma unroll
                for (int j = 0; j < 2 * kKvRows; ++j)
#pragma unroll
                    for (int k = 0; k < V; ++k) { lo[k] = fminf(lo[k], v[j][k]); hi[k] = fmaxf(hi[k], v[j][k]); }
            }
#pragma unroll
            for (int k = 0; k < V; ++k) { s_red[group * dim + cv * V + k] = lo[k]; s_hi[group * dim + cv * V + k] = hi[k]; }
        }
    }
    __syncthreads();
    float* out = partial + ((int64_t)head * gridDim.x + chunk) * 2 * dim;
    for (int c = threadIdx.x; c < dim; c += kRangeThreads) {
        float lo = s_red[c], hi = s_hi[c];
        for (int g = 1; g < groups; ++g) { lo = fminf(lo, s_red[g * dim + c]); hi = fmaxf(hi, s_hi[g * dim + c]); }
        out[c] = lo;
        out[dim + c] = hi;
    }
}

struct KvWidths { uint8_t w[QVB8_KV_MAX_HEADS]; };

__device__ __forceinline__ float block_max(float v, float* s4) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    if ((threadIdx.x & 63) == 0) s4[threadIdx.x >> 6] = v;
    __syncthreads();
    v = fmaxf(fmaxf(s4[0], s4[1]), fmaxf(s4[2], s4[3]));
    __syncthreads();
    return v;
}
__device__ __forceinline__ float step_of(float span, int width) {
    return fmaxf(span / (float)((1u << width) - 1u), kKvStepFloor);
}
__device__ __forceinline__ float id_of(float x, float lo, float step, float top) {
    return fminf(fmaxf(rintf((x - lo) / step), 0.f), top);
}

// Joins the partial minima and maxima: grid (ceil(dim / 64), heads); wave w takes every sixteenth chunk, the waves meet in LDS.  A
// chain of trips; the calls that wait for it (qvb8_kv_measure) join in the check instead.
constexpr int kJoinWaves = 16;
__global__ void __launch_bounds__(64 * kJoinWaves) kv_join_kernel(int dim, int chunks, const float* partial, float* lo_out, float* span_out) {
    __shared__ float s_lo[kJoinWaves][64], s_hi[kJoinWaves][64];
    const int head = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = blockIdx.x * 64 + lane;
    const float* p = partial + (int64_t)head * chunks * 2 * dim + min(c, dim - 1);
    float lo = __builtin_inff(), hi = -__builtin_inff();
#pragma unroll 8
    for (int k = wave; k < chunks; k += kJoinWaves) { lo = fminf(lo, p[(int64_t)k * 2 * dim]); hi = fmaxf(hi, p[(int64_t)k * 2 * dim + dim]); }
    s_lo[wave][lane] = lo;
    s_hi[wave][lane] = hi;
    __syncthreads();
    if (wave == 0 && c < dim) {
#pragma unroll
        for (int w = 1; w < kJoinWaves; ++w) { lo = fminf(lo, s_lo[w][lane]); hi = fmaxf(hi, s_hi[w][lane]); }
        lo_out[(int64_t)head * dim + c] = lo;
        span_out[(int64_t)head * dim + c] = hi - lo;
    }
}

// What qvb8_kv_measure adds: the partial ranges to join, two zeroed words per head (largest error, workgroups that are done), and
// where the figures go -- found[head][3] in memory the host reads: largest span, width, largest error.
constexpr int kJoinAtOnce = 16;                // (a partial result past the last: that one again)
struct KvShown { const float* partial; int partials; uint32_t* state; float* found; };

// grid (chunks, heads).  Fixes the head's width -- `given`, or the least one >= bits with half a step within tau -- and measures
// the chunk's largest |decoded - x|.  report[head][2 + chunks]: largest span, width, the chunks' errors.
template <int DT, int V>
__global__ void __launch_bounds__(kKvThreads) kv_check_kernel(const void* x, int seq, int dim, int rows_per_chunk, int orig_dt,
                                                              int bits, double tau, int use_given, KvWidths given, float* lo_io, float* span_io,
                                                              float* report, KvShown shown) {
    __shared__ float s_lo[kKvMaxDim], s_step[kKvMaxDim], s4[4];
    const int head = blockIdx.y, chunk = blockIdx.x, chunks = gridDim.x;
    const int nv = dim / V, across = min(nv, kKvThreads), groups = kKvThreads / across;
    const int cv0 = threadIdx.x % across, group = threadIdx.x / across;
    const int r0 = chunk * rows_per_chunk, r1 = min(seq, r0 + rows_per_chunk);
    Values<DT, V> v[kKvRows];
    auto load_rows = [&](int r, int cv) __attribute__((always_inline)) {   // (a row past the end: the last one again)
#pragma unroll
        for (int j = 0; j < kKvRows; ++j) v[j].load(x, ((int64_t)head * seq + min(r + j * groups, r1 - 1)) * dim + cv * V);
    };
    const bool any = group < groups && r0 + group < r1;
    if (any) load_rows(r0 + group, cv0);                       // on their way while the ranges are joined
    float widest = 0.f;
    for (int c = threadIdx.x; c < dim; c += kKvThreads) {
        float lo, span;
        if (shown.found) {
            // every workgroup joins the partial ranges itself (a few dozen per channel): a launch less in front of the host's wait
            const float* p = shown.partial + (int64_t)head * shown.partials * 2 * dim + c;
            float hi = -__builtin_inff();
            lo = __builtin_inff();
            for (int k0 = 0; k0 < shown.partials; k0 += kJoinAtOnce) {
                float l[kJoinAtOnce], h[kJoinAtOnce];
#pragma unroll
                for (int j = 0; j < kJoinAtOnce; ++j) {
                    const float* at = p + (int64_t)min(k0 + j, shown.partials - 1) * 2 * dim;
                    l[j] = at[0];
                    h[j] = at[dim];
                }
#pragma unroll
                for (int j = 0; j < kJoinAtOnce; ++j) { lo = fminf(lo, l[j]); hi = fmaxf(hi, h[j]); }
            }
            span = hi - lo;
            if (chunk == 0) { lo_io[(int64_t)head * dim + c] = lo; span_io[(int64_t)head * dim + c] = span; }
        } else {
            lo = lo_io[(int64_t)head * dim + c];
            span = span_io[(int64_t)head * dim + c];
        }
        s_lo[c] = lo;
        s_step[c] = span;
        widest = fmaxf(widest, span);
    }
    widest = block_max(widest, s4);
    int width = use_given ? (int)given.w[head] : bits;
    if (!use_given && widest > 0.f) {
        const double v = (double)widest / (2.0 * tau) + 1.0;
        const uint64_t b = __builtin_bit_cast(uint64_t, v);            // smallest w with 2^w >= v, v >= 1
        const int e = (int)((b >> 52) & 2047) - 1023;
        width = min(16, max(bits, e + ((b & 0xFFFFFFFFFFFFFull) ? 1 : 0)));
    }
    for (int c = threadIdx.x; c < dim; c += kKvThreads) s_step[c] = step_of(s_step[c], width);
    __syncthreads();
    const float top = (float)((1u << width) - 1u);
    float worst = 0.f;
    if (any) {
        for (int cv = cv0; cv < nv; cv += across) {
            float lo[V], step[V];
#pragma unroll
            for (int k = 0; k < V; ++k) { lo[k] = s_lo[cv * V + k]; step[k] = s_step[cv * V + k]; }
            for (int r = r0 + group; r < r1; r += groups * kKvRows) {
                if (r != r0 + group || cv != cv0) load_rows(r, cv);
#pragma unroll
                for (int j = 0; j < kKvRows; ++j) {
                    if (j > 0 && r + j * groups >= r1) break;
#pragma unroll
                    for (int k = 0; k < V; ++k) {
                        const float given_value = v[j][k];
                        float shown = lo[k] + id_of(given_value, lo[k], step[k], top) * step[k];
                        if (orig_dt == QVB8_F16) shown = f16_bits_to_f32(f32_to_f16_bits(shown));
                        else if (orig_dt == QVB8_BF16) shown = bf16_bits_to_f32(f32_to_bf16_bits(shown));
                        worst = fmaxf(worst, __builtin_fabsf(shown - given_value));
                    }
                }
            }
        }
    }
    worst = block_max(worst, s4);
    if (shown.found) {
        if (threadIdx.x == 0) {
            // The head's largest error and the number of its workgroups that have added theirs, both as atomics at the device's
            // point of coherence, the second issued when the first has returned: the last one finds every error in.
            uint32_t *state = shown.state + 2 * head * kStateApart, *done = state + kStateApart;
            const uint32_t before = __hip_atomic_fetch_max(state, __builtin_bit_cast(uint32_t, worst), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            asm volatile("" :: "v"(before) : "memory");
            __builtin_amdgcn_s_waitcnt(0x0F70);                        // vmcnt(0)
            if (__hip_atomic_fetch_add(done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (uint32_t)chunks - 1u) {
                const uint32_t all = __hip_atomic_fetch_max(state, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                // three words a head across the bus (a word per workgroup, written by each: 6 of 15.8 us)
                uint32_t* to = reinterpret_cast<uint32_t*>(shown.found) + 3 * head;
                __hip_atomic_store(to, __builtin_bit_cast(uint32_t, widest), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                __hip_atomic_store(to + 1, __builtin_bit_cast(uint32_t, (float)width), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                __hip_atomic_store(to + 2, all, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            }
        }
        return;
    }
    if (threadIdx.x == 0) {
        float* rep = report + (int64_t)head * (2 + chunks);
        rep[2 + chunk] = worst;
        if (chunk == 0) { rep[0] = widest; rep[1] = (float)width; }
    }
}

struct KvPackArgs {
    const void* x; const float* lo; const float* span; float* step;
    int64_t n;                     // ids per head
    int dim, vec;
    uint8_t w[QVB8_KV_MAX_HEADS];
    uint8_t* out[QVB8_KV_MAX_HEADS];
};

// grid (blocks, heads).  A thread makes 32 consecutive ids: `width` whole dwords of the head's stream (the last, shorter group of
// a head: bytes).
template <int DT>
__global__ void __launch_bounds__(kKvThreads) kv_pack_kernel(KvPackArgs a) {
    __shared__ __align__(16) float s_lo[kKvMaxDim], s_step[kKvMaxDim];
    const int head = blockIdx.y, width = a.w[head];
    for (int c = threadIdx.x; c < a.dim; c += kKvThreads) {
        const float step = step_of(a.span[(int64_t)head * a.dim + c], width);
        s_lo[c] = a.lo[(int64_t)head * a.dim + c];
        s_step[c] = step;
        if (blockIdx.x == 0) a.step[(int64_t)head * a.dim + c] = step;
    }
    __syncthreads();
    const int64_t i0 = ((int64_t)blockIdx.x * kKvThreads + threadIdx.x) * 32;
    if (i0 >= a.n) return;
    const int count = (int)(a.n - i0 < 32 ? a.n - i0 : 32);
    const float top = (float)((1u << width) - 1u);
    const int64_t base = (int64_t)head * a.n + i0;
    int c = (int)(i0 % a.dim);
    uint8_t* to = a.out[head] + i0 / 8 * width;
    uint64_t acc = 0;
    int have = 0;
    auto put = [&](float v) __attribute__((always_inline)) {
        acc |= (uint64_t)(uint32_t)id_of(v, s_lo[c], s_step[c], top) << have;
        have += width;
        if (++c == a.dim) c = 0;
    };
    if (count == 32) {
        uint32_t* to4 = reinterpret_cast<uint32_t*>(to);
        auto flush = [&]() __attribute__((always_inline)) { if (have >= 32) { *to4++ = (uint32_t)acc; acc >>= 32; have -= 32; } };
        if (a.vec) {                                           // eight channels at a time: they are neighbours in LDS
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float v[8];
                load_values<DT, 8>(a.x, base + 8 * j, v);
                const float4 l0 = *reinterpret_cast<const float4*>(s_lo + c), l1 = *reinterpret_cast<const float4*>(s_lo + c + 4);
                const float4 t0 = *reinterpret_cast<const float4*>(s_step + c), t1 = *reinterpret_cast<const float4*>(s_step + c + 4);
                const float l[8] = {l0.x, l0.y, l0.z, l0.w, l1.x, l1.y, l1.z, l1.w}, t[8] = {t0.x, t0.y, t0.z, t0.w, t1.x, t1.y, t1.z, t1.w};
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    acc |= (uint64_t)(uint32_t)id_of(v[k], l[k], t[k], top) << have;
                    have += width;
                    flush();
                }
                c += 8;
                if (c == a.dim) c = 0;
            }
        } else {
            for (int k = 0; k < 32; ++k) {
                float v[1];
                load_values<DT, 1>(a.x, base + k, v);
                put(v[0]);
                flush();
            }
        }
    } else {
        for (int k = 0; k < count; ++k) {
            float v[1];
            load_values<DT, 1>(a.x, base + k, v);
            put(v[0]);
            while (have >= 8) { *to++ = (uint8_t)acc; acc >>= 8; have -= 8; }
        }
        if (have > 0) *to = (uint8_t)acc;
    }
}

struct KvUnpackArgs {
    qvb8_kv_head h[QVB8_KV_MAX_HEADS];
    int dim, id_bytes;
    int64_t row_stride;            // ids from a key to the next in the layout
};

// grid (blocks, entries).  A thread takes 32 consecutive ids of a head's stream: with dim % 32 == 0 they lie in one key's row.
__global__ void __launch_bounds__(kKvThreads) kv_unpack_kernel(KvUnpackArgs a) {
    const qvb8_kv_head& q = a.h[blockIdx.y];
    const int bits = q.bits;
    const float c = (float)((1u << bits) - 1u) * 0.5f;
    if (blockIdx.x == 0) {
        for (int k = threadIdx.x; k < a.dim; k += kKvThreads) {
            const float step = q.step[k];
            q.mid_out[k] = q.min[k] + step * c;
            q.step_out[k] = step;
        }
        if (threadIdx.x == 0) *q.centre_out = c;
    }
    const int64_t n = q.seq * a.dim, i0 = ((int64_t)blockIdx.x * kKvThreads + threadIdx.x) * 32;
    if (i0 >= n) return;
    const uint32_t mask = (1u << bits) - 1u;
    if ((a.dim & 31) == 0) {
        const uint32_t* p = reinterpret_cast<const uint32_t*>(q.packed + i0 / 8 * bits);
        const int64_t at = i0 / a.dim * a.row_stride + i0 % a.dim;
        uint64_t acc = 0;
        int have = 0;
        auto next = [&]() __attribute__((always_inline)) {
            if (have < bits) { acc |= (uint64_t)*p++ << have; have += 32; }
            const uint32_t v = (uint32_t)acc & mask;
            acc >>= bits;
            have -= bits;
            return v;
        };
        if (a.id_bytes == 1) {
            uint4* to = reinterpret_cast<uint4*>(reinterpret_cast<uint8_t*>(q.ids_out) + at);
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                uint32_t w[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) { w[k] = next(); w[k] |= next() << 8; w[k] |= next() << 16; w[k] |= next() << 24; }
                to[j] = uint4{w[0], w[1], w[2], w[3]};
            }
        } else {
            uint4* to = reinterpret_cast<uint4*>(reinterpret_cast<uint16_t*>(q.ids_out) + at);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                uint32_t w[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) { w[k] = next(); w[k] |= next() << 16; }
                to[j] = uint4{w[0], w[1], w[2], w[3]};
            }
        }
    } else {
        const int64_t last = (n * bits + 7) / 8 - 1;
        for (int64_t i = i0; i < n && i < i0 + 32; ++i) {
            const int64_t bit = i * bits, b = bit >> 3;
            uint32_t v = q.packed[b] | ((uint32_t)q.packed[b + 1 > last ? last : b + 1] << 8) | ((uint32_t)q.packed[b + 2 > last ? last : b + 2] << 16);
            v = (v >> (bit & 7)) & mask;
            const int64_t at = i / a.dim * a.row_stride + i % a.dim;
            if (a.id_bytes == 1) reinterpret_cast<uint8_t*>(q.ids_out)[at] = (uint8_t)v;
            else reinterpret_cast<uint16_t*>(q.ids_out)[at] = (uint16_t)v;
        }
    }
}

constexpr int kKvTileSegs = 256;
struct KvTileArgs { int len[kKvTileSegs]; int n_seg, first_seg, pos, at, block_n, n_tiles; };
__global__ void __launch_bounds__(kKvThreads) kv_tiles_kernel(KvTileArgs a, int32_t* table) {
    int pos = a.pos, at = a.at;
    for (int s = 0; s < a.n_seg; ++s) {
        const int len = a.len[s], tiles = (len + a.block_n - 1) / a.block_n;
        for (int i = threadIdx.x; i < tiles; i += kKvThreads) {
            table[at + i] = pos + i * a.block_n;
            table[a.n_tiles + at + i] = min(a.block_n, len - i * a.block_n);
            table[2 * a.n_tiles + at + i] = a.first_seg + s;
        }
        pos += len;
        at += tiles;
    }
}

template <typename F>
int by_dtype(int dt, F f) {
    if (dt == QVB8_F32) f(std::integral_constant<int, QVB8_F32>{});
    else if (dt == QVB8_F16) f(std::integral_constant<int, QVB8_F16>{});
    else f(std::integral_constant<int, QVB8_BF16>{});
    return 0;
}
int bad_shape(const char* who, const void* x, int x_dtype, int64_t heads, int64_t seq, int64_t dim) {
    if (!x || x_dtype < QVB8_F32 || x_dtype > QVB8_BF16) return host::fail(QVB8_ERR_ARG, "%s: null input or unknown dtype", who);
    if (heads < 1 || heads > QVB8_KV_MAX_HEADS || seq < 1 || dim < 1 || seq * dim > 0x7fffffff) return host::fail(QVB8_ERR_ARG, "%s: bad shape", who);
    if (dim > kKvMaxDim) return host::fail(QVB8_ERR_UNSUPPORTED, "%s: more than %d channels", who, kKvMaxDim);
    return 0;
}
bool vectors_ok(const void* x, int64_t dim) { return dim % 8 == 0 && (reinterpret_cast<uintptr_t>(x) & 15u) == 0; }
int rows_per_chunk(int64_t seq, int64_t chunks) { return (int)((seq + chunks - 1) / chunks); }

}  // namespace
}  // namespace qvb8

using namespace qvb8;

// four workgroups per CU over the heads, at least 16 rows each
extern "C" int64_t qvb8_kv_chunks(int64_t heads, int64_t seq) {
    if (heads < 1 || seq < 1) return 1;
    const int64_t want = std::max<int64_t>(1, 4 * host::device_cus() / heads);
    return std::max<int64_t>(1, std::min<int64_t>({want, (seq + 15) / 16, 256}));
}

namespace {
int kv_range(const void* x, int x_dtype, int64_t heads, int64_t seq, int64_t dim, float* partial, int64_t chunks, uint32_t* clear, void* stream) {
    if (int rc = bad_shape("qvb8_kv_range", x, x_dtype, heads, seq, dim)) return rc;
    if (!partial || chunks < 1 || chunks > 65535) return host::fail(QVB8_ERR_ARG, "qvb8_kv_range: bad partial results");
    const bool vec = vectors_ok(x, dim);
    const int nv = (int)(vec ? dim / 8 : dim), across = std::min(nv, kRangeThreads), groups = kRangeThreads / across;
    const size_t lds = (size_t)groups * dim * 8;
    const dim3 grid((unsigned)chunks, (unsigned)heads);
    by_dtype(x_dtype, [&](auto dt) {
        constexpr int DT = decltype(dt)::value;
        if (vec) hipLaunchKernelGGL((kv_range_kernel<DT, 8>), grid, dim3(kRangeThreads), lds, (hipStream_t)stream, x, (int)seq, (int)dim, rows_per_chunk(seq, chunks), partial, clear);
        else hipLaunchKernelGGL((kv_range_kernel<DT, 1>), grid, dim3(kRangeThreads), lds, (hipStream_t)stream, x, (int)seq, (int)dim, rows_per_chunk(seq, chunks), partial, clear);
    });
    return host::check_launch("qvb8_kv_range");
}
}  // namespace

extern "C" int qvb8_kv_range(const void* x, int x_dtype, int64_t heads, int64_t seq, int64_t dim, float* partial, int64_t chunks, void* stream) {
    return kv_range(x, x_dtype, heads, seq, dim, partial, chunks, nullptr, stream);
}

extern "C" int qvb8_kv_check(const void* x, int x_dtype, int64_t heads, int64_t seq, int64_t dim, const float* partial, int64_t chunks, int orig_dtype,
                             int bits, double tau, const uint8_t* widths, float* lo, float* span, float* report, void* stream) {
    if (int rc = bad_shape("qvb8_kv_check", x, x_dtype, heads, seq, dim)) return rc;
    if (!partial || !lo || !span || chunks < 1 || chunks > 65535 || orig_dtype < QVB8_F32 || orig_dtype > QVB8_BF16)
        return host::fail(QVB8_ERR_ARG, "qvb8_kv_check: bad argument");
    if (!widths)                                               // (asked again with other widths: minima and spans are there)
        hipLaunchKernelGGL(kv_join_kernel, dim3((unsigned)((dim + 63) / 64), (unsigned)heads), dim3(64 * kJoinWaves), 0, (hipStream_t)stream, (int)dim, (int)chunks, partial, lo, span);
    if (!report) return host::check_launch("qvb8_kv_check");   // nothing to certify
    if (bits < 1 || bits > 16 || !(tau > 0)) return host::fail(QVB8_ERR_ARG, "qvb8_kv_check: widths are 1..16 bits, tau > 0");
    KvWidths given = {};
    if (widths)
        for (int64_t h = 0; h < heads; ++h) {
            if (widths[h] < 1 || widths[h] > 16) return host::fail(QVB8_ERR_ARG, "qvb8_kv_check: widths are 1..16 bits");
            given.w[h] = widths[h];
        }
    const dim3 grid((unsigned)chunks, (unsigned)heads);
    by_dtype(x_dtype, [&](auto dt) {
        constexpr int DT = decltype(dt)::value;
        if (vectors_ok(x, dim)) hipLaunchKernelGGL((kv_check_kernel<DT, 8>), grid, dim3(kKvThreads), 0, (hipStream_t)stream, x, (int)seq, (int)dim, rows_per_chunk(seq, chunks), orig_dtype, bits, tau, widths ? 1 : 0, given, lo, span, report, KvShown{});
        else hipLaunchKernelGGL((kv_check_kernel<DT, 1>), grid, dim3(kKvThreads), 0, (hipStream_t)stream, x, (int)seq, (int)dim, rows_per_chunk(seq, chunks), orig_dtype, bits, tau, widths ? 1 : 0, given, lo, span, report, KvShown{});
    });
    return host::check_launch("qvb8_kv_check");
}

extern "C" int qvb8_kv_pack(const void* x, int x_dtype, int64_t heads, int64_t seq, int64_t dim, const float* lo, const float* span, const uint8_t* widths,
                            float* step, uint8_t* const* packed, void* stream) {
    if (int rc = bad_shape("qvb8_kv_pack", x, x_dtype, heads, seq, dim)) return rc;
    if (!lo || !span || !widths || !step || !packed) return host::fail(QVB8_ERR_ARG, "qvb8_kv_pack: null pointer");
    KvPackArgs a = {};
    a.x = x; a.lo = lo; a.span = span; a.step = step; a.n = seq * dim; a.dim = (int)dim; a.vec = vectors_ok(x, dim) && a.n % 8 == 0 ? 1 : 0;
    for (int64_t h = 0; h < heads; ++h) {
        if (widths[h] < 1 || widths[h] > 16 || !packed[h] || (reinterpret_cast<uintptr_t>(packed[h]) & 3u))
            return host::fail(QVB8_ERR_ARG, "qvb8_kv_pack: widths are 1..16 bits, outputs 4-byte aligned");
        a.w[h] = widths[h];
        a.out[h] = packed[h];
    }
    const dim3 grid((unsigned)((a.n + 32 * kKvThreads - 1) / (32 * kKvThreads)), (unsigned)heads);
    by_dtype(x_dtype, [&](auto dt) { hipLaunchKernelGGL((kv_pack_kernel<decltype(dt)::value>), grid, dim3(kKvThreads), 0, (hipStream_t)stream, a); });
    return host::check_launch("qvb8_kv_pack");
}

// Ranges, least widths and their errors as two launches, the figures on their way to the host when it has packed at the widths it
// expects (qvb8_kv_pack) and comes to wait for them (qvb8_kv_wait).
namespace {
// Partial ranges per head: every workgroup of the check joins them all.  Few heads and long segments leave CUs idle in the range pass (32
// workgroups a head), and still gain by the launch saved; a tensor as asked, range + join + check with up to 256 partials a head / this,
// us: 1 x 32768 x 128 55 / 42, 1 x 131072 x 256 166 / 152, 2 x 131072 x 128 127 / 107, 1 x 16384 x 2048 246 / 246, 4 x 4096 x 256 65 / 37.
constexpr int64_t kMeasurePartials = 32;
int64_t measure_partials(int64_t seq) { return std::max<int64_t>(1, std::min<int64_t>(kMeasurePartials, (seq + 15) / 16)); }
constexpr uint32_t kUnwritten = 0xBF800000u;                   // -1: none of the figures is negative
}
extern "C" int64_t qvb8_kv_measure_floats(int64_t heads, int64_t seq, int64_t dim) {
    return heads < 1 || seq < 1 || dim < 1 ? 0 : heads * (measure_partials(seq) * 2 * dim + 2 * kStateApart);
}
extern "C" int qvb8_kv_measure(const void* x, int x_dtype, int64_t heads, int64_t seq, int64_t dim, int orig_dtype, int bits, double tau,
                               float* scratch, float* lo, float* span, float* found, void* stream) {
    if (int rc = bad_shape("qvb8_kv_measure", x, x_dtype, heads, seq, dim)) return rc;
    if (!scratch || !lo || !span || !found || (reinterpret_cast<uintptr_t>(found) & 3u) || orig_dtype < QVB8_F32 || orig_dtype > QVB8_BF16 || bits < 1 || bits > 16 || !(tau > 0))
        return host::fail(QVB8_ERR_ARG, "qvb8_kv_measure: bad argument");
    const int64_t partials = measure_partials(seq), chunks = std::min<int64_t>(qvb8_kv_chunks(heads, seq), std::max<int64_t>(1, 2 * host::device_cus() / heads));
    KvShown shown = {scratch, (int)partials, reinterpret_cast<uint32_t*>(scratch + heads * partials * 2 * dim), found};
    uint32_t* words = reinterpret_cast<uint32_t*>(found);
    for (int64_t i = 0; i < 3 * heads; ++i) __atomic_store_n(words + i, kUnwritten, __ATOMIC_RELEASE);
    if (int rc = kv_range(x, x_dtype, heads, seq, dim, scratch, partials, shown.state, stream)) return rc;
    const dim3 grid((unsigned)chunks, (unsigned)heads);
    by_dtype(x_dtype, [&](auto dt) {
        constexpr int DT = decltype(dt)::value;
        if (vectors_ok(x, dim)) hipLaunchKernelGGL((kv_check_kernel<DT, 8>), grid, dim3(kKvThreads), 0, (hipStream_t)stream, x, (int)seq, (int)dim, rows_per_chunk(seq, chunks), orig_dtype, bits, tau, 0, KvWidths{}, lo, span, nullptr, shown);
        else hipLaunchKernelGGL((kv_check_kernel<DT, 1>), grid, dim3(kKvThreads), 0, (hipStream_t)stream, x, (int)seq, (int)dim, rows_per_chunk(seq, chunks), orig_dtype, bits, tau, 0, KvWidths{}, lo, span, nullptr, shown);
    });
    return host::check_launch("qvb8_kv_measure");
}

extern "C" int qvb8_kv_wait(const float* found, int64_t heads, void* stream) {
    if (!found || heads < 1 || heads > QVB8_KV_MAX_HEADS) return host::fail(QVB8_ERR_ARG, "qvb8_kv_wait: bad argument");
    const uint32_t* words = reinterpret_cast<const uint32_t*>(found);
    const int64_t n = 3 * heads;
    int64_t at = 0;
    for (int64_t spins = 1; at < n; ++spins) {                 // ends with the stream at the latest
        while (at < n && __atomic_load_n(words + at, __ATOMIC_ACQUIRE) != kUnwritten) ++at;
        if (at == n || spins % host::kPollsPerQuery) continue;
        const hipError_t e = hipStreamQuery((hipStream_t)stream);
        if (e == hipErrorNotReady) continue;
        if (e != hipSuccess) return host::fail(QVB8_ERR_LAUNCH, "qvb8_kv_wait: the check did not run: %s", hipGetErrorString(e));
        for (; at < n; ++at)
            if (__atomic_load_n(words + at, __ATOMIC_ACQUIRE) == kUnwritten) return host::fail(QVB8_ERR_LAUNCH, "qvb8_kv_wait: the check left no figures");
    }
    return 0;
}

extern "C" int qvb8_kv_unpack(const qvb8_kv_head* list, int64_t n_list, int64_t dim, int id_bytes, int64_t row_stride, void* stream) {
    if (!list || n_list < 1 || dim < 1 || (id_bytes != 1 && id_bytes != 2) || row_stride < dim) return host::fail(QVB8_ERR_ARG, "qvb8_kv_unpack: bad argument");
    for (int64_t at = 0; at < n_list; at += QVB8_KV_MAX_HEADS) {
        KvUnpackArgs a = {};
        a.dim = (int)dim; a.id_bytes = id_bytes; a.row_stride = row_stride;
        const int64_t n = std::min<int64_t>(QVB8_KV_MAX_HEADS, n_list - at);
        int64_t most = 0;
        for (int64_t i = 0; i < n; ++i) {
            const qvb8_kv_head& h = list[at + i];
            if (!h.packed || !h.min || !h.step || !h.ids_out || !h.mid_out || !h.step_out || !h.centre_out || h.seq < 1 || h.bits < 1 || h.bits > 8 * id_bytes
                || (reinterpret_cast<uintptr_t>(h.packed) & 3u) || (dim % 32 == 0 && ((reinterpret_cast<uintptr_t>(h.ids_out) & 15u) || row_stride * id_bytes % 16)))
                return host::fail(QVB8_ERR_ARG, "qvb8_kv_unpack: bad entry %lld", (long long)(at + i));
            a.h[i] = h;
            most = std::max(most, h.seq);
        }
        const dim3 grid((unsigned)((most * dim + 32 * kKvThreads - 1) / (32 * kKvThreads)), (unsigned)n);
        hipLaunchKernelGGL(kv_unpack_kernel, grid, dim3(kKvThreads), 0, (hipStream_t)stream, a);
    }
    return host::check_launch("qvb8_kv_unpack");
}

extern "C" int qvb8_kv_tiles(const int64_t* seg_len, int64_t n_seg, int64_t block_n, int32_t* table, int64_t n_tiles, void* stream) {
    if (!seg_len || n_seg < 1 || block_n < 1 || !table) return host::fail(QVB8_ERR_ARG, "qvb8_kv_tiles: bad argument");
    int64_t keys = 0, tiles = 0;
    for (int64_t s = 0; s < n_seg; ++s) {
        if (seg_len[s] < 0) return host::fail(QVB8_ERR_ARG, "qvb8_kv_tiles: negative segment length");
        keys += seg_len[s];
        tiles += (seg_len[s] + block_n - 1) / block_n;
    }
    if (tiles != n_tiles || keys > 0x7fffffff - block_n) return host::fail(QVB8_ERR_ARG, "qvb8_kv_tiles: the table holds %lld tiles, the segments make %lld", (long long)n_tiles, (long long)tiles);
    KvTileArgs a = {};
    a.block_n = (int)block_n;
    a.n_tiles = (int)n_tiles;
    for (int64_t s0 = 0; s0 < n_seg; s0 += kKvTileSegs) {
        a.n_seg = (int)std::min<int64_t>(kKvTileSegs, n_seg - s0);
        a.first_seg = (int)s0;
        for (int i = 0; i < a.n_seg; ++i) a.len[i] = (int)seg_len[s0 + i];
        hipLaunchKernelGGL(kv_tiles_kernel, dim3(1), dim3(kKvThreads), 0, (hipStream_t)stream, a, table);
        for (int i = 0; i < a.n_seg; ++i) { a.pos += a.len[i]; a.at += (a.len[i] + a.block_n - 1) / a.block_n; }
    }
    return host::check_launch("qvb8_kv_tiles");
}
