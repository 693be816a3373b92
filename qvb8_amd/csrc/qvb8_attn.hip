// Attention of a block of query rows over a banded KV cache: keys and values stay in memory as 1- or 2-byte ids with
// one (centre value, step) per segment / kv head / channel and one id centre per segment / kv head,
//
//     k = fp16(kmid[c] + kstep[c] * (id - kc))          v likewise,
//
// and are restored tile by tile inside the kernel -- the full-precision K / V of the context never exist.  Semantics
// of the reference's kernel (kv/cuda_attn/qvattn_cuda.cu:97-255): one workgroup = one kv head x one split of the key
// tiles x one block of query rows (row r = token * G + g); tiles of at most 32 keys come from a table (first key,
// length, segment) and never straddle a segment; key position <= query position; online softmax with the
// probabilities rounded to fp16 before they are summed and multiplied; the result per split is the unnormalised
// accumulator plus (running max, running sum), which the caller combines.
//
// Shape of this kernel (gfx950): 256 threads = 4 waves per workgroup, 16 query rows (or 2 / 4 blocks of 16), 32 keys per tile.
//   * ids are requested TWO tiles ahead into two register sets (a trip to memory under load takes longer than one tile's
//     arithmetic): a wave reads whole key rows (64 lanes x 4 ids = 256 channels), every thread keeps the same four
//     channels for all its keys, so it holds 4 + 4 constants per operand; no request sits under a branch (a tile past
//     the split's end re-reads one cached line), so the counted waits leave the younger set in flight; the tile table
//     comes through the scalar unit;
//   * restored K goes to LDS as [key][channel], restored V as [channel][key] (a thread owns 4 keys x 4 channels, so the
//     transposition is free) with the 8-byte cells of a row swizzled by the channel group;
//   * S = Q K^T: wave w takes keys 16 (w % 2) .. + 15 and half w / 2 of the channels (v_mfma_f32_16x16x16_f16, its part
//     of Q kept in registers as the A operand); the two halves are added when S is read back;
//   * the softmax is computed once per workgroup (wave w rows 4 w .. 4 w + 3, sixteen lanes a row, two keys a lane, row
//     maxima and sums by data-parallel rotations inside the row); the probabilities, rounded to fp16, and the rows'
//     rescale factors reach the four waves through LDS in the A-operand layout of the second product;
//   * O += P V: wave w owns a quarter of the output channels, its operands asked for ahead of the softmax.
// A workgroup has few tiles (6 of 1024 for one token over 32768 keys), so its start counts: the tile table, then ids, queries and the
// first segment's constants in one trip.  With the queries loaded before, each waited for, and the operands of either product two at a
// time: 27.4 us a call, 26.7 now.
#include <hip/hip_runtime.h>
#include <math.h>
#include <algorithm>
#include <type_traits>
#include <stdint.h>

#include "qvb8_amd.h"
#include "qvb8_device.h"
#include "qvb8_host.h"

namespace qvb8 {
namespace {

typedef _Float16 h4_t __attribute__((ext_vector_type(4)));
typedef float f4_t __attribute__((ext_vector_type(4)));

constexpr int kRows = 16;          // query rows per workgroup
constexpr int kKeys = 32;          // keys per tile (the table's tiles are never longer)
constexpr int kAttnThreads = 256;
constexpr int kSStride = kKeys + 4;

struct AttnArgs {
    const void* q; int64_t sq_r, sq_h;                          // strides in elements
    int q_dt; float q_scale;                                    // kQReady: fp16 as the products take it; else QVB8_F32 / _F16 / _BF16, to be prepared
    const void* ki; const void* vi; int64_t s_n, s_h;           // strides in ids
    const float* kmid; const float* kstep; const float* vmid; const float* vstep; const float* kc; const float* vc;
    const int32_t* ts; const int32_t* tl; const int32_t* tseg;
    float* o; float* m; float* l;
    int q_pos0, n_tiles, tps, n_rows, G, nhkv;
    float scale;
};

// N x four channels of one query, 16 apart, from element offset `at`.  What is not ready is multiplied by the softmax scale, then
// clamped to fp16's finite range and rounded -- in this order, so that an outlier channel does not become an infinity.  Done by
// the row-block kernel where it reads its queries, 16 or 32 rows a workgroup; the kernel of many rows takes them ready (every one of its
// splits would prepare them again: 120 tokens over 16001 keys 97.4 us that way, 95.6 with a launch that does it once).
// All N requests stand together under one choice of type: with a choice per request every one was waited for before the next.
constexpr int kQReady = -1;
template <int N>
__device__ __forceinline__ void load_query(const AttnArgs& a, int64_t at, h4_t (&q)[N]) {
    auto narrow = [&](const float (&v)[4]) __attribute__((always_inline)) {
        uint32_t h[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) h[k] = sat_half_bits(v[k] * a.q_scale);
        return __builtin_bit_cast(h4_t, uint2{h[0] | (h[1] << 16), h[2] | (h[3] << 16)});
    };
    if (a.q_dt == QVB8_F32) {
        float4 f[N];
#pragma unroll
        for (int i = 0; i < N; ++i) f[i] = *reinterpret_cast<const float4*>(reinterpret_cast<const float*>(a.q) + at + 16 * i);
#pragma unroll
        for (int i = 0; i < N; ++i) q[i] = narrow({f[i].x, f[i].y, f[i].z, f[i].w});
        return;
    }
    uint2 w[N];
#pragma unroll
    for (int i = 0; i < N; ++i) w[i] = *reinterpret_cast<const uint2*>(reinterpret_cast<const uint16_t*>(a.q) + at + 16 * i);
    if (a.q_dt == kQReady) {
#pragma unroll
        for (int i = 0; i < N; ++i) q[i] = __builtin_bit_cast(h4_t, w[i]);
    } else if (a.q_dt == QVB8_F16) {
#pragma unroll
        for (int i = 0; i < N; ++i) q[i] = narrow({f16_bits_to_f32(w[i].x & 0xFFFFu), f16_bits_to_f32(w[i].x >> 16), f16_bits_to_f32(w[i].y & 0xFFFFu), f16_bits_to_f32(w[i].y >> 16)});
    } else {
#pragma unroll
        for (int i = 0; i < N; ++i) q[i] = narrow({bf16_bits_to_f32(w[i].x & 0xFFFFu), bf16_bits_to_f32(w[i].x >> 16), bf16_bits_to_f32(w[i].y & 0xFFFFu), bf16_bits_to_f32(w[i].y >> 16)});
    }
}

// Four neighbouring channels of one key, as they lie in memory.
template <typename T> struct Quad;
template <> struct Quad<uint8_t> {
    typedef uint32_t type;
    static __device__ __forceinline__ float id(type w, int c) { return (float)((w >> (8 * c)) & 0xFFu); }
};
template <> struct Quad<uint16_t> {
    typedef uint2 type;
    static __device__ __forceinline__ float id(type w, int c) { return (float)(((c < 2 ? w.x : w.y) >> (16 * (c & 1))) & 0xFFFFu); }
};

// Two restored values as one dword of fp16: lo = fp16(fma(s0, d0, m0)), hi = fp16(fma(s1, d1, m1)), the fused
// multiply-add rounded to fp32 FIRST and then to fp16, as the reference's `__floats2half2_rn(md + sp * (v - c))` does.
// Written as `(_Float16)fmaf(...)` the compiler emits v_fma_mixlo_f16, which rounds the exact sum to fp16 in one step:
// one fp16 ulp off in about one value of 4000 (measured against the oracle).  The conversion is kept out of its sight.
__device__ __forceinline__ uint32_t restore_pair(float s0, float d0, float m0, float s1, float d1, float m1) {
    const float lo = __builtin_fmaf(s0, d0, m0), hi = __builtin_fmaf(s1, d1, m1);
    uint32_t r;
    asm("v_cvt_pk_f16_f32 %0, %1, %2" : "=v"(r) : "v"(lo), "v"(hi));
    return r;
}

// The value of the lane N places further on in its row of 16 lanes (a data-parallel move inside the vector unit; four of
// them -- 8, 4, 2, 1 -- leave a row's maximum or sum in every lane, without the LDS trips of a general shuffle).
template <int N>
__device__ __forceinline__ float row_rotate(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x120 + N, 0xF, 0xF, false));
}
__device__ __forceinline__ float row_max16(float v) {
    v = fmaxf(v, row_rotate<8>(v)); v = fmaxf(v, row_rotate<4>(v)); v = fmaxf(v, row_rotate<2>(v)); return fmaxf(v, row_rotate<1>(v));
}
__device__ __forceinline__ float row_sum16(float v) {
    v += row_rotate<8>(v); v += row_rotate<4>(v); v += row_rotate<2>(v); return v + row_rotate<1>(v);
}

// One entry of the tile table through the scalar unit.  A plain load would do, but behind a barrier the compiler turns
// it into a vector load, and waiting for that one (the youngest request) also waits for every id request still in
// flight -- the prefetch would be worth nothing.
struct TileRef { int start, nlen, seg; bool ok; };
__device__ __forceinline__ void tile_entry(const int32_t* ts, const int32_t* tl, const int32_t* tseg, int t, TileRef& r) {
    const uint32_t off = (uint32_t)__builtin_amdgcn_readfirstlane(t) * 4u;
    int start, nlen, seg;
    asm volatile("s_load_dword %0, %3, %6\n\ts_load_dword %1, %4, %6\n\ts_load_dword %2, %5, %6\n\ts_waitcnt lgkmcnt(0)"
                 : "=&s"(start), "=&s"(nlen), "=&s"(seg) : "s"(ts), "s"(tl), "s"(tseg), "s"(off) : "memory");
    r.start = start; r.nlen = nlen; r.seg = seg;
}

// Three workgroups per compute unit (two with 16-bit ids and 256 channels, whose two register sets are twice as large):
// the third one is what hides a workgroup's barriers and dependent chains -- 74.9 against 82.3 us over 131072 keys.
// RB = blocks of 16 query rows a workgroup serves from one restored tile (1, 2 or 4): the restore, most of the work, is
// shared; every block has its own Q registers, scores, softmax state and accumulators (two workgroups per CU then).
template <int D, typename T, int RB>
__global__ __launch_bounds__(kAttnThreads, ((D == 256 && sizeof(T) == 2) || RB > 1) ? 2 : 3) void attn_kernel(const AttnArgs a) {
    constexpr int CG = D / 4;                  // channel groups (four channels each) of a key
    constexpr int KSTEP = kAttnThreads / CG;   // key groups (four keys each) that one pass of the workgroup covers
    constexpr int UNITS = D / 128;             // (4 keys x 4 channels) units per thread and tile
    constexpr int KROW = D + 4;                // halfs per key in LDS: 16 keys' 8-byte reads fall on all banks once
    constexpr int NF = D / 64;                 // 16-channel output fragments per wave
    constexpr int NKS = D / 32;                // 16-channel steps of S = Q K^T per wave
    using QD = Quad<T>;
    using U = typename QD::type;
    __shared__ __align__(16) _Float16 Ks[kKeys * KROW];
    __shared__ __align__(16) _Float16 Vt[D * kKeys];
    __shared__ __align__(16) float Ss[RB * 2 * kRows * kSStride];
    constexpr int kPStride = kKeys + 8;                       // halfs per row of P
    __shared__ __align__(16) _Float16 Ps[RB * kRows * kPStride];
    __shared__ __align__(16) float Al[RB * kRows];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n16 = lane & 15, kg = lane >> 4;
    const int kf = wave & 1, dh = wave >> 1;                  // this wave's 16 keys and its half of the channels in S
    const int h = blockIdx.x, sp = blockIdx.y, row0 = blockIdx.z * (RB * kRows);
    const int cg = tid % CG, kgp0 = tid / CG;

    // the lane's query rows (one per block) as the A operand of S = Q K^T: Q[row][16 ks + 4 kg .. + 3], ks in the wave's half
    h4_t qa[RB][NKS];
    auto queries = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            const int row = row0 + rb * kRows + n16;
            const bool row_ok = row < a.n_rows;
            const int rr = row_ok ? row : 0;
            load_query<NKS>(a, (int64_t)(rr / a.G) * a.sq_r + (int64_t)(h * a.G + rr % a.G) * a.sq_h + dh * (D / 2) + 4 * kg, qa[rb]);
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) qa[rb][ks] = row_ok ? qa[rb][ks] : h4_t{0, 0, 0, 0};
        }
    };
    const int qmin = a.q_pos0 + row0 / a.G;                                   // first position of the block's rows
    // the softmax's own split of the block: this lane's row and pair of keys
    const int srow = 4 * wave + (lane >> 4), kpair = lane & 15;             // row within a block
    const int qmax = a.q_pos0 + (min(row0 + RB * kRows, a.n_rows) - 1) / a.G; // last position any row of the workgroup sees

    // the head's ids: a scalar base; the thread's four channels are part of its (32-bit) offset
    const T* ki = reinterpret_cast<const T*>(a.ki) + (int64_t)h * a.s_h;
    const T* vi = reinterpret_cast<const T*>(a.vi) + (int64_t)h * a.s_h;
    const uint32_t cg_off = (uint32_t)(4 * cg) * (uint32_t)sizeof(T);
    const int t0 = (int)min((int64_t)sp * a.tps, (int64_t)a.n_tiles), t1 = (int)min((int64_t)t0 + a.tps, (int64_t)a.n_tiles);
    // ids of tile t into one register set: always 8 UNITS requests, none under a branch; keys past the tile's length
    // re-read its last key, and a tile that is not wanted -- past the split's end, or starting behind the last visible
    // position (tiles ascend: so do all after it) -- re-reads key 0 of the head (one cached line); neither is used.
    // A request's address is the tile's first key (scalar) plus the thread's key offset, fixed for the whole kernel
    // and clamped to the tile's last key (host-checked: 32 keys' stride fits 31 bits).
    const uint32_t key_stride = (uint32_t)a.s_n * (uint32_t)sizeof(T);      // bytes from one key to the next
    const uint32_t key_off0 = (uint32_t)(4 * kgp0) * key_stride;            // the thread's first key; its others lie a scalar further
    const unsigned char* kbytes = reinterpret_cast<const unsigned char*>(ki);
    const unsigned char* vbytes = reinterpret_cast<const unsigned char*>(vi);
    auto fetch = [&](int t, U (&rk)[UNITS][4], U (&rv)[UNITS][4], TileRef& ref) {
        tile_entry(a.ts, a.tl, a.tseg, min(t, t1 - 1), ref);
        ref.ok = __builtin_amdgcn_readfirstlane((int)(t < t1 && ref.start <= qmax)) != 0;      // scalar: the loop's branches stay uniform
        const int start = ref.ok ? ref.start : 0, nlen = ref.ok ? ref.nlen : 1;
        const int64_t tile_byte = (int64_t)start * a.s_n * (int64_t)sizeof(T);
        const uint32_t last_off = (uint32_t)max(nlen - 1, 0) * (uint32_t)a.s_n * (uint32_t)sizeof(T);
        const unsigned char* kb = kbytes + tile_byte;
        const unsigned char* vb = vbytes + tile_byte;
#pragma unroll
        for (int u = 0; u < UNITS; ++u)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t off = min(key_off0 + (uint32_t)(4 * KSTEP * u + j) * key_stride, last_off) + cg_off;
                rk[u][j] = *reinterpret_cast<const U*>(kb + off);
                rv[u][j] = *reinterpret_cast<const U*>(vb + off);
            }
    };

    float m_run[RB], l_run[RB];
    f4_t acc[RB][NF];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
        m_run[rb] = -INFINITY; l_run[rb] = 0.f;
#pragma unroll
        for (int f = 0; f < NF; ++f) acc[rb][f] = f4_t{0.f, 0.f, 0.f, 0.f};
    }

    int cur_seg = -1;
    float km[4] = {0.f, 0.f, 0.f, 0.f}, ks_[4] = {0.f, 0.f, 0.f, 0.f}, vm[4] = {0.f, 0.f, 0.f, 0.f}, vs_[4] = {0.f, 0.f, 0.f, 0.f}, kc = 0.f, vc = 0.f;
    // a segment's constants for this thread's four channels
    auto constants = [&](int seg) __attribute__((always_inline)) {
        const int64_t pb = ((int64_t)seg * a.nhkv + h) * D + 4 * cg;
        const float4 kmid = *reinterpret_cast<const float4*>(a.kmid + pb), kstep = *reinterpret_cast<const float4*>(a.kstep + pb);
        const float4 vmid = *reinterpret_cast<const float4*>(a.vmid + pb), vstep = *reinterpret_cast<const float4*>(a.vstep + pb);
        kc = a.kc[seg * a.nhkv + h]; vc = a.vc[seg * a.nhkv + h];
        km[0] = kmid.x; km[1] = kmid.y; km[2] = kmid.z; km[3] = kmid.w;
        ks_[0] = kstep.x; ks_[1] = kstep.y; ks_[2] = kstep.z; ks_[3] = kstep.w;
        vm[0] = vmid.x; vm[1] = vmid.y; vm[2] = vmid.z; vm[3] = vmid.w;
        vs_[0] = vstep.x; vs_[1] = vstep.y; vs_[2] = vstep.z; vs_[3] = vstep.w;
        cur_seg = seg;
    };
    // One tile: restore the ids of register set (rk, rv) into LDS, refill the set with tile t + 2, S, softmax, O.
    auto tile = [&](int t, U (&rk)[UNITS][4], U (&rv)[UNITS][4], TileRef& ref) {
        const int start = ref.start, nlen = ref.ok ? ref.nlen : 0, seg = ref.seg;      // a tile that is not wanted: no key counts
        if (seg != cur_seg) {
            // A new segment (every few thousand keys).  The wait stands INSIDE the branch: the requests of the next tiles' ids are
            // older than these, and a wait placed where the constants are first used would hold every tile until its successors'
            // ids had arrived.
            constants(seg);
            __builtin_amdgcn_s_waitcnt(0x0F70);               // vmcnt(0)
        }
        // Keys past the tile's length hold a copy of its last key: their scores are replaced by -inf before any use, so K
        // needs no blanking; their V must be zero (0 * inf would poison the sums), done on the packed halves.
        const bool whole = nlen == kKeys;
#pragma unroll
        for (int u = 0; u < UNITS; ++u) {
            const int kgp = kgp0 + KSTEP * u;
            uint2 vcell[4];
            float dv[4][4];                                         // [key j][channel c]: id - centre of V
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int key = 4 * kgp + j;
                float dk[4];
#pragma unroll
                for (int c = 0; c < 4; ++c) { dk[c] = QD::id(rk[u][j], c) - kc; dv[j][c] = QD::id(rv[u][j], c) - vc; }
                uint2 kv;
                kv.x = restore_pair(ks_[0], dk[0], km[0], ks_[1], dk[1], km[1]);
                kv.y = restore_pair(ks_[2], dk[2], km[2], ks_[3], dk[3], km[3]);
                *reinterpret_cast<uint2*>(Ks + key * KROW + 4 * cg) = kv;
            }
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                vcell[c].x = restore_pair(vs_[c], dv[0][c], vm[c], vs_[c], dv[1][c], vm[c]);
                vcell[c].y = restore_pair(vs_[c], dv[2][c], vm[c], vs_[c], dv[3][c], vm[c]);
            }
            if (!whole) {
                const uint32_t m0 = (4 * kgp + 0 < nlen ? 0x0000FFFFu : 0u) | (4 * kgp + 1 < nlen ? 0xFFFF0000u : 0u);
                const uint32_t m1 = (4 * kgp + 2 < nlen ? 0x0000FFFFu : 0u) | (4 * kgp + 3 < nlen ? 0xFFFF0000u : 0u);
#pragma unroll
                for (int c = 0; c < 4; ++c) { vcell[c].x &= m0; vcell[c].y &= m1; }
            }
#pragma unroll
            for (int c = 0; c < 4; ++c)
                *reinterpret_cast<uint2*>(Vt + (4 * cg + c) * kKeys + 4 * (kgp ^ (cg & 7))) = vcell[c];
        }
        __syncthreads();
        fetch(t + 2, rk, rv, ref);

        // ---- S = Q K^T: this wave's 16 keys, its half of the channels; a K operand serves every row block ----
        {
            f4_t sc[RB];
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) sc[rb] = f4_t{0.f, 0.f, 0.f, 0.f};
            const _Float16* kp = Ks + (16 * kf + n16) * KROW + dh * (D / 2) + 4 * kg;
            h4_t kb[NKS];                                         // all asked for before the first product
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) kb[ks] = *reinterpret_cast<const h4_t*>(kp + 16 * ks);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
                for (int rb = 0; rb < RB; ++rb) sc[rb] = __builtin_amdgcn_mfma_f32_16x16x16f16(qa[rb][ks], kb[ks], sc[rb], 0, 0, 0);
#pragma unroll
            for (int rb = 0; rb < RB; ++rb)
#pragma unroll
                for (int e = 0; e < 4; ++e) Ss[((2 * rb + dh) * kRows + 4 * kg + e) * kSStride + 16 * kf + n16] = sc[rb][e];
        }
        __syncthreads();

        // ---- softmax, once per workgroup: wave w takes rows 4 w .. 4 w + 3 of every block, sixteen lanes a row, two keys
        //      a lane; the probabilities (fp16) and the rows' rescale factors go to LDS for all four waves ----
        h4_t vb[2][NF];                                   // the second product's operands: here when the softmax is done
        {
            // every key of the tile counts for every row of the workgroup (rows past n_rows compute on zeros, never stored)
            const bool all_seen = nlen == kKeys && start + kKeys - 1 <= qmin;
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) {
                const int prow = rb * kRows + srow;                // row within the workgroup
                const bool srow_ok = row0 + prow < a.n_rows;
                const int sqpos = a.q_pos0 + (srow_ok ? (row0 + prow) / a.G : 0);
                const float2 sa = *reinterpret_cast<const float2*>(Ss + ((2 * rb) * kRows + srow) * kSStride + 2 * kpair);
                const float2 sb = *reinterpret_cast<const float2*>(Ss + ((2 * rb + 1) * kRows + srow) * kSStride + 2 * kpair);
                if (rb == 0) {
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
                        for (int f = 0; f < NF; ++f) {
                            const int ch = wave * (D / 4) + 16 * f + n16;
                            vb[kk][f] = *reinterpret_cast<const h4_t*>(Vt + ch * kKeys + 4 * ((4 * kk + kg) ^ ((ch >> 2) & 7)));
                        }
                    __builtin_amdgcn_sched_barrier(0);
                }
                const bool ok0 = all_seen || (srow_ok && 2 * kpair < nlen && start + 2 * kpair <= sqpos);
                const bool ok1 = all_seen || (srow_ok && 2 * kpair + 1 < nlen && start + 2 * kpair + 1 <= sqpos);
                const float sv0 = ok0 ? (sa.x + sb.x) * a.scale : -INFINITY, sv1 = ok1 ? (sa.y + sb.y) * a.scale : -INFINITY;
                const float mx = row_max16(fmaxf(sv0, sv1));
                const float m_new = fmaxf(m_run[rb], mx);
                const float m_safe = m_new == -INFINITY ? 0.f : m_new;
                const _Float16 p0 = (_Float16)(sv0 == -INFINITY ? 0.f : __expf(sv0 - m_safe));
                const _Float16 p1 = (_Float16)(sv1 == -INFINITY ? 0.f : __expf(sv1 - m_safe));
                const float sum = row_sum16((float)p0 + (float)p1);    // the rounded p, as the second product sees it
                const float alpha = m_run[rb] == -INFINITY ? 0.f : (m_new == m_run[rb] ? 1.f : __expf(m_run[rb] - m_safe));
                l_run[rb] = l_run[rb] * alpha + sum;
                m_run[rb] = m_new;
                typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
                *reinterpret_cast<h2_t*>(Ps + prow * kPStride + 2 * kpair) = h2_t{p0, p1};
                if (kpair == 0) Al[prow] = alpha;
            }
        }
        __syncthreads();
        // ---- O = alpha O + P V; the accumulator holds rows 4 kg + e of channel n16 of each fragment; a V operand serves
        //      every row block ----
        h4_t pa[RB][2];
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            pa[rb][0] = *reinterpret_cast<const h4_t*>(Ps + (rb * kRows + n16) * kPStride + 4 * kg);
            pa[rb][1] = *reinterpret_cast<const h4_t*>(Ps + (rb * kRows + n16) * kPStride + 16 + 4 * kg);
            const f4_t ae = *reinterpret_cast<const f4_t*>(Al + rb * kRows + 4 * kg);
            if (__builtin_amdgcn_ballot_w64(ae[0] != 1.f || ae[1] != 1.f || ae[2] != 1.f || ae[3] != 1.f)) {
#pragma unroll
                for (int f = 0; f < NF; ++f)
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[rb][f][e] *= ae[e];
            }
        }
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
            for (int f = 0; f < NF; ++f)
#pragma unroll
                for (int rb = 0; rb < RB; ++rb) acc[rb][f] = __builtin_amdgcn_mfma_f32_16x16x16f16(pa[rb][kk], vb[kk][f], acc[rb][f], 0, 0, 0);
        __syncthreads();                                  // the tile in LDS is free again
    };

    if (t0 < t1) {
        U rk0[UNITS][4], rv0[UNITS][4], rk1[UNITS][4], rv1[UNITS][4];
        TileRef ref0, ref1;
        fetch(t0, rk0, rv0, ref0);
        __builtin_amdgcn_sched_barrier(0);                 // set 0 is the older one, as in every later round of the loop
        fetch(t0 + 1, rk1, rv1, ref1);
        __builtin_amdgcn_sched_barrier(0);
        // queries and the first segment's constants travel with the first ids: one trip to memory where there were ten
        constants(ref0.seg);
        queries();
        // The loop has one way out, at its head, and takes tiles in pairs; when the last pair has no second tile, that
        // one is run as an empty tile (no key counts: nothing changes).  A way out of the middle would be turned into a
        // path through the loop's end back to its head, on which set 0 is the younger one, and the compiler would make
        // every round wait for both sets; a copy of the tile's code behind the loop costs registers that end in scratch.
        for (int t = t0; ref0.ok; t += 2) {
            tile(t, rk0, rv0, ref0);
            tile(t + 1, rk1, rv1, ref1);
        }
    }

    // Where the results go is worked out only now, from a thread index the compiler cannot connect with the one above:
    // otherwise it computes the addresses before the loop and, short of registers, parks them in scratch memory (measured:
    // 5.6 MB written and read back per launch).
    int tid_e = threadIdx.x;
    asm volatile("" : "+v"(tid_e));
    const int lane_e = tid_e & 63, wave_e = tid_e >> 6, n16_e = lane_e & 15, kg_e = lane_e >> 4;
    const int64_t base = ((int64_t)sp * a.nhkv + h) * a.n_rows;
    const int srow_e = 4 * wave_e + kg_e;                    // the row (of every block) whose softmax state this lane holds
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int r = row0 + rb * kRows + 4 * kg_e + e;
                if (r < a.n_rows) a.o[(base + r) * D + wave_e * (D / 4) + 16 * f + n16_e] = acc[rb][f][e];
            }
        const int r = row0 + rb * kRows + srow_e;
        if (n16_e == 0 && r < a.n_rows) {
            a.m[base + r] = m_run[rb];
            a.l[base + r] = l_run[rb];
        }
    }
}

// ---- many query rows (a prompt chunk, a wide draft): 128 or 256 rows per workgroup -----------------------------------------
// With hundreds of rows the products bound the work, and what has to be shared is the restored tile: 4 or 8 waves x 32 query
// rows share one, in two LDS buffers (tile t is multiplied while tile t + 1 is restored; one barrier per tile).  The
// products run transposed, S^T = K Q^T and O^T = V^T P^T on v_mfma_f32_32x32x16_f16: a lane then holds the scores of ONE
// query (column lane % 32), so
//   * the softmax needs one exchange between the two halves of the wave and no LDS: a lane's sixteen scores per tile are
//     its own, its running maximum and sum are scalars of the lane, and rescaling O is a multiply by a lane's own factor;
//   * with K's rows read in the order `swap bits 2 and 3`, the scores a lane holds are of eight consecutive keys per half
//     and 16-key step, which is the B operand of the second product as it stands: P never leaves the registers.
// Q stays in registers (B operands), V is restored as [channel % 4][channel / 4][key]: a thread's four channels then lie a
// plane apart and its 16-byte stores, 80 bytes from lane to lane, meet no bank twice; the operand reads are 80 bytes apart too.
// O is rescaled whenever a row's maximum rises, as in the row-block kernel: p is then rounded to fp16 with the row's largest at
// 1, and the keys that matter most lie just below it, where fp16 is finest for their size.  (A reference that lags behind
// the maximum by up to 2^8 saves the multiplications but puts them anywhere in their binade: 1 .. 2.5 % more error against
// 64 bits over 33 .. 1024 rows.)
// Two workgroups of four waves per CU (78 KB of LDS, at most 256 registers): one restores while the other one's products run.  One of
// eight waves restores half as much per wave; its waves run apart by what the barrier allows.
// Bound by what a CU issues beside its products (restoring, exp2, conversions): 720 rows x 4 kv heads over 16001 keys of 256
// channels, whole calls: 107.2 us with four waves and the scale multiplied before the maximum is taken, 100.0 with eight, 98.5 with
// the scale in the exponent's subtraction and the products first.  (Half of the eight waves at their products while the others restore,
// by program order: 103.)  The ids of tile t + 2 are asked for between the two products where both sets of registers would not fit
// (before the first one they are spilled away from Q); with 128 channels and eight waves before them: 960 rows 76.6 against
// 78.5.
constexpr int kWaveRows = 32;
constexpr int kWideFrom = 33;                                 // fewest rows that take it: fused_attn.py has the measurements
constexpr int kVRow = kKeys + 8;                              // halfs per row of V in LDS
typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
typedef float f16_t __attribute__((ext_vector_type(16)));
constexpr int krow_wide(int D) { return D + 8; }              // halfs per key of K in LDS
constexpr size_t wide_lds(int D) { return (size_t)2 * kKeys * krow_wide(D) * 2 + (size_t)2 * D * kVRow * 2 + (size_t)4 * D * 4; }
constexpr float kLog2e = 1.4426950408889634f, kLn2 = 0.6931471805599453f;

// The lane's number, worked out anew where it is asked for: the addresses made from it then need no registers between their
// uses (kept across the loop they are spilled, and waiting for a spilled one also waits for the ids in flight).
__device__ __forceinline__ int lane_now() {
    int l;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
    return l;
}

template <int D, typename T, int NW>
__global__ __launch_bounds__(64 * NW, (D == 256 && sizeof(T) == 2) ? 1 : 2) void attn_wide_kernel(const AttnArgs a) {
    constexpr int CG = D / 4;                  // channel groups (four channels each) of a key
    constexpr int kWideRows = NW * kWaveRows;
    constexpr bool kAskEarly = D == 128 && NW == 8;           // the ids of tile t + 2 before the products of tile t, where registers allow it
    // operands of a product on their way from LDS, as many as registers hold without a spill (one at a time: 720 rows x 4 heads over
    // 16001 keys 98.9 .. 99.9 us a call, 95.3 .. 97.6 this way)
    constexpr int kAhead = NW == 8 ? 6 : 4;
    constexpr int KPT = kKeys * CG / (64 * NW);               // consecutive keys a thread restores: 32 (D = 256) or 16 over the waves
    constexpr int KROW = krow_wide(D), NKS = D / 16, NF = D / 32, NFC = NF / 4;
    using QD = Quad<T>;
    using U = typename QD::type;
    extern __shared__ __align__(16) unsigned char smem[];
    _Float16* const Ks = reinterpret_cast<_Float16*>(smem);                     // [2][kKeys][KROW]
    _Float16* const Vt = Ks + 2 * kKeys * KROW;                                 // [2][4][CG][kVRow]
    float* const Cs = reinterpret_cast<float*>(Vt + 2 * D * kVRow);             // [4][D]: kmid, kstep, vmid, vstep of the segment

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n32 = lane & 31, hf = lane >> 5;
    // Workgroups go to the XCDs in turn.  The row blocks of one (head, split) read the same ids: where the pairs divide by
    // eight, a pair's row blocks go to one XCD one after the other and its L2 serves all but the first.
    int h = blockIdx.x, sp = blockIdx.y, z = blockIdx.z;
    {
        const int nx = gridDim.x, nz = gridDim.z, pairs = nx * (int)gridDim.y;
        if (nz > 1 && (pairs & 7) == 0) {
            const int flat = h + nx * (sp + (int)gridDim.y * z), k = flat >> 3;
            const int pair = (k / nz) * 8 + (flat & 7);
            z = k % nz; h = pair % nx; sp = pair / nx;
        }
    }
    const int row0 = z * kWideRows, wrow0 = row0 + wave * kWaveRows, myrow = wrow0 + n32;
    const int per_wave = 64 / CG;                             // key groups a wave restores: 1 (D = 256) or 2
    const bool row_ok = myrow < a.n_rows;
    const bool wave_ok = wrow0 < a.n_rows;                                      // uniform

    h8_t qb[NKS];
    {
        const int rr = row_ok ? myrow : 0;
        const uint16_t* qp = reinterpret_cast<const uint16_t*>(a.q) + (int64_t)(rr / a.G) * a.sq_r + (int64_t)(h * a.G + rr % a.G) * a.sq_h + 8 * hf;
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) {
            const h4_t lo = *reinterpret_cast<const h4_t*>(qp + 16 * ks), hi = *reinterpret_cast<const h4_t*>(qp + 16 * ks + 4);
            const h8_t v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            qb[ks] = row_ok ? v : h8_t{0, 0, 0, 0, 0, 0, 0, 0};
        }
    }
    const int qpos = a.q_pos0 + (row_ok ? myrow / a.G : 0);
    const int wqmin = a.q_pos0 + wrow0 / a.G;                                   // of the wave's rows: first position,
    const int wqmax = a.q_pos0 + (min(wrow0 + kWaveRows, a.n_rows) - 1) / a.G;  // last
    const int qmax = a.q_pos0 + (min(row0 + kWideRows, a.n_rows) - 1) / a.G;    // last position any row of the workgroup sees

    const int t0 = (int)min((int64_t)sp * a.tps, (int64_t)a.n_tiles), t1 = (int)min((int64_t)t0 + a.tps, (int64_t)a.n_tiles);
    const uint32_t key_stride = (uint32_t)a.s_n * (uint32_t)sizeof(T);
    const unsigned char* const kbytes = reinterpret_cast<const unsigned char*>(reinterpret_cast<const T*>(a.ki) + (int64_t)h * a.s_h);
    const unsigned char* const vbytes = reinterpret_cast<const unsigned char*>(reinterpret_cast<const T*>(a.vi) + (int64_t)h * a.s_h);
    U rk[KPT], rv[KPT];
    // ids of tile t; a tile that is not wanted (past the split's end or behind the last visible position) re-reads key 0
    auto fetch = [&](int t, TileRef& ref) __attribute__((always_inline)) {
        tile_entry(a.ts, a.tl, a.tseg, min(t, t1 - 1), ref);
        ref.ok = __builtin_amdgcn_readfirstlane((int)(t < t1 && ref.start <= qmax)) != 0;
        const int start = ref.ok ? ref.start : 0, nlen = ref.ok ? ref.nlen : 1;
        const int64_t tile_byte = (int64_t)start * a.s_n * (int64_t)sizeof(T);
        const uint32_t last_off = (uint32_t)max(nlen - 1, 0) * key_stride;
        const int ln = lane_now();
        const uint32_t cg_off = (uint32_t)(4 * (ln % CG)) * (uint32_t)sizeof(T), key_off0 = (uint32_t)((wave * per_wave + ln / CG) * KPT) * key_stride;
        const unsigned char* kb = kbytes + tile_byte;
        const unsigned char* vb = vbytes + tile_byte;
#pragma unroll
        for (int j = 0; j < KPT; ++j) {
            const uint32_t off = min(key_off0 + (uint32_t)j * key_stride, last_off) + cg_off;
            rk[j] = *reinterpret_cast<const U*>(kb + off);
            rv[j] = *reinterpret_cast<const U*>(vb + off);
        }
    };

    int cur_seg = -1;
    float kc = 0.f, vc = 0.f;
    // the ids in the registers -> keys and values of LDS buffer `buf`
    auto restore = [&](int buf, const TileRef& ref) __attribute__((always_inline)) {
        const int ln = lane_now(), cg = ln % CG, key0 = (wave * per_wave + ln / CG) * KPT;
        if (ref.seg != cur_seg) {
            // a new segment: its constants for this thread's channels.  Threads of the same channels write the same values,
            // all in the interval between two barriers in which this tile is restored; each reads back what it wrote.
            const int64_t pb = ((int64_t)ref.seg * a.nhkv + h) * D + 4 * cg;
            *reinterpret_cast<float4*>(Cs + 4 * cg) = *reinterpret_cast<const float4*>(a.kmid + pb);
            *reinterpret_cast<float4*>(Cs + D + 4 * cg) = *reinterpret_cast<const float4*>(a.kstep + pb);
            *reinterpret_cast<float4*>(Cs + 2 * D + 4 * cg) = *reinterpret_cast<const float4*>(a.vmid + pb);
            *reinterpret_cast<float4*>(Cs + 3 * D + 4 * cg) = *reinterpret_cast<const float4*>(a.vstep + pb);
            kc = a.kc[ref.seg * a.nhkv + h]; vc = a.vc[ref.seg * a.nhkv + h];
            cur_seg = ref.seg;
        }
        {
            const float4 mid = *reinterpret_cast<const float4*>(Cs + 4 * cg), st = *reinterpret_cast<const float4*>(Cs + D + 4 * cg);
#pragma unroll
            for (int j = 0; j < KPT; ++j) {
                uint2 kv;
                kv.x = restore_pair(st.x, QD::id(rk[j], 0) - kc, mid.x, st.y, QD::id(rk[j], 1) - kc, mid.y);
                kv.y = restore_pair(st.z, QD::id(rk[j], 2) - kc, mid.z, st.w, QD::id(rk[j], 3) - kc, mid.w);
                *reinterpret_cast<uint2*>(Ks + (buf * kKeys + key0 + j) * KROW + 4 * cg) = kv;
            }
        }
        const float4 mid4 = *reinterpret_cast<const float4*>(Cs + 2 * D + 4 * cg), st4 = *reinterpret_cast<const float4*>(Cs + 3 * D + 4 * cg);
        const float mid[4] = {mid4.x, mid4.y, mid4.z, mid4.w}, st[4] = {st4.x, st4.y, st4.z, st4.w};
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            uint32_t w[KPT / 2];
#pragma unroll
            for (int j = 0; j < KPT; j += 2) w[j / 2] = restore_pair(st[c], QD::id(rv[j], c) - vc, mid[c], st[c], QD::id(rv[j + 1], c) - vc, mid[c]);
            if (ref.nlen != kKeys) {                          // keys past the tile's length: zero (0 * inf would poison the sums)
#pragma unroll
                for (int j = 0; j < KPT; j += 2) w[j / 2] &= (key0 + j < ref.nlen ? 0x0000FFFFu : 0u) | (key0 + j + 1 < ref.nlen ? 0xFFFF0000u : 0u);
            }
            _Float16* dst = Vt + ((buf * 4 + c) * CG + cg) * kVRow + key0;
            if constexpr (KPT == 8) *reinterpret_cast<uint4*>(dst) = uint4{w[0], w[1], w[2], w[3]};
            else if constexpr (KPT == 4) *reinterpret_cast<uint2*>(dst) = uint2{w[0], w[1]};
            else *reinterpret_cast<uint32_t*>(dst) = w[0];
        }
    };
    static_assert(KPT == 8 || KPT == 4 || KPT == 2);

    float m_run = -INFINITY, l_run = 0.f;                    // m: in powers of two; l: this half's keys
    f16_t acc[NF];
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[f][i] = 0.f;
    const float to_log2 = a.scale * kLog2e;

    // register i of a lane: the score of key 16 (i / 8) + 8 hf + i % 8
    auto scores = [&](int buf, const TileRef& ref, h8_t (&p)[2]) __attribute__((always_inline)) {
        f16_t s;
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = 0.f;
        const int ln = lane_now(), half8 = 8 * (ln >> 5);
        const int key = (ln & 19) | ((ln & 4) << 1) | ((ln & 8) >> 1);                   // A row ln % 32 of S^T is this key of the tile
        const _Float16* const ka = Ks + (buf * kKeys + key) * KROW + half8;
        h8_t k[kAhead];
#pragma unroll
        for (int i = 0; i < kAhead; ++i) k[i] = *reinterpret_cast<const h8_t*>(ka + 16 * i);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) {
            s = __builtin_amdgcn_mfma_f32_32x32x16_f16(k[ks % kAhead], qb[ks], s, 0, 0, 0);
            if (ks + kAhead < NKS) k[ks % kAhead] = *reinterpret_cast<const h8_t*>(ka + 16 * (ks + kAhead));
            __builtin_amdgcn_sched_barrier(0);
        }
        float times = to_log2;                                // > 0: multiplied in the exponent's subtraction, below
        if (!(times > 0.f)) {
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] *= times;
            times = 1.f;
        }
        if (!(ref.nlen == kKeys && ref.start + kKeys - 1 <= wqmin)) {
            const int seen = row_ok ? min(ref.nlen, qpos - ref.start + 1) - half8 : 0;      // keys of the tile this row sees
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] = 16 * (i >> 3) + (i & 7) < seen ? s[i] : -INFINITY;
        }
        float mx = s[0];
#pragma unroll
        for (int i = 1; i < 16; ++i) mx = fmaxf(mx, s[i]);
        mx = fmaxf(mx, __shfl_xor(mx, 32)) * times;
        const bool rises = mx > m_run;                        // also the first visible key: m_run is -inf
        if (__builtin_amdgcn_ballot_w64(rises)) {
            const float alpha = rises ? (m_run == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_run - mx)) : 1.f;
            m_run = rises ? mx : m_run;
            l_run *= alpha;
#pragma unroll
            for (int f = 0; f < NF; ++f)
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[f][i] *= alpha;
        }
        const float m_safe = m_run == -INFINITY ? 0.f : m_run;
#pragma unroll
        for (int i = 0; i < 16; i += 2) {
            const h2_t pp = {(_Float16)__builtin_amdgcn_exp2f(__builtin_fmaf(s[i], times, -m_safe)), (_Float16)__builtin_amdgcn_exp2f(__builtin_fmaf(s[i + 1], times, -m_safe))};
            l_run = __builtin_amdgcn_fdot2(pp, h2_t{(_Float16)1.f, (_Float16)1.f}, l_run, false);    // the rounded p, as the product sees it
            p[i >> 3][i & 7] = pp[0];
            p[i >> 3][(i & 7) + 1] = pp[1];
        }
    };
    auto values = [&](int buf, const h8_t (&p)[2]) __attribute__((always_inline)) {
        const int ln = lane_now();
        const _Float16* const va = Vt + (buf * D + (ln & 31)) * kVRow + 8 * (ln >> 5);
        auto operand = [&](int i) __attribute__((always_inline)) { return *reinterpret_cast<const h8_t*>(va + 32 * (i % NF) * kVRow + 16 * (i / NF)); };
        h8_t v[kAhead];
#pragma unroll
        for (int i = 0; i < kAhead; ++i) v[i] = operand(i);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 2 * NF; ++i) {
            acc[i % NF] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v[i % kAhead], p[i / NF], acc[i % NF], 0, 0, 0);
            if (i + kAhead < 2 * NF) v[i % kAhead] = operand(i + kAhead);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    if (t0 < t1) {
        TileRef cur, next;
        fetch(t0, cur);
        if (cur.ok) restore(0, cur);
        fetch(t0 + 1, next);
        __syncthreads();
        int buf = 0;
        for (int t = t0; cur.ok; ++t) {
            const TileRef now = cur;
            cur = next;
            if (cur.ok) restore(buf ^ 1, cur);
            if (kAskEarly) { fetch(t + 2, next); __builtin_amdgcn_sched_barrier(0); }
            const bool mine = wave_ok && now.start <= wqmax;
            h8_t p[2] = {};
            __builtin_amdgcn_s_setprio(1);                    // the wave at its products goes first, the one that restores fills in
            if (mine) scores(buf, now, p);
            if (!kAskEarly) fetch(t + 2, next);
            __builtin_amdgcn_sched_barrier(0);
            if (mine) values(buf, p);
            __builtin_amdgcn_s_setprio(0);
            __syncthreads();                                  // buffer buf ^ 1 is filled, buffer buf is free
            buf ^= 1;
        }
    }
    if (!row_ok) return;
    // register i of fragment c NFC + fi: channel 4 (32 fi + 8 (i / 4) + 4 hf + i % 4) + c of the lane's row
    const int ln = lane_now(), hf_e = ln >> 5;
    const int64_t at = ((int64_t)sp * a.nhkv + h) * a.n_rows + wrow0 + (ln & 31);
#pragma unroll
    for (int fi = 0; fi < NFC; ++fi)
#pragma unroll
        for (int i = 0; i < 16; ++i)
            *reinterpret_cast<float4*>(a.o + at * D + 4 * (32 * fi + 8 * (i >> 2) + 4 * hf_e + (i & 3))) =
                make_float4(acc[fi][i], acc[NFC + fi][i], acc[2 * NFC + fi][i], acc[3 * NFC + fi][i]);
    const float l = l_run + __shfl_xor(l_run, 32);
    if (hf_e == 0) {
        a.m[at] = m_run == -INFINITY ? -INFINITY : m_run * kLn2;
        a.l[at] = l;
    }
}

// Splits -> the normalised result and the log-sum-exp.  A unit of W waves takes one (kv head, row, 16 channels): 16 W groups of 4
// threads share the splits (group g takes splits g, g + 16 W, ...), a thread holds four channels.  A thread asks for everything of
// its next splits at once and weighs them against their own largest maximum; the groups of a wave then join by lane exchanges and
// the waves through LDS, each join weighing both sides against the larger maximum, all in a fixed order: one trip to memory, at most
// one barrier.
struct Joined { float top, total; f4_t acc; };
__device__ __forceinline__ void join(Joined& a, float top, float total, const f4_t& acc) {
    const float t = fmaxf(a.top, top), safe = t == -INFINITY ? 0.f : t;
    const float wa = expf(a.top - safe), wb = expf(top - safe);
    a.total = a.total * wa + total * wb;
    a.acc = a.acc * wa + acc * wb;
    a.top = t;
}
// K splits of the group, `step` apart, from s0 on (those past the end count nothing)
template <int K>
__device__ __forceinline__ void join_splits(Joined& j, const float* o, const float* m, const float* l, int s0, int step, int n_splits,
                                            int64_t stride, int64_t hr, int D, int ch) {
    float mv[K], lv[K];
    f4_t ov[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int64_t at = min(s0 + step * k, n_splits - 1) * stride + hr;
        mv[k] = m[at];
        lv[k] = l ? l[at] : 1.f;
        ov[k] = *reinterpret_cast<const f4_t*>(o + at * D + ch);
    }
    float top = -INFINITY;
#pragma unroll
    for (int k = 0; k < K; ++k) { if (s0 + step * k >= n_splits) mv[k] = -INFINITY; top = fmaxf(top, mv[k]); }
    const float safe = top == -INFINITY ? 0.f : top;
    float total = 0.f;
    f4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const float w = expf(mv[k] - safe);
        if (s0 + step * k < n_splits) { total += lv[k] * w; acc += ov[k] * w; }
    }
    join(j, top, total, acc);
}
__device__ __forceinline__ void store_joined(const Joined& j, int64_t hr, int n_rows, int nhkv, int G, int D, int ch, float* out, float* lse) {
    const int h = (int)(hr / n_rows), r = (int)(hr - (int64_t)h * n_rows);
    const int64_t dst = (int64_t)(r / G) * (nhkv * G) + h * G + r % G;
    *reinterpret_cast<f4_t*>(out + dst * D + ch) = j.acc * (1.f / fmaxf(j.total, 1e-30f));
    if (ch == 0) lse[dst] = j.total > 0.f ? j.top + logf(fmaxf(j.total, 1e-30f)) : -INFINITY;
}
template <int W>
__global__ __launch_bounds__(256) void attn_combine_kernel(const float* __restrict__ o, const float* __restrict__ m, const float* __restrict__ l,
                                                            int n_splits, int nhkv, int n_rows, int D, int G,
                                                            float* __restrict__ out, float* __restrict__ lse) {
    constexpr int kGroups = 16 * W;
    __shared__ float s_top[4], s_total[4];
    __shared__ __align__(16) f4_t s_acc[4][4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int grp = (int)(threadIdx.x >> 2) % kGroups, cl = threadIdx.x & 3, ch = blockIdx.y * 16 + cl * 4, chc = min(ch, D - 4);
    const int64_t stride = (int64_t)nhkv * n_rows, unit = (int64_t)blockIdx.x * (4 / W) + wave / W, hr = min(unit, stride - 1);
    Joined j = {-INFINITY, 0.f, {0.f, 0.f, 0.f, 0.f}};
    if (W > 1 && n_splits <= kGroups) join_splits<1>(j, o, m, l, grp, kGroups, n_splits, stride, hr, D, chc);
    else for (int s0 = grp; s0 < n_splits; s0 += 4 * kGroups) join_splits<4>(j, o, m, l, s0, kGroups, n_splits, stride, hr, D, chc);
#pragma unroll
    for (int d = 4; d < 64; d <<= 1) {
        f4_t acc;
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[c] = __shfl_xor(j.acc[c], d);
        const float top = __shfl_xor(j.top, d), total = __shfl_xor(j.total, d);
        join(j, top, total, acc);
    }
    if constexpr (W > 1) {
        if (lane == 0) { s_top[wave] = j.top; s_total[wave] = j.total; }
        if (lane < 4) s_acc[wave][cl] = j.acc;
        __syncthreads();
        if (wave > 0) return;
#pragma unroll
        for (int w = 1; w < 4; ++w) join(j, s_top[w], s_total[w], s_acc[w][cl]);
    }
    if (lane < 4 && unit < stride && ch < D) store_joined(j, hr, n_rows, nhkv, G, D, ch, out, lse);
}

// The same with no exchange: a thread holds four channels of one row and takes the splits in ascending order, eight at a time.
__global__ __launch_bounds__(256) void attn_combine_rows_kernel(const float* __restrict__ o, const float* __restrict__ m, const float* __restrict__ l,
                                                                int n_splits, int nhkv, int n_rows, int D, int G,
                                                                float* __restrict__ out, float* __restrict__ lse) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x, stride = (int64_t)nhkv * n_rows;
    const int per_row = D / 4;
    const int64_t hr = i / per_row;
    if (hr >= stride) return;
    const int ch = (int)(i - hr * per_row) * 4;
    Joined j = {-INFINITY, 0.f, {0.f, 0.f, 0.f, 0.f}};
    for (int s = 0; s < n_splits; s += 8) join_splits<8>(j, o, m, l, s, 1, n_splits, stride, hr, D, ch);
    store_joined(j, hr, n_rows, nhkv, G, D, ch, out, lse);
}

// Eight waves where at least 13/16 of their rows are used, and where workgroups of four waves would have to share CUs.  Whole calls in us,
// four waves / eight, 4 kv heads: 256 channels, 720 rows (94 % used) over 16001 keys 107.2 / 98.5, 240 (94 %) over 65536 137.0 / 123.0, 1104
// (86 %) 145.5 / 138.9; 600 (78 %) 98.0 / 95.8 but 808 (79 %) 119.5 / 122.4, 288 (56 %) 78.2 / 83.0; 128 channels, 960 rows (94 %) over
// 16001 keys 86.9 / 76.6, 1024 (100 %) over 40000 171.4 / 149.7, 630 (82 %) over 30000 96.5 / 94.7.  Few workgroups: 2048 rows x 2
// heads over 2048 keys (256 of four waves) 48.4 / 51.5, 256 rows over 5000 keys (184) 47.3 / 48.9.  16-bit ids stay with four waves.
// The only place of this rule: kv/fused_attn.py asks it (qvb8_attn_rows_per_workgroup) for the splits it plans.
bool eight_waves(int64_t rows, int64_t heads_and_splits, int id_bytes, int64_t cus) {
    return id_bytes == 1 && 16 * rows >= 13 * 256 * ((rows + 255) / 256) && heads_and_splits * ((rows + 127) / 128) > cus;
}

template <int D, typename T, int NW>
int launch_attn_wide(const AttnArgs& a, int64_t n_splits, hipStream_t s) {
    if (int rc = host::raise_lds_limit<attn_wide_kernel<D, T, NW>>(wide_lds(D), "qvb8_attn_fwd")) return rc;
    const dim3 grid((unsigned)a.nhkv, (unsigned)n_splits, (unsigned)((a.n_rows + NW * kWaveRows - 1) / (NW * kWaveRows)));
    hipLaunchKernelGGL((attn_wide_kernel<D, T, NW>), grid, dim3(64 * NW), wide_lds(D), s, a);
    return host::check_launch("qvb8_attn_fwd");
}

template <int D, typename T>
int launch_attn(const AttnArgs& a, int64_t n_splits, hipStream_t s) {
    // up to 16 rows: one block per workgroup; up to 32: two; beyond: the kernel of 128 or 256 rows.  QVB8_ATTN_ROW_BLOCKS forces this
    // kernel with 1, 2 or 4 blocks (256 channels: at most 2, four blocks' accumulators and Q do not fit the registers).
    int rb = a.n_rows <= kRows ? 1 : a.n_rows <= 2 * kRows ? 2 : 4;
    const int forced = host::env_int("QVB8_ATTN_ROW_BLOCKS", 0);
    if (forced == 0 && a.n_rows >= kWideFrom) {
        if constexpr (sizeof(T) == 1) if (eight_waves(a.n_rows, n_splits * a.nhkv, 1, host::device_cus())) return launch_attn_wide<D, T, 8>(a, n_splits, s);
        return launch_attn_wide<D, T, 4>(a, n_splits, s);
    }
    if (forced == 1 || forced == 2 || forced == 4) rb = forced;
    if (D == 256 && rb > 2) rb = 2;
    const dim3 grid((unsigned)a.nhkv, (unsigned)n_splits, (unsigned)((a.n_rows + rb * kRows - 1) / (rb * kRows)));
    if (grid.z > 65535u) return host::fail(-1, "qvb8_attn_fwd: %d rows are more than one launch takes", a.n_rows);
    if (rb == 1) hipLaunchKernelGGL((attn_kernel<D, T, 1>), grid, dim3(kAttnThreads), 0, s, a);
    else if (rb == 2) hipLaunchKernelGGL((attn_kernel<D, T, 2>), grid, dim3(kAttnThreads), 0, s, a);
    else if constexpr (D == 128) hipLaunchKernelGGL((attn_kernel<D, T, 4>), grid, dim3(kAttnThreads), 0, s, a);
    return host::check_launch("qvb8_attn_fwd");
}

bool aligned(const void* p, uintptr_t n) { return (reinterpret_cast<uintptr_t>(p) & (n - 1)) == 0; }

}  // namespace
}  // namespace qvb8

namespace {
// q_dt: qvb8::kQReady, or the type of queries that still have to be prepared with q_scale
int attn_forward(const void* q, int q_dt, float q_scale, int64_t sq_r, int64_t sq_h, const void* ki, const void* vi, int id_bytes,
                 int64_t s_n, int64_t s_h, const float* kmid, const float* kstep, const float* vmid,
                 const float* vstep, const float* kc, const float* vc, const int32_t* ts, const int32_t* tl,
                 const int32_t* tseg, int64_t n_tiles, float* o, float* m, float* l, int64_t n_splits,
                 int64_t n_rows, int64_t n_kv_heads, int64_t head_dim, int64_t q_pos0, int64_t tps,
                 double scale, int64_t G, const char* who, void* stream) {
    using namespace qvb8;
    if (head_dim != 128 && head_dim != 256) return host::fail(-1, "%s: head_dim must be 128 or 256, got %lld", who, (long long)head_dim);
    if (id_bytes != 1 && id_bytes != 2) return host::fail(-1, "%s: ids are 1 or 2 bytes wide, got %d", who, id_bytes);
    if (n_rows < 0 || n_tiles < 0 || n_splits < 1 || tps < 1 || G < 1 || n_kv_heads < 1)
        return host::fail(-1, "%s: negative or zero size (rows %lld, tiles %lld, splits %lld, tiles per split %lld, G %lld, kv heads %lld)",
                          who, (long long)n_rows, (long long)n_tiles, (long long)n_splits, (long long)tps, (long long)G, (long long)n_kv_heads);
    if (n_rows % G != 0) return host::fail(-1, "%s: %lld rows are not whole tokens of %lld heads", who, (long long)n_rows, (long long)G);
    if (n_splits * tps < n_tiles) return host::fail(-1, "%s: %lld splits of %lld tiles do not cover %lld tiles", who, (long long)n_splits, (long long)tps, (long long)n_tiles);
    if (n_rows == 0) return 0;
    if (!q || !o || !m || !l) return host::fail(-1, "%s: null q / o / m / l", who);
    if (n_tiles > 0 && (!ki || !vi || !kmid || !kstep || !vmid || !vstep || !kc || !vc || !ts || !tl || !tseg))
        return host::fail(-1, "%s: null ids, constants or tile table", who);
    if (!aligned(q, q_dt == QVB8_F32 ? 16 : 8) || (sq_r & 3) || (sq_h & 3))
        return host::fail(-1, "%s: q must be aligned to four elements with strides that are multiples of 4", who);
    if (n_tiles > 0) {
        if (!aligned(ki, 4 * id_bytes) || !aligned(vi, 4 * id_bytes) || (s_n & 3) || (s_h & 3))
            return host::fail(-1, "%s: ids must be aligned to four ids with strides that are multiples of 4", who);
        if (!aligned(kmid, 16) || !aligned(kstep, 16) || !aligned(vmid, 16) || !aligned(vstep, 16))
            return host::fail(-1, "%s: the per-channel constants must be 16-byte aligned", who);
    }
    if (n_tiles > 0 && (s_n < 0 || s_n * 32 * id_bytes > INT32_MAX)) return host::fail(-1, "%s: key stride %lld out of range", who, (long long)s_n);
    const int64_t row_blocks = (n_rows + kRows - 1) / kRows;
    if (n_splits > 65535 || row_blocks > 65535 || n_tiles > INT32_MAX || n_rows > INT32_MAX || q_pos0 > INT32_MAX / 2 || q_pos0 < INT32_MIN / 2)
        return host::fail(-1, "%s: size beyond what one launch takes", who);
    AttnArgs a;
    a.q = q; a.q_dt = q_dt; a.q_scale = q_scale; a.sq_r = sq_r; a.sq_h = sq_h;
    a.ki = ki; a.vi = vi; a.s_n = s_n; a.s_h = s_h;
    a.kmid = kmid; a.kstep = kstep; a.vmid = vmid; a.vstep = vstep; a.kc = kc; a.vc = vc;
    a.ts = ts; a.tl = tl; a.tseg = tseg; a.o = o; a.m = m; a.l = l;
    a.q_pos0 = (int)q_pos0; a.n_tiles = (int)n_tiles; a.tps = (int)std::min<int64_t>(INT32_MAX / 2, tps); a.n_rows = (int)n_rows;
    a.G = (int)G; a.nhkv = (int)n_kv_heads; a.scale = (float)scale;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (head_dim == 256) return id_bytes == 1 ? launch_attn<256, uint8_t>(a, n_splits, s) : launch_attn<256, uint16_t>(a, n_splits, s);
    return id_bytes == 1 ? launch_attn<128, uint8_t>(a, n_splits, s) : launch_attn<128, uint16_t>(a, n_splits, s);
}
}  // namespace

extern "C" int qvb8_attn_fwd(const void* q, int64_t sq_r, int64_t sq_h, const void* ki, const void* vi, int id_bytes,
                             int64_t s_n, int64_t s_h, const float* kmid, const float* kstep, const float* vmid,
                             const float* vstep, const float* kc, const float* vc, const int32_t* ts, const int32_t* tl,
                             const int32_t* tseg, int64_t n_tiles, float* o, float* m, float* l, int64_t n_splits,
                             int64_t n_rows, int64_t n_kv_heads, int64_t head_dim, int64_t q_pos0, int64_t tps,
                             double scale, int64_t G, void* stream) {
    return attn_forward(q, qvb8::kQReady, 1.f, sq_r, sq_h, ki, vi, id_bytes, s_n, s_h, kmid, kstep, vmid, vstep, kc, vc, ts, tl, tseg,
                        n_tiles, o, m, l, n_splits, n_rows, n_kv_heads, head_dim, q_pos0, tps, scale, G, "qvb8_attn_fwd", stream);
}

extern "C" int64_t qvb8_attn_rows_per_workgroup(int64_t n_rows, int64_t n_splits, int64_t n_kv_heads, int id_bytes, int64_t cus) {
    if (n_rows < qvb8::kWideFrom || n_splits < 1 || n_kv_heads < 1) return 0;
    return qvb8::eight_waves(n_rows, n_splits * n_kv_heads, id_bytes, cus) ? 256 : 128;
}

extern "C" int64_t qvb8_attn_workspace_bytes(int64_t n_splits, int64_t n_kv_heads, int64_t n_rows, int64_t head_dim) {
    if (n_splits <= 0 || n_kv_heads <= 0 || n_rows <= 0 || head_dim <= 0) return 0;
    return 4 * n_splits * n_kv_heads * n_rows * (head_dim + 2) + (n_rows >= qvb8::kWideFrom ? 16 + 2 * n_kv_heads * n_rows * head_dim : 0);
}

extern "C" int qvb8_attend(const void* q, int q_dtype, double q_scale, int64_t sq_r, int64_t sq_h, const void* ki, const void* vi, int id_bytes,
                           int64_t s_n, int64_t s_h, const float* kmid, const float* kstep, const float* vmid,
                           const float* vstep, const float* kc, const float* vc, const int32_t* ts, const int32_t* tl,
                           const int32_t* tseg, int64_t n_tiles, int64_t n_splits, int64_t n_rows, int64_t n_kv_heads,
                           int64_t head_dim, int64_t q_pos0, int64_t tps, int64_t G, float* out, float* lse, void* workspace,
                           int64_t workspace_bytes, void* stream) {
    using namespace qvb8;
    const char* who = "qvb8_attend";
    if (q_dtype < QVB8_F32 || q_dtype > QVB8_BF16) return host::fail(QVB8_ERR_ARG, "%s: unknown query type %d", who, q_dtype);
    // ahead of the first launch: the workspace is laid out by these, and as many queries are read as they say
    if (n_rows < 0 || n_splits < 1 || G < 1 || n_kv_heads < 1 || head_dim < 1 || n_rows % G != 0)
        return host::fail(QVB8_ERR_ARG, "%s: bad size (rows %lld, splits %lld, G %lld, kv heads %lld, head_dim %lld)", who, (long long)n_rows, (long long)n_splits,
                          (long long)G, (long long)n_kv_heads, (long long)head_dim);
    const int64_t need = qvb8_attn_workspace_bytes(n_splits, n_kv_heads, n_rows, head_dim);
    if (need > 0 && (!workspace || workspace_bytes < need || !aligned(workspace, 16)))
        return host::fail(QVB8_ERR_WORKSPACE, "%s: needs %lld bytes of 16-byte aligned workspace", who, (long long)need);
    float* const o = static_cast<float*>(workspace);
    const int64_t rows = n_splits * n_kv_heads * n_rows;
    float* const m = o + rows * head_dim;
    if (n_rows >= kWideFrom && q) {
        // prepared once for all splits of the kernel of 128 or 256 rows
        if (sq_h != head_dim || sq_r != n_kv_heads * G * head_dim) return host::fail(QVB8_ERR_UNSUPPORTED, "%s: %d rows and more must be contiguous", who, kWideFrom);
        void* const q16 = reinterpret_cast<void*>((reinterpret_cast<uintptr_t>(m + 2 * rows) + 15) & ~(uintptr_t)15);
        if (int rc = qvb8_scale_sat_half(q, q_dtype, n_kv_heads * n_rows * head_dim, (float)q_scale, q16, stream)) return rc;
        q = q16;
        q_dtype = kQReady;
    }
    if (int rc = attn_forward(q, q_dtype, (float)q_scale, sq_r, sq_h, ki, vi, id_bytes, s_n, s_h, kmid, kstep, vmid, vstep, kc, vc, ts, tl, tseg,
                              n_tiles, o, m, m + rows, n_splits, n_rows, n_kv_heads, head_dim, q_pos0, tps, 1.0, G, who, stream)) return rc;
    return qvb8_attn_combine(o, m, m + rows, n_splits, n_kv_heads, n_rows, head_dim, G, out, lse, stream);
}

extern "C" int qvb8_attn_combine(const float* o, const float* m, const float* l, int64_t n_splits, int64_t n_kv_heads,
                                 int64_t n_rows, int64_t head_dim, int64_t G, float* out, float* lse, void* stream) {
    using namespace qvb8;
    const char* who = "qvb8_attn_combine";
    if (n_splits < 1 || n_kv_heads < 1 || n_rows < 0 || G < 1 || head_dim < 4 || head_dim % 4 != 0)
        return host::fail(-1, "%s: bad size (splits %lld, kv heads %lld, rows %lld, G %lld, head_dim %lld)", who, (long long)n_splits,
                          (long long)n_kv_heads, (long long)n_rows, (long long)G, (long long)head_dim);
    if (n_rows % G != 0) return host::fail(-1, "%s: %lld rows are not whole tokens of %lld heads", who, (long long)n_rows, (long long)G);
    if (n_rows == 0) return 0;
    if (!o || !m || !out || !lse) return host::fail(-1, "%s: null pointer", who);
    if (!aligned(o, 16) || !aligned(out, 16)) return host::fail(-1, "%s: o and out must be 16-byte aligned", who);
    if (n_kv_heads * n_rows > INT32_MAX || n_splits > INT32_MAX) return host::fail(-1, "%s: size beyond what one launch takes", who);
    const int64_t units = n_kv_heads * n_rows, quads = units * (head_dim / 4);
    const unsigned parts = (unsigned)((head_dim + 15) / 16);
    hipStream_t st = static_cast<hipStream_t>(stream);
#define QVB8_COMBINE_ARGS o, m, l, (int)n_splits, (int)n_kv_heads, (int)n_rows, (int)head_dim, (int)G, out, lse
    // Measured alone, partial results in the caches (us; a thread a quad / a wave / four waves a unit): 1536 quads from 8 splits
    // 3.0 / 3.5 / 3.7, from 171 26.5 / 6.1 / 4.6; 6144 from 8 3.1 / 3.6 / 5.3, from 24 5.0 / 4.3 / 5.4; 15360 from 24 5.1 / 5.2 / 9.2, from 64
    // 11.7 / 6.4 / 9.7; 30720 from 32 7.3 / 8.0 / 15.5, from 64 12.4 / 9.7 / 16.8; 46592 from 64 13.8 / 16.9 / 24.0.  Behind the attention
    // kernel, whole calls: 2304 quads from 299 splits 69 / 30.4 / 27.8, 6144 from 125 49 / 33.4 / 34.5, 7680 from 77 34.8 / 30.7 / 28.0, 9216 from
    // 94 40.1 / 35.4 / 31.6, 10240 from 79 34.6 / 27.0 / 29.2.  (Two passes over the splits and a walk over 64 groups' results, four waves a
    // unit up to 65536 quads: 6.5 us at 1536 quads from 171 splits, 19.7 at 46592 from 16.)
    if (quads >= 40960 || n_splits <= 8 + quads / 1024) {
        if (quads > (int64_t)INT32_MAX * 256) return host::fail(-1, "%s: size beyond what one launch takes", who);
        hipLaunchKernelGGL(attn_combine_rows_kernel, dim3((unsigned)((quads + 255) / 256)), dim3(256), 0, st, QVB8_COMBINE_ARGS);
    } else if (quads > 9216) hipLaunchKernelGGL(attn_combine_kernel<1>, dim3((unsigned)((units + 3) / 4), parts), dim3(256), 0, st, QVB8_COMBINE_ARGS);
    else hipLaunchKernelGGL(attn_combine_kernel<4>, dim3((unsigned)units, parts), dim3(256), 0, st, QVB8_COMBINE_ARGS);
#undef QVB8_COMBINE_ARGS
    return host::check_launch(who);
}
