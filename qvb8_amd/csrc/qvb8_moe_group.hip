// Routed MoE expert stack for many tokens (more than 16: draft trees, batches, prompt chunks), gfx950.
//
// The routing plan groups the (token, choice) pairs by expert.  A workgroup takes up to 64 pairs of ONE expert and eight
// waves' worth of its rows; every wave owns two 16-row tiles (the gate rows and the matching up rows, so that the
// activation is applied to the registers it ends up in; elsewhere two neighbouring tiles) over all columns.  The pairs'
// activations go through LDS a chunk of columns at a time, double buffered and shared by the eight waves; the ids go from
// memory into registers -- a step is requested as soon as the one before it has been decoded, 48 KB in flight per CU with
// two workgroups -- and are decoded there into the other operand of v_mfma_f32_16x16x32_f16.  So an
// expert's bytes are read once per 64 of its pairs, and every id is decoded once for all of them.
//
// Arithmetic: the operand of a weight is id - c, exact in fp16, c being the id nearest to a weight of zero (or the row's first or
// last id); what that leaves out returns with the row's constants:  y = tau_s * sum(x (id - c)) + (min_s + c tau_s) * sum(x), joined
// in double.  (The 16-row kernels multiply 1024 + id and take the bias off the sum; here the subtraction is one packed
// instruction per two ids in the shadow of the loads.)  The sums are then as small as their results, which decides their
// precision: a matrix instruction rounds its running sum more coarsely than an fp32 addition.  Up: x is narrowed like
// saturating_half.  Down: H arrives as fp32 and is used as fp16 hi + lo of H * 2^s, s per pair such that its largest |H| lies in
// [8192, 16384): 22 significant bits for values within 2^-16 of the pair's largest, an absolute 2^-38 of the largest below
// that (lo ends at fp16's 2^-24).
// Error of a call's fp32 results against 64 bits (17 .. 64 tokens, activations that fp16 holds): 2.3e-7 .. 3.3e-7 of their norm; the
// general path's fp32 products 5.4e-7 .. 6.9e-7; with c in the middle of the width instead, 1.0e-6 .. 1.4e-6.
//
// Measured (hidden 2048, 128 experts of 2 x 768 / 768 columns, top-8, bf16): a layer of 509 tokens 184 us, where one pass per
// expert over its own modules took 12.2 ms, nearly all of it launches; kernels alone, under the profiler, up 87, down 77, plan 13,
// combine 8.  With the rows back to back 210 us, up 109, down 89: a request then touches sixteen rows, and L1 was busy 59 % of the time
// with that.  In planes (PL) a request is one run and the tiles' places are scalar registers.  The up launch moves 300 MB at 3.4 TB/s; its
// first 512 workgroups, two a CU, run at 4.9 and the other 256 alone on their CUs.  A second step of ids on its way, operands of X
// a quarter of a step ahead, three workgroups a CU (80 registers) and non-temporal ids changed nothing or lost (88, 94, 121, 89 us).
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <algorithm>

#include "../../include/qvb8_amd.h"
#include "qvb8_device.h"
#include "qvb8_host.h"
#include "qvb8_mma_device.h"
#include "qvb8_moe_plan.h"

namespace qvb8 {

namespace {

constexpr int kGroupWaves = 8;
constexpr int kGroupThreads = 64 * kGroupWaves;

// LDS of a chunk: NT x 16 rows of CK columns; rows 16 bytes apart from a multiple of 256, so that the sixteen rows an
// operand read touches lie on different banks.  CK is what keeps two buffers under 70 KB (two workgroups per CU).
template <int NT, bool DOWN, int XDT> struct GroupTile {
    static constexpr int NTP = NT == 1 ? 1 : NT == 2 ? 2 : 4;
    static constexpr int TPR = 32 / NTP;                       // threads that stage one row
    static constexpr int CK = (XDT == QVB8_F32 ? 512 : 1024) / NTP;   // columns per chunk (fp32 arrives in twice the registers)
    static constexpr int CS = CK / kStepCols;                  // steps per chunk
    static constexpr int pitch = 2 * CK + 16;
    static constexpr int plane = 16 * NT * pitch;              // down: hi plane, then lo plane
    static constexpr int buf = DOWN ? 2 * plane : plane;
    static constexpr int pieces = CK / 8 / TPR;                // pieces of eight columns a thread stages per chunk
};
constexpr int kGroupBufBytes = 2 * 34816;                      // two buffers of the largest tile (NT = 4, down)
constexpr int kGroupLds = kGroupBufBytes + kGroupTokens * 12;

// every LDS access of the workgroup done, nothing said about its loads from memory (the ids stay in flight)
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// eight activations as they lie in memory: fp16 / bf16 bits (one 16-byte piece) or fp32 (two)
template <int XDT> struct Piece { v4u_t v[XDT == QVB8_F32 ? 2 : 1]; };
template <int XDT>
__device__ __forceinline__ Piece<XDT> load_piece(const void* row, int col) {
    Piece<XDT> p;
    const unsigned char* at = reinterpret_cast<const unsigned char*>(row) + (size_t)col * (XDT == QVB8_F32 ? 4 : 2);
    p.v[0] = *reinterpret_cast<const v4u_t*>(at);
    if constexpr (XDT == QVB8_F32) p.v[1] = *reinterpret_cast<const v4u_t*>(at + 16);
    return p;
}
__device__ __forceinline__ uint32_t pack_half2(_Float16 a, _Float16 b) {
    return (uint32_t)__builtin_bit_cast(uint16_t, a) | ((uint32_t)__builtin_bit_cast(uint16_t, b) << 16);
}
// (by value: a bit cast straight from a vector's element reads the vector's first element with this compiler)
__device__ __forceinline__ half2_t as_half2(uint32_t w) { return __builtin_bit_cast(half2_t, w); }
// ... as fp16 within its finite range (NaN kept); `keep_inf`: fp16 as it is
template <int XDT>
__device__ __forceinline__ v4u_t narrow_piece(const Piece<XDT>& p, bool keep_inf) {
    v4u_t o;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        if constexpr (XDT == QVB8_F16) {
            const half2_t top = {(_Float16)65504.0f, (_Float16)65504.0f}, h = as_half2(p.v[0][k]);
            o[k] = keep_inf ? p.v[0][k] : __builtin_bit_cast(uint32_t, (half2_t)__builtin_elementwise_maximum(__builtin_elementwise_minimum(h, top), -top));
        }
        else if constexpr (XDT == QVB8_BF16) o[k] = XIn<false, true>::pair(p.v[0][k]);
        else o[k] = sat_half_bits(__uint_as_float(p.v[k / 2][(2 * k) % 4])) | (sat_half_bits(__uint_as_float(p.v[k / 2][(2 * k + 1) % 4])) << 16);
    }
    return o;
}
__device__ __forceinline__ float sum_piece(const v4u_t& h, float s) {
    const half2_t one = {(_Float16)1.0f, (_Float16)1.0f};
#pragma unroll
    for (int k = 0; k < 4; ++k) s = __builtin_amdgcn_fdot2(as_half2(h[k]), one, s, false);
    return s;
}

// ids of one step -> operands id - c (negb = -(1024 + c) in both halves), width NB
template <int NB>
__device__ __forceinline__ void decode_centred(const uint4& lo, const uint4& hi, uint32_t negb, v4u_t (&b)[4]) {
    decode_slice<NB, false>(lo, hi, b);
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int k = 0; k < 4; ++k) b[j][k] = __builtin_bit_cast(uint32_t, (half2_t)(as_half2(b[j][k]) + as_half2(negb)));
}

// a row tile of the wave: what a lane needs for its row (r = lane % 16)
struct GroupRow {
    const uint8_t* base;           // in planes: the next step of the tile
    uint64_t at;                   // byte of the first four dwords of the lane's slice of the next step
    uint32_t tail, stride;         // from there to its last four dwords; to the next step
    uint32_t negb;
    int nb, centre, mode;          // width; the id taken off every id; the width all 16 rows share (0: they differ, or some are read id by id)
    bool sliced, ok;
};

template <int NT, bool DOWN, int XDT, bool PL>
__device__ __forceinline__ void moe_group_body(const MoeGroupArgs& a, unsigned char* smem, int e, int first, int n, int rb) {
    using L = GroupTile<NT, DOWN, XDT>;
    using F = Fmt<false>;
    float* s_sum = reinterpret_cast<float*>(smem + kGroupBufBytes);
    float* s_inv = s_sum + kGroupTokens;
    int* s_pair = reinterpret_cast<int*>(s_inv + kGroupTokens);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, kg = lane >> 4;
    const int n_steps = a.P / kStepCols;

    // ---- the wave's two row tiles ----
    const int v = rb * kGroupWaves + wave;                     // up, gated: 16 outputs; else two neighbouring tiles
    const bool paired = !DOWN && a.gated;
    const int n_tiles = (paired ? a.units : a.Q) / 16;         // tiles along one output dimension
    int row0[2];
    bool on[2];
    if (paired) { on[0] = on[1] = v < n_tiles; row0[0] = min(v, n_tiles - 1) * 16; row0[1] = row0[0] + a.units; }
    else {
#pragma unroll
        for (int t = 0; t < 2; ++t) { on[t] = 2 * v + t < n_tiles; row0[t] = min(2 * v + t, n_tiles - 1) * 16; }
    }
    const size_t row_at = (size_t)e * a.Q + r;
    GroupRow g[2];
    int64_t off[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        // in planes: one width, and the tile's first row says where it is
        const size_t at = PL ? (size_t)e * a.Q + row0[t] : row_at + row0[t];
        g[t].nb = a.nbits[at];
        off[t] = a.bit_off[at];
        if constexpr (PL) g[t].nb = __builtin_amdgcn_readfirstlane(g[t].nb);
    }
    // ---- the row this thread stages, its pair ----
    const int rho = tid / L::TPR, sub = tid % L::TPR;
    const bool stages = rho < 16 * NT;                         // (48 rows: a quarter of the threads has none)
    const int pair = a.plan.order[first + min(rho, n - 1)];
    if (sub == 0 && rho < kGroupTokens) s_pair[rho] = pair;
    const unsigned char* xrow = reinterpret_cast<const unsigned char*>(a.X) + (size_t)(DOWN ? pair : pair / a.topk) * a.P * (XDT == QVB8_F32 ? 4 : 2);

    Piece<XDT> px[L::pieces];
    auto request_x = [&](int chunk) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < L::pieces; ++i) px[i] = load_piece<XDT>(xrow, min(chunk * L::CK + (sub + i * L::TPR) * 8, a.P - 8));
    };
    float scale = 1.0f, xsum = 0.f;
    auto store_x = [&](int chunk) __attribute__((always_inline)) {
        unsigned char* to = smem + (chunk & 1) * L::buf + rho * L::pitch;
#pragma unroll
        for (int i = 0; i < L::pieces; ++i) {
            const int c = (sub + i * L::TPR) * 8;
            const bool in = stages && chunk * L::CK + c < a.P;
            if constexpr (DOWN) {
                v4u_t hi, lo;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const float f0 = __uint_as_float(px[i].v[k / 2][(2 * k) % 4]) * scale, f1 = __uint_as_float(px[i].v[k / 2][(2 * k + 1) % 4]) * scale;
                    const _Float16 h0 = (_Float16)f0, h1 = (_Float16)f1;
                    hi[k] = pack_half2(h0, h1);
                    lo[k] = pack_half2((_Float16)(f0 - (float)h0), (_Float16)(f1 - (float)h1));
                }
                if (in) {
                    xsum = sum_piece(lo, sum_piece(hi, xsum));
                    *reinterpret_cast<v4u_t*>(to + 2 * c) = hi;
                    *reinterpret_cast<v4u_t*>(to + L::plane + 2 * c) = lo;
                }
            } else {
                const v4u_t h = narrow_piece<XDT>(px[i], a.keep_inf != 0);
                if (in) {
                    xsum = sum_piece(h, xsum);
                    *reinterpret_cast<v4u_t*>(to + 2 * c) = h;
                }
            }
        }
    };
    request_x(0);

    // ---- where the rows' ids are; the first step's requests ----
    // In operand order a request touches sixteen rows, a lane each.  With up to 16 pairs the lanes ask for chunk lane % 4 of row
    // lane / 4 instead, so that four neighbours read consecutive bytes, and the registers change lanes afterwards: 40 tokens of 128
    // experts 141.6 -> 134.2 us, 20 of 64 91.8 -> 84.5; with more pairs LDS has operands enough to serve: 509 tokens 209.5 -> 218.5.
    // Tiles in planes: lane l asks for entry l, which is operand order and one contiguous run.
    constexpr bool kByRow = NT == 1 && !PL;
    const int ask_row = kByRow ? lane >> 2 : r, ask_chunk = kByRow ? lane & 3 : kg, pull = 4 * (4 * r + kg);
    auto to_operand = [&](const uint4& v) __attribute__((always_inline)) -> uint4 {
        if constexpr (!kByRow) return v;
        return uint4{(uint32_t)__builtin_amdgcn_ds_bpermute(pull, (int)v.x), (uint32_t)__builtin_amdgcn_ds_bpermute(pull, (int)v.y),
                     (uint32_t)__builtin_amdgcn_ds_bpermute(pull, (int)v.z), (uint32_t)__builtin_amdgcn_ds_bpermute(pull, (int)v.w)};
    };
    uint4 lo[2], hi[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        GroupRow& q = g[t];
        q.ok = off_is_plane(off[t]) == PL && row_in_bounds(off[t], q.nb, a.P, a.ids_bytes);           // stored as the call says
        off[t] &= kOffBitsMask;
        const uint32_t nb = (uint32_t)q.nb;
        q.sliced = q.ok && nb >= 4 && nb <= 8 && (off[t] & 31) == 0;
        if (PL) q.ok = q.sliced;
        // the row this lane asks for: its own, or the one of the lane that owns it
        uint64_t base = q.sliced ? (uint64_t)(off[t] >> 3) : 0;
        uint32_t ask_nb = q.sliced ? nb : 0u;
        if constexpr (kByRow) {
            const uint32_t low = __shfl((uint32_t)base, ask_row, 64), high = __shfl((uint32_t)(base >> 32), ask_row, 64);
            base = (uint64_t)high << 32 | low;
            ask_nb = __shfl(ask_nb, ask_row, 64);
        }
        if constexpr (PL) {                                    // the same for all lanes: kept in scalar registers
            q.base = a.ids + (((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(base >> 32)) << 32) | (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)base));
        }
        else if (ask_nb) { q.at = base + (uint32_t)ask_chunk * 4u * ask_nb; q.tail = 4u * (ask_nb - 4u); q.stride = 16u * ask_nb; }
        else { q.at = 0; q.tail = 16; q.stride = 0; }
        const float zero = rintf(-a.min_s[row_at + row0[t]] / a.tau_s[row_at + row0[t]]);
        const int c = q.sliced ? (int)fminf(fmaxf(zero, 0.f), (float)((1 << q.nb) - 1)) : 0;          // (NaN: 0)
        q.centre = c;
        q.negb = pack_half2((_Float16)(float)(-1024 - c), (_Float16)(float)(-1024 - c));
        const int mine = q.sliced ? q.nb : 0, lead = __builtin_amdgcn_readfirstlane(mine);
        q.mode = PL || __builtin_amdgcn_ballot_w64(mine != lead) == 0 ? lead : 0;
    }
    auto issue = [&](bool last) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            if constexpr (PL) {
                // (a tile outside the buffer reads the buffer's first bytes)
                const uint32_t nb = g[t].ok ? (uint32_t)g[t].nb : 4u;
                lo[t] = *reinterpret_cast<const uint4*>(g[t].base + (g[t].ok ? (uint32_t)lane * 16u : 0u));
                hi[t] = *reinterpret_cast<const uint4*>(g[t].base + (g[t].ok ? 1008u + (uint32_t)(lane + 1) * (4u * (nb - 4u)) : 0u));
                g[t].base += last || !g[t].ok ? 0u : 256u * nb;
                continue;
            }
            lo[t] = *reinterpret_cast<const uint4*>(a.ids + g[t].at);
            hi[t] = *reinterpret_cast<const uint4*>(a.ids + g[t].at + g[t].tail);
            g[t].at += last ? 0u : g[t].stride;                // past the end: the last step's lines again, nothing under a branch
        }
    };
    issue(n_steps == 1);

    // ---- down: the power of two that brings the row's largest |H| into [8192, 16384) ----
    if constexpr (DOWN) {
        float top = 0.f;
        const float* hrow = reinterpret_cast<const float*>(xrow);
        // eight requests at a time: one by one, the 12 trips of a 768-column row were 8 of the launch's 95 us
        for (int c0 = sub * 4; c0 < a.P; c0 += L::TPR * 4 * 8) {
            float4 h[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) h[k] = *reinterpret_cast<const float4*>(hrow + min(c0 + k * L::TPR * 4, a.P - 4));
#pragma unroll
            for (int k = 0; k < 8; ++k) top = fmaxf(fmaxf(fmaxf(top, fabsf(h[k].x)), fabsf(h[k].y)), fmaxf(fabsf(h[k].z), fabsf(h[k].w)));
        }
#pragma unroll
        for (int o = L::TPR / 2; o >= 1; o >>= 1) top = fmaxf(top, __shfl_xor(top, o, 64));
        int ex = 0;
        if (top > 0.f && top < __builtin_inff()) ex = 14 - __builtin_amdgcn_frexp_expf(top);     // top = m 2^e, m in [0.5, 1)
        ex = max(-126, min(ex, 126));
        scale = __uint_as_float((uint32_t)(127 + ex) << 23);
        if (sub == 0 && rho < kGroupTokens) s_inv[rho] = __uint_as_float((uint32_t)(127 - ex) << 23);
    }
    store_x(0);
    lds_barrier();

    // ---- the columns ----
    v4f_t acc[2][NT];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int m = 0; m < NT; ++m) acc[t][m] = v4f_t{0.f, 0.f, 0.f, 0.f};
    const int n_chunks = (n_steps + L::CS - 1) / L::CS;
    for (int s = 0; s < n_steps; ++s) {
        const int chunk = s / L::CS;
        const bool stage = s % L::CS == L::CS - 1 && chunk + 1 < n_chunks;
        v4u_t b[2][4];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const GroupRow& q = g[t];
            const uint4 l = to_operand(lo[t]), h = to_operand(hi[t]);
            switch (q.mode) {
                case 4: decode_centred<4>(l, h, q.negb, b[t]); break;
                case 5: decode_centred<5>(l, h, q.negb, b[t]); break;
                case 6: decode_centred<6>(l, h, q.negb, b[t]); break;
                case 7: decode_centred<7>(l, h, q.negb, b[t]); break;
                case 8: decode_centred<8>(l, h, q.negb, b[t]); break;
                default:
#pragma unroll
                    for (int j = 0; j < 4; ++j) b[t][j] = v4u_t{0u, 0u, 0u, 0u};
                    if constexpr (PL) break;
                    if (q.sliced && q.nb == 4) decode_centred<4>(l, h, q.negb, b[t]);
                    if (q.sliced && q.nb == 5) decode_centred<5>(l, h, q.negb, b[t]);
                    if (q.sliced && q.nb == 6) decode_centred<6>(l, h, q.negb, b[t]);
                    if (q.sliced && q.nb == 7) decode_centred<7>(l, h, q.negb, b[t]);
                    if (q.sliced && q.nb == 8) decode_centred<8>(l, h, q.negb, b[t]);
            }
        }
        issue(s + 2 >= n_steps);
        if (stage) request_x(chunk + 1);
        const unsigned char* x0 = smem + (chunk & 1) * L::buf + r * L::pitch + (s % L::CS) * (2 * kStepCols) + kg * 64;
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int m = 0; m < NT; ++m) {
                const v4u_t xa = *reinterpret_cast<const v4u_t*>(x0 + m * 16 * L::pitch + 16 * j);
#pragma unroll
                for (int t = 0; t < 2; ++t) acc[t][m] = F::mfma(xa, b[t][j], acc[t][m]);
                if constexpr (DOWN) {
                    const v4u_t xl = *reinterpret_cast<const v4u_t*>(x0 + L::plane + m * 16 * L::pitch + 16 * j);
#pragma unroll
                    for (int t = 0; t < 2; ++t) acc[t][m] = F::mfma(xl, b[t][j], acc[t][m]);
                }
            }
        if (stage) {                                           // everybody is past the buffer's previous chunk since the last barrier
            store_x(chunk + 1);
            lds_barrier();
        }
    }

    // ---- the pairs' sums ----
#pragma unroll
    for (int o = L::TPR / 2; o >= 1; o >>= 1) xsum += __shfl_xor(xsum, o, 64);
    if (sub == 0 && stages) s_sum[rho] = xsum;
    lds_barrier();

    // ---- rows the slicing cannot read (width outside 4..8, not dword aligned): id by id, in place of what stands there ----
    const int64_t clamp_byte = (a.ids_bytes - 8) & ~(int64_t)3;
    if constexpr (!PL)
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        uint64_t odd = __builtin_amdgcn_ballot_w64(kg == 0 && !g[t].sliced && g[t].ok);
        while (odd) {
            const int rr = __builtin_ctzll(odd);
            odd &= odd - 1;
            const int nb = __shfl(g[t].nb, rr, 64);
            const int64_t off = a.bit_off[(size_t)e * a.Q + row0[t] + rr];
            for (int tok = 0; tok < n; ++tok) {
                const int p = s_pair[tok];
                float part = 0.f;
                for (int c = lane; c < a.P; c += kWave) {
                    float x;
                    if constexpr (DOWN) x = reinterpret_cast<const float*>(a.X)[(size_t)p * a.P + c] * (1.0f / s_inv[tok]);
                    else {
                        x = load_as_f32<XDT>(a.X, (int64_t)(p / a.topk) * a.P + c);
                        if (XDT != QVB8_F16 || !a.keep_inf) x = f16_bits_to_f32(sat_half_bits(x));
                    }
                    part = __builtin_fmaf(x, (float)load_field(a.ids, off + (int64_t)c * nb, nb, clamp_byte), part);
                }
                const float tot = wave_sum(part);
#pragma unroll
                for (int m = 0; m < NT; ++m)
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        if (r == rr && tok == m * 16 + kg * 4 + k) acc[t][m][k] = tot;
            }
        }
    }

    // ---- y = tau_s * sum(x (id - c)) + (min_s + c tau_s) * sum(x) ----
    double ts[2], mid[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        ts[t] = g[t].ok ? (double)a.tau_s[row_at + row0[t]] : (double)__builtin_nanf("");
        mid[t] = (double)a.min_s[row_at + row0[t]] + (g[t].sliced ? (double)g[t].centre * ts[t] : 0.0);
    }
    auto value = [&](int t, int m, int k) {
        const int tok = m * 16 + kg * 4 + k;
        double y = ts[t] * (double)acc[t][m][k] + mid[t] * (double)s_sum[tok];
        if constexpr (DOWN) y *= (double)s_inv[tok];
        return (float)y;
    };
#pragma unroll
    for (int m = 0; m < NT; ++m)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int tok = m * 16 + kg * 4 + k;
            if (tok >= n) continue;
            float* to = a.out + (size_t)s_pair[tok] * (DOWN ? a.Q : a.units) + r;
            if (paired) {
                const float y = value(0, m, k);
                if (on[0]) to[row0[0]] = (y / (1.0f + __expf(-y))) * value(1, m, k);
            } else {
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    float y = value(t, m, k);
                    if constexpr (!DOWN) { const float p = fmaxf(y, 0.f); y = y != y ? y : p * p; }
                    if (on[t]) to[row0[t]] = y;
                }
            }
        }
}

template <bool DOWN, int XDT, bool PL>
__global__ void __launch_bounds__(kGroupThreads, 4) moe_group_kernel(MoeGroupArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    // workgroup b runs on XCD b % 8: an item's row blocks follow each other on ONE XCD, whose L2 then serves its
    // activations to all of them
    const int b = (int)blockIdx.x, on_xcd = b >> 3;
    const int item = (b & 7) + 8 * (on_xcd / a.row_blocks), rb = on_xcd % a.row_blocks;
    if (item >= a.plan.n_bad[2]) return;                       // the whole workgroup
    // the slot this item's token block belongs to: the last one with no more than `item` blocks before it
    const int n_slots = a.plan.n_bad[1], lane = threadIdx.x & 63;
    int at = -1;
    for (int i = 0; i < n_slots; i += 64) {
        const int w = i + lane < n_slots ? a.plan.slot[i + lane].w : 0x7fffffff;
        at += __builtin_popcountll(__builtin_amdgcn_ballot_w64(w <= item));
    }
    at = __builtin_amdgcn_readfirstlane(at);
    const int4 slot = a.plan.slot[at];
    const int first = slot.y + (item - slot.w) * kGroupTokens;
    const int n = __builtin_amdgcn_readfirstlane(min(kGroupTokens, slot.z - first));
    const int e = __builtin_amdgcn_readfirstlane(slot.x);
    switch ((n + 15) / 16) {
        case 1: moe_group_body<1, DOWN, XDT, PL>(a, smem, e, first, n, rb); break;
        case 2: moe_group_body<2, DOWN, XDT, PL>(a, smem, e, first, n, rb); break;
        case 3: moe_group_body<3, DOWN, XDT, PL>(a, smem, e, first, n, rb); break;
        default: moe_group_body<4, DOWN, XDT, PL>(a, smem, e, first, n, rb); break;
    }
}

template <bool DOWN, int XDT, bool PL>
int launch_stored(const MoeGroupArgs& a, unsigned blocks, hipStream_t s) {
    if (int rc = host::raise_lds_limit<moe_group_kernel<DOWN, XDT, PL>>(kGroupLds, "qvb8_moe_experts")) return rc;
    hipLaunchKernelGGL((moe_group_kernel<DOWN, XDT, PL>), dim3(blocks), dim3(kGroupThreads), kGroupLds, s, a);
    return host::check_launch("qvb8_moe_experts");
}
template <bool DOWN, int XDT>
int launch_as(const MoeGroupArgs& a, unsigned blocks, hipStream_t s) {
    return a.planes ? launch_stored<DOWN, XDT, true>(a, blocks, s) : launch_stored<DOWN, XDT, false>(a, blocks, s);
}

}  // namespace

// whole 128-column steps and 16-row tiles; anything else takes the general path
bool moe_group_shapes_ok(int64_t P_up, int64_t Q_dn, int64_t P_dn) {
    return P_up % kStepCols == 0 && P_dn % kStepCols == 0 && Q_dn % 16 == 0 && host::env_int("QVB8_MOE_GROUPED", 1) != 0;
}

int launch_moe_group(bool down, int x_dtype, MoeGroupArgs a, int64_t npairs, hipStream_t s) {
    const int tiles = (!down && a.gated) ? a.units / 16 : (a.Q / 16 + 1) / 2;
    a.row_blocks = (tiles + kGroupWaves - 1) / kGroupWaves;
    // every expert in use may have one block that is not full
    a.items = (int)(moe_slots(a.E, npairs) + npairs / kGroupTokens);
    const unsigned blocks = (unsigned)((a.items + 7) / 8 * 8 * a.row_blocks);
    if (down) return launch_as<true, QVB8_F32>(a, blocks, s);
    if (x_dtype == QVB8_F32) return launch_as<false, QVB8_F32>(a, blocks, s);
    if (x_dtype == QVB8_F16) return launch_as<false, QVB8_F16>(a, blocks, s);
    return launch_as<false, QVB8_BF16>(a, blocks, s);
}

}  // namespace qvb8
