// Fused QVB8 decode + GEMM for 17..64 rows of X, rows of W in width order (gfx950): every wave has columns of its own.
//
// A workgroup of eight waves takes up to eight 16-row tiles of one width x all rows of X; wave w multiplies the 128-column steps w, w + 8,
// ... of all of them, so nothing is shared while it runs: no barrier, no LDS.  Ids come in the operand's order (rows in planes: contiguous
// kilobytes, read once, non-temporal), X too (columns_prep_kernel lays it out and narrows it), a quarter of a step at a time and three
// quarters ahead; a tile's ids are asked for again as soon as their last quarter is decoded, or a step further ahead where registers allow.
// The eight partial sums of a result meet in LDS at the end, in a fixed order.
//
//   y = tau_s * sum(x (id - c)) + (min_s + c tau_s) * sum(x),  c the middle of the width, id - c exact in fp16, joined in double.
//
// Error of fp32 results against 64 bits: 2.0e-7 .. 4.3e-7 of their norm (x of mean 0), 4.0e-6 .. 1.8e-5 (x of mean 3, where the terms
// cancel); with 1024 + id as the operand, as gemm_kernel has it, 1.0e-5 .. 2.7e-5 and 1.3e-4 .. 9.3e-4.
//
// Bound by memory: 24576 x 4096 of 7 bits, 64 rows: 25.3 us, of it 17 in the loop (88 MB at 5.2 TB/s), 3 at the end (6 with the rows' constants
// fetched there); columns_prep_kernel 3.  gemm_kernel took 35.2 and 4.3 for its column ranges' sums: 194 workgroups of 256 CUs, and its ids'
// way through LDS into operand order and the operands of X shared there kept LDS busy half of the time.  What decides here: X from L2 is
// 512 KB a CU, more than its ids, so a wave should have as many tiles as registers hold (three tiles a wave, two waves a step 30.5 us), without a spill
// (a few registers spilled 49); one unit more than CUs is a second round (47), so runs of a width are whole units (module.py).
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <algorithm>
#include <type_traits>

#include "../../include/qvb8_amd.h"
#include "qvb8_columns.h"
#include "qvb8_device.h"
#include "qvb8_host.h"
#include "qvb8_mma_device.h"

namespace qvb8 {
namespace {

// One workgroup per row of X (rows M.. of the last token tile: zeros).
// X16[step][token tile][j][lane = token + 16 kg][8]: columns 128 step + 32 kg + 8 j .. + 7 of the token, what the lane feeds MFMA j.
template <bool XC>
__global__ void __launch_bounds__(256) columns_prep_kernel(const uint16_t* __restrict__ X, int M, int P, int MT, uint16_t* __restrict__ X16, float* __restrict__ sx) {
    __shared__ float red[4];
    const int m = blockIdx.x, tid = threadIdx.x, n_steps = P / kStepCols;
    uint4* const to = reinterpret_cast<uint4*>(X16) + (m >> 4) * 256 + (m & 15);
    float part = 0.f;
    for (int p = tid; p < n_steps * 16; p += 256) {                                       // 8-column pieces
        uint32_t w[4] = {0u, 0u, 0u, 0u};
        if (m < M) {
            const uint4 v = *reinterpret_cast<const uint4*>(X + (size_t)m * P + 8 * p);
            w[0] = v.x; w[1] = v.y; w[2] = v.z; w[3] = v.w;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                w[k] = XIn<false, XC>::pair(w[k]);
                part += f16_bits_to_f32(w[k] & 0xFFFFu) + f16_bits_to_f32(w[k] >> 16);
            }
        }
        to[(size_t)(p >> 4) * MT * 256 + (p & 3) * 64 + ((p >> 2) & 3) * 16] = uint4{w[0], w[1], w[2], w[3]};
    }
    if (tid < 16) to[(size_t)n_steps * MT * 256 + (tid & 3) * 64 + (tid >> 2) * 16] = uint4{0u, 0u, 0u, 0u};
    part = wave_sum(part);
    if ((tid & 63) == 0) red[tid >> 6] = part;
    __syncthreads();
    if (tid == 0 && m < M) sx[m] = (red[0] + red[1]) + (red[2] + red[3]);
}

// a lane's slice of one tile and step: the first four dwords and the NB - 4 others
template <int NB> struct Slice { uint32_t w[NB]; };
template <int NB>
__device__ __forceinline__ void load_slice_at(const uint8_t* lo, const uint8_t* hi, Slice<NB>& s) {
    const v4u_t l = __builtin_nontemporal_load(reinterpret_cast<const v4u_t*>(lo));
#pragma unroll
    for (int k = 0; k < 4; ++k) s.w[k] = l[k];
    if constexpr (NB == 8) {
        const v4u_t h = __builtin_nontemporal_load(reinterpret_cast<const v4u_t*>(hi));
#pragma unroll
        for (int k = 0; k < 4; ++k) s.w[4 + k] = h[k];
    } else {
#pragma unroll
        for (int k = 4; k < NB; ++k) s.w[k] = __builtin_nontemporal_load(reinterpret_cast<const uint32_t*>(hi) + (k - 4));
    }
}
// What is taken off every id of a width: the middle of its range, so that the sums are about as small as their results (1024 + id, with the
// 1024 taken off the sum, rounds 10 to 30 times as coarsely).
constexpr int centre_of(int nb) { return 1 << (nb - 1); }
// quarter J of a slice: eight ids, one operand
template <int NB, int PR, int END>
__device__ __forceinline__ void quarter_pairs(const uint32_t (&w)[kMaxFastNb], uint32_t (&e)[4]) {
    if constexpr (PR < END) { e[PR % 4] = pair_extract<NB, PR>(w); quarter_pairs<NB, PR + 1, END>(w, e); }
}
template <int NB, int PR, int END>
__device__ __forceinline__ void quarter_spread(uint32_t (&e)[4]) {
    if constexpr (PR < END) { e[PR % 4] = pair_spread<NB, PR>(e[PR % 4]); quarter_spread<NB, PR + 1, END>(e); }
}
template <int NB, int J>
__device__ __forceinline__ void decode_quarter(const uint32_t (&w)[kMaxFastNb], v4u_t& b) {
    uint32_t e[4];
    quarter_pairs<NB, 4 * J, 4 * J + 4>(w, e);
    quarter_spread<NB, 4 * J, 4 * J + 4>(e);
    uint32_t m = ((1u << NB) - 1u) * 0x00010001u, bias = Fmt<false>::bias_bits;
    asm("" : "+v"(m), "+v"(bias));
    const half2_t off = {(_Float16)(float)(-1024 - centre_of(NB)), (_Float16)(float)(-1024 - centre_of(NB))};
#pragma unroll
    for (int p = 0; p < 4; ++p) { const uint32_t w1 = and_or3(e[p], m, bias); b[p] = __builtin_bit_cast(uint32_t, (half2_t)(__builtin_bit_cast(half2_t, w1) + off)); }
}
// (values, not references: a choice between variables would put them in memory)
template <typename V> __device__ __forceinline__ V of_run(int c, V v0, V v1, V v2) { return c == 0 ? v0 : c == 1 ? v1 : v2; }
// The lane's number, worked out anew where it is asked for: what is made from it is not kept in registers across the loop.
__device__ __forceinline__ int lane_now() {
    int l;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
    return l;
}
// a unit of row tiles: positions pos0 .. end of the run of NB-bit rows first .. run_end, which starts at byte `byte0`
struct Unit { int pos0, end, first, run_end; uint64_t byte0; };

// tiles whose sums meet in LDS at a time: at most 128 KB
constexpr int columns_tiles_at_once(int MT, int G) { return 8 * G * MT <= 128 ? G : G / 2; }
constexpr int kColumnsWaves = 8;

template <int NB, bool PL, int MT, int G>
__device__ __forceinline__ void columns_run(const ColumnsArgs& a, const uint16_t* X16, const uint8_t* ids_base, unsigned char* smem, const Unit& u) {
    constexpr int W = kColumnsWaves;
    // registers of a lane: sums, activations, ids of a step, and what the rest takes: a second step of ids where it fits
    constexpr int kSums = 4 * MT * G, kX = 16 * MT, kIds = NB * G, kRest = 36;
    constexpr int RB = kSums + kX + 2 * kIds + kRest <= 232 ? 2 : 1;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, kg = lane >> 4;
    const int n_steps = a.P / kStepCols;
    const uint32_t row_bytes = (uint32_t)a.P / 8u * NB;
    const uint8_t* const tiles = ids_base + u.byte0 + (uint64_t)(uint32_t)(u.pos0 - u.first) * row_bytes;
    const int n_tiles = (u.end - u.pos0 + 15) / 16;
    // the lane's slice of tile t, step s (past the end: the last one again; past the last tile or row: the last one, not stored)
    auto request = [&](int t, int s, Slice<NB>& to) __attribute__((always_inline)) {
        [[maybe_unused]] const uint8_t* at = tiles + ((uint64_t)(uint32_t)min(t, n_tiles - 1) * (16u * row_bytes) + (uint64_t)(uint32_t)min(s, n_steps - 1) * (PL ? 256u * NB : 16u * NB));
        if constexpr (PL) load_slice_at<NB>(at + (uint32_t)lane * 16u, at + 1024u + (uint32_t)lane * (4u * (NB - 4u)), to);
        else {
            const int ln = lane_now(), pos = min(u.pos0 + 16 * min(t, n_tiles - 1) + (ln & 15), u.end - 1), t0 = pos & ~15;
            const bool whole = a.planes && t0 >= u.first && t0 + 16 <= u.run_end;
            const uint32_t slot = (uint32_t)(pos & 15) + (uint32_t)(ln & 48), g = (uint32_t)(ln >> 4), sc = (uint32_t)min(s, n_steps - 1);
            const uint8_t* lo = ids_base + u.byte0 + (uint64_t)(uint32_t)((whole ? t0 : pos) - u.first) * row_bytes + (whole ? sc * (256u * NB) + slot * 16u : sc * (16u * NB) + g * (4u * NB));
            load_slice_at<NB>(lo, lo + (whole ? 1024u - slot * 16u + slot * (4u * (NB - 4u)) : 16u), to);
        }
    };
    auto decode = [&](const Slice<NB>& from, auto quarter, v4u_t& b) __attribute__((always_inline)) {
        uint32_t w[kMaxFastNb];
#pragma unroll
        for (int k = 0; k < NB; ++k) w[k] = from.w[k];
        decode_quarter<NB, decltype(quarter)::value>(w, b);
    };
    // X a quarter of a step at a time (what the MFMAs j take), three quarters ahead
    v4u_t x[4][MT];
    auto request_x = [&](int s, int j) __attribute__((always_inline)) {
        // past the end: the step of zeros
        const uint8_t* at = reinterpret_cast<const uint8_t*>(X16) + ((uint64_t)(uint32_t)min(s, n_steps) * (MT * 4096) + (uint32_t)j * 1024u);
#pragma unroll
        for (int m = 0; m < MT; ++m) x[j][m] = *reinterpret_cast<const v4u_t*>(at + m * 4096 + (uint32_t)lane * 16u);
    };
    Slice<NB> raw[RB][G];
    v4f_t acc[G][MT];
#pragma unroll
    for (int t = 0; t < G; ++t)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[t][m] = v4f_t{0.f, 0.f, 0.f, 0.f};

    // what the end needs: asked for first, in LDS when the requests of the first steps are out
    constexpr int CT = columns_tiles_at_once(MT, G);               // of every wave's tiles
    v4f_t* const parts = reinterpret_cast<v4f_t*>(smem);           // [wave][tile][token tile][lane]
    uint4* const s_fin = reinterpret_cast<uint4*>(smem + W * CT * MT * 1024);
    float* const s_sx = reinterpret_cast<float*>(s_fin + 16 * G);
    const uint4 my_fin = a.fin[min(u.pos0 + min(tid, 16 * G - 1), u.end - 1)];
    const float my_sx = a.sx[min(lane, a.M - 1)];
    __builtin_amdgcn_sched_barrier(0);
    const int s0 = wave, n_it = (n_steps + W - 1) / W;
    request_x(s0, 0);
    request_x(s0, 1);
    request_x(s0, 2);
#pragma unroll
    for (int t = 0; t < G; ++t) request(t, s0, raw[0][t]);
    if constexpr (RB == 2)
#pragma unroll
        for (int t = 0; t < G; ++t) request(t, s0 + W, raw[RB - 1][t]);
    if (tid < 16 * G) s_fin[tid] = my_fin;
    if (tid < 64) s_sx[tid] = my_sx;
    auto quarter_step = [&](int s, auto quarter, Slice<NB> (&ids)[G]) __attribute__((always_inline)) {
        constexpr int J = decltype(quarter)::value;
        request_x(J == 0 ? s : s + W, (J + 3) % 4);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < G; ++t) {
            v4u_t b;
            decode(ids[t], quarter, b);
            if constexpr (J == 3) request(t, s + RB * W, ids[t]);
#pragma unroll
            for (int m = 0; m < MT; ++m) acc[t][m] = Fmt<false>::mfma(x[J][m], b, acc[t][m]);
            if constexpr (kSums + kX + RB * kIds + kRest > 230) __builtin_amdgcn_sched_barrier(0);   // (the next tile's operand beside this one's would not fit)
        }
    };
    auto step = [&](int s, Slice<NB> (&ids)[G]) __attribute__((always_inline)) {
        quarter_step(s, std::integral_constant<int, 0>{}, ids);
        quarter_step(s, std::integral_constant<int, 1>{}, ids);
        quarter_step(s, std::integral_constant<int, 2>{}, ids);
        quarter_step(s, std::integral_constant<int, 3>{}, ids);
    };
    for (int i = 0; i < n_it; i += RB) {
        step(s0 + W * i, raw[0]);
        if constexpr (RB == 2) step(s0 + W * (i + 1), raw[RB - 1]);       // (an odd number of steps: the step of zeros)
    }
    // ---- the waves' columns meet ----
#pragma unroll
    for (int t0 = 0; t0 < G; t0 += CT) {
        if (t0 > 0) __syncthreads();
#pragma unroll
        for (int t = 0; t < CT; ++t)
#pragma unroll
            for (int m = 0; m < MT; ++m) parts[((wave * CT + t) * MT + m) * 64 + lane] = acc[t0 + t][m];
        __syncthreads();
        for (int i = tid; i < CT * MT * 64; i += 64 * W) {
            const int t = t0 + i / (MT * 64), m = (i / 64) % MT;
            if (u.pos0 + 16 * t + r >= u.end) continue;
            v4f_t sum = parts[i];
#pragma unroll
            for (int w = 1; w < W; ++w) sum += parts[w * CT * MT * 64 + i];
            const uint4 f = s_fin[16 * t + r];
            if (f.z >= (uint32_t)a.Q) continue;
            const double ts = (double)__uint_as_float(f.x), mid = (double)__uint_as_float(f.y) + (double)centre_of(NB) * ts;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int tok = m * 16 + kg * 4 + k;
                if (tok < a.M) {
                    store_y(a.out, a.out_dt, (int64_t)tok * a.Q + f.z, (float)(ts * (double)sum[k] + mid * (double)s_sx[tok]));
                }
            }
        }
    }
}

template <bool PL, int MT, int G>
__device__ __forceinline__ void columns_of_width(int nb, const ColumnsArgs& a, const uint16_t* X16, const uint8_t* ids, unsigned char* smem, const Unit& u) {
    switch (nb) {
        case 4: columns_run<4, PL, MT, G>(a, X16, ids, smem, u); break;
        case 5: columns_run<5, PL, MT, G>(a, X16, ids, smem, u); break;
        case 6: columns_run<6, PL, MT, G>(a, X16, ids, smem, u); break;
        case 7: columns_run<7, PL, MT, G>(a, X16, ids, smem, u); break;
        default: columns_run<8, PL, MT, G>(a, X16, ids, smem, u); break;
    }
}

template <bool PL, int MT, int G>
__global__ void __launch_bounds__(64 * kColumnsWaves, kColumnsWaves / 4) columns_kernel(const uint16_t* __restrict__ X16, const uint8_t* __restrict__ ids, ColumnsArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    // the rows behind the last whole tile in planes are a unit of their own, read row by row (its run: the one of the last row)
    const bool rest = PL && (int)blockIdx.x == a.units3;
    const int bx = (int)blockIdx.x, c = rest ? (a.Q > a.first1 ? 1 : 0) + (a.Q > a.first2 ? 1 : 0) : (bx >= a.units1 ? 1 : 0) + (bx >= a.units2 ? 1 : 0);
    const uint32_t nb0 = a.widths & 255u, nb1 = (a.widths >> 8) & 255u, nb2 = (a.widths >> 16) & 255u;
    const uint64_t byte1 = (uint64_t)a.first1 * ((uint32_t)a.P / 8u * nb0), byte2 = byte1 + (uint64_t)(a.first2 - a.first1) * ((uint32_t)a.P / 8u * nb1);
    Unit u;
    u.first = of_run(c, 0, a.first1, a.first2);
    u.byte0 = of_run(c, (uint64_t)0, byte1, byte2);
    const int nb = (int)of_run(c, nb0, nb1, nb2), run_end = u.run_end = of_run(c, a.first1, a.first2, a.Q);
    u.pos0 = u.first + 16 * G * (bx - of_run(c, 0, a.units1, a.units2));
    const int whole = PL ? run_end & ~15 : run_end;
    if (rest) {
        u.pos0 = whole;
        u.end = run_end;
        columns_of_width<false, MT, 1>(nb, a, X16, ids, smem, u);
        return;
    }
    u.end = min(u.pos0 + 16 * G, whole);
    if (u.pos0 >= u.end) return;
    columns_of_width<PL, MT, G>(nb, a, X16, ids, smem, u);
}

template <int MT, int G>
int launch_as(const ColumnsPlan& p, const ColumnsArgs& a, hipStream_t s) {
    constexpr size_t lds = (size_t)kColumnsWaves * columns_tiles_at_once(MT, G) * MT * 1024 + 16 * G * 16 + 64 * 4;
    const dim3 grid((unsigned)p.units), block(64 * kColumnsWaves);
    if (int rc = p.by_tile ? host::raise_lds_limit<columns_kernel<true, MT, G>>(lds, "qvb8_mma") : host::raise_lds_limit<columns_kernel<false, MT, G>>(lds, "qvb8_mma")) return rc;
    if (p.by_tile) hipLaunchKernelGGL((columns_kernel<true, MT, G>), grid, block, lds, s, a.X16, a.ids, a);
    else hipLaunchKernelGGL((columns_kernel<false, MT, G>), grid, block, lds, s, a.X16, a.ids, a);
    return host::check_launch("qvb8_mma");
}
template <int MT>
int launch_rows(const ColumnsPlan& p, const ColumnsArgs& a, hipStream_t s) {
    switch (p.G) {
        case 1: return launch_as<MT, 1>(p, a, s);
        case 2: return launch_as<MT, 2>(p, a, s);
        case 3: return launch_as<MT, 3>(p, a, s);
        case 4: return launch_as<MT, 4>(p, a, s);
        case 6: return launch_as<MT, 6>(p, a, s);
        default:
            if constexpr (MT == 2) return launch_as<MT, 8>(p, a, s);
            else return launch_as<MT, 6>(p, a, s);
    }
}
int64_t align256(int64_t n) { return (n + 255) & ~(int64_t)255; }

}  // namespace

namespace {
constexpr int kMostRanges = 4;
constexpr int kGroups[] = {1, 2, 3, 4, 6, 8};                      // row tiles a unit may have
constexpr int most_tiles(int MT) { return MT == 2 ? 8 : 6; }       // ... as the registers hold
// What a call takes, in 1/100 us: rounds of units (start and end of each, then its wave's steps -- bound by the ids' share of memory, by the
// activations' share of L2 or by decode and products).  `ranges`: as if the columns were cut into so many, joined by another launch; with
// more than one the kernel is not taken.
int64_t columns_cost(int64_t units, int MT, int G, int64_t M, int64_t Q, int64_t n_steps, int ranges = 1) {
    const int64_t cus = host::device_cus(), rounds = (units * ranges + cus - 1) / cus;
    const int64_t steps = ((n_steps + ranges - 1) / ranges + kColumnsWaves - 1) / kColumnsWaves;
    const int64_t memory = 68 * G * std::min<int64_t>(units * ranges, rounds * cus) / (rounds * cus);
    const int64_t step = std::max<int64_t>({memory, 62 * MT, 22 * G + 6 * G * MT});
    return rounds * (700 + steps * step) + (ranges > 1 ? 500 + 100 * ranges + ranges * M * Q / 5000 : 0);
}
}  // namespace

static ColumnsPlan make_plan(int64_t M, int64_t Q, int64_t P) {
    ColumnsPlan p = {};
    p.MT = M <= 32 ? 2 : M <= 48 ? 3 : 4;
    // By the weight's size alone, not by how its rows are stored: a row's products are then the same bit for bit.
    const int64_t n_steps = P / kStepCols, tiles = (Q + 15) / 16;
    const int64_t cus = host::device_cus();
    int64_t best = INT64_MAX, units_best = 0;
    int ranges = 1;
    for (int z = 1; z <= kMostRanges && (z == 1 || n_steps / z >= kColumnsWaves); ++z)
        for (int g : kGroups) {
            if (g > most_tiles(p.MT)) break;
            const int64_t units = (tiles + g - 1) / g, cost = columns_cost(units, p.MT, g, M, Q, n_steps, z);
            if (cost < best) { best = cost; ranges = z; units_best = units; }
        }
    // The kernels that stage X in LDS (gemm_kernel) keep: up to 32 rows, weights of more than a round of units (34816 x 5120, 20 rows, 40.8 us
    // against 45.7) or of more than 8192 columns (20000 x 9984, 20 rows, 35.9 / 42.0); few rows of W and long ones, whose columns they split over the chip (5120 x 17408, 24 rows 23.8 / 36.5, 64 rows 33.3 / 37).
    p.taken = ranges == 1 && (M > 32 || (units_best <= cus && n_steps <= 8 * kColumnsWaves)) && (10 * units_best >= 7 * cus || n_steps <= 4 * kColumnsWaves);
    // ... and, where they can read the weight (P a multiple of 256), long rows with any number of rows of X (us them / here: 26675 x 8960, 33
    // rows 64.6 / 70.1, 64 rows 67.7 / 79.3; up to 32 rows those of more than 48 steps: 12290 x 7936, 17 rows 27.5 / 29.4, 40 rows 36.6 / 33.5) and large weights whose waves would have a single step each (32603 x 1024, 17 rows 14.9 / 18.5,
    // 64 rows 24.2 / 24.6; of ten steps, 15339 x 1280, 19.4 / 16.6 and 30.3 / 22.6).  The tile kernel, which takes the others, is behind (29291 x 8320,
    // 40 rows, 136 / 80).
    if (P % 256 == 0 && (n_steps > (M <= 32 ? 6 : 8) * kColumnsWaves || (n_steps <= kColumnsWaves && tiles >= 1024))) p.taken = false;
    p.x16_at = align256(qvb8_mma_rowinfo_bytes(Q));
    p.sx_at = p.x16_at + (n_steps + 1) * p.MT * 4096;
    p.bytes = p.sx_at + align256(M * 4);
    return p;
}

ColumnsPlan plan_columns(int64_t M, int64_t Q, int64_t P) {
    // (a call asks twice, for its workspace and to launch, and working it out takes a microsecond of the host)
    static thread_local struct { int64_t M, Q, P, cus; ColumnsPlan plan; } last = {};
    const int64_t cus = host::device_cus();
    if (last.M != M || last.Q != Q || last.P != P || last.cus != cus) last = {M, Q, P, cus, make_plan(M, Q, P)};
    return last.plan;
}

int launch_columns(ColumnsPlan p, ColumnsArgs a, const uint16_t* X, int mode, uint16_t* x16, float* sx, hipStream_t s) {
    // units of G tiles of one width
    const int rows[3] = {a.first1, a.first2 - a.first1, a.Q - a.first2};
    // (whole tiles in planes lie at multiples of 16: where a run starts elsewhere, every lane works out where its row is)
    const bool planes = a.planes && (a.first1 % 16 == 0 || a.first1 == a.Q) && (a.first2 % 16 == 0 || a.first2 == a.Q);
    p.by_tile = planes;
    int64_t best = INT64_MAX;
    for (int g : kGroups) {
        if (g > most_tiles(p.MT)) break;
        int units[3];
        for (int c = 0; c < 3; ++c) units[c] = ((planes ? rows[c] / 16 : (rows[c] + 15) / 16) + g - 1) / g;
        const int whole = units[0] + units[1] + units[2], all = whole + (planes && a.Q % 16 != 0 ? 1 : 0);
        const int64_t cost = columns_cost(all, p.MT, g, a.M, a.Q, a.P / kStepCols);
        if (cost >= best) continue;
        best = cost;
        p.G = g; p.units = all;
        a.units1 = units[0]; a.units2 = units[0] + units[1]; a.units3 = whole;
    }
    const dim3 grid((unsigned)(16 * p.MT));
    if (mode == 1) hipLaunchKernelGGL((columns_prep_kernel<true>), grid, dim3(256), 0, s, X, a.M, a.P, p.MT, x16, sx);
    else hipLaunchKernelGGL((columns_prep_kernel<false>), grid, dim3(256), 0, s, X, a.M, a.P, p.MT, x16, sx);
    if (int rc = host::check_launch("qvb8_mma activations")) return rc;
    a.X16 = x16; a.sx = sx;
    if (p.MT == 2) return launch_rows<2>(p, a, s);
    if (p.MT == 3) return launch_rows<3>(p, a, s);
    return launch_rows<4>(p, a, s);
}

}  // namespace qvb8
