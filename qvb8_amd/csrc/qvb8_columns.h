// The kernel of 17..64 rows of X on rows stored in planes (qvb8_columns.hip), as qvb8_mma launches it.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace qvb8 {

constexpr int kColumnsMaxM = 64;

struct ColumnsArgs {
    const uint16_t* X16;           // activations in operand order, kStepCols columns a step, one step of zeros behind the last
    const float* sx;               // sums of the rows of X
    const uint8_t* ids;
    const uint4* fin;
    float* out;                    // Y
    int M, Q, P;
    int out_dt;                    // what `out` holds: 0 fp32, 1 fp16, 2 bf16
    int planes;                    // whole tiles are stored in planes (see qvb8_device.h)
    int first1, first2;            // positions where the second and the third width start (Q when there is none)
    int units1, units2, units3;    // units before the second, the third width, and behind its whole tiles
    uint32_t widths;               // nb0 | nb1 << 8 | nb2 << 16, each 4..8
};

struct ColumnsPlan {
    int MT, G;                     // token tiles, row tiles per workgroup
    int units;
    bool taken;                    // whether this kernel is the one for the sizes
    bool by_tile;                  // tiles of one width in planes at multiples of 16
    int64_t x16_at, sx_at, bytes;  // workspace layout, bytes from its start (after the row records' place)
};

ColumnsPlan plan_columns(int64_t M, int64_t Q, int64_t P);
// mode 0: fp16 X; 1: bf16 X, narrowed to saturated fp16
int launch_columns(ColumnsPlan p, ColumnsArgs a, const uint16_t* X, int mode, uint16_t* x16, float* sx, hipStream_t s);

}  // namespace qvb8
