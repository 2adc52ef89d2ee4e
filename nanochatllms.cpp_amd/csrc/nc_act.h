// nc_act.h -- activation-row access for the elementwise / norm / attention
// kernels.  The thread that handles element e of a row sits on lane e % 64
// of some wavefront, so each 32-value Q8 block lives on one 32-lane half of
// a wavefront and can be (re)quantized with half-wave shuffles.
#pragma once

#include "nc_device.h"

namespace nc {

// Value of element e of an activation row (read_row_to_float,
// gten/ops.cpp:41-84): Q8 code * fp16 delta (one exact product), F16
// widened, F32 as is.
template <int ADT>
__device__ __forceinline__ float act_load(const uint8_t* row, int e, int dofs)
{
    if (ADT == Q8) {
        const int8_t q = reinterpret_cast<const int8_t*>(row)[e];
        return (float)q * h2f(reinterpret_cast<const uint16_t*>(row + dofs)[e >> 5]);
    } else if (ADT == F16) {
        return h2f(reinterpret_cast<const uint16_t*>(row)[e]);
    } else {
        return reinterpret_cast<const float*>(row)[e];
    }
}

// write_row_from_float for one element held by this lane (all 32 lanes of
// the block call together; lanes with valid = false skip the store).
template <int ADT>
__device__ __forceinline__ void act_store(uint8_t* row, int e, int dofs, float v, bool valid)
{
    if (ADT == Q8) {
        uint16_t d16;
        const int8_t q = q8_quant_lane(v, valid, &d16);
        if (valid) {
            reinterpret_cast<int8_t*>(row)[e] = q;
            if ((e & 31) == 0) reinterpret_cast<uint16_t*>(row + dofs)[e >> 5] = d16;
        }
    } else if (ADT == F16) {
        if (valid) reinterpret_cast<uint16_t*>(row)[e] = f2h(v);
    } else {
        if (valid) reinterpret_cast<float*>(row)[e] = v;
    }
}

// The value an activation of dtype ADT holds after write + read back.
template <int ADT>
__device__ __forceinline__ float act_roundtrip(float v, bool valid)
{
    if (ADT == Q8) return q8_roundtrip_lane(v, valid);
    if (ADT == F16) return f16_roundtrip(v);
    return v;
}

// ---- eight values per lane --------------------------------------------------
//
// The same per lane for eight consecutive values 8 c .. 8 c + 7 of a row
// whose width is a multiple of 32 (Q8; a block on a quad of lanes, all four
// active) or 8: one 8- or 16-byte access instead of eight, and the block's
// absmax takes seven in-lane maxima and two lane moves instead of five moves
// per value.  Rows must be 16-byte aligned (8 for Q8 rows).

template <int ADT>
__device__ __forceinline__ void act_load8(const uint8_t* row, int c, int dofs, float (&v)[8])
{
    if (ADT == Q8) {
        const uint2 q = reinterpret_cast<const uint2*>(row)[c];
        const float d = h2f(reinterpret_cast<const uint16_t*>(row + dofs)[c >> 2]);
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = (float)(int8_t)((i < 4 ? q.x >> (8 * i) : q.y >> (8 * (i - 4))) & 0xFFu) * d;
    } else if (ADT == F16) {
        const uint4 q = reinterpret_cast<const uint4*>(row)[c];
        const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = h2f((uint16_t)(i & 1 ? w[i >> 1] >> 16 : w[i >> 1] & 0xFFFFu));
    } else {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const float4 q = reinterpret_cast<const float4*>(row)[2 * c + h];
            v[4 * h] = q.x;
            v[4 * h + 1] = q.y;
            v[4 * h + 2] = q.z;
            v[4 * h + 3] = q.w;
        }
    }
}

// q8_quant_lane for a block on four lanes.
__device__ __forceinline__ void q8_quant8(const float (&v)[8], int8_t (&q)[8], uint16_t* d16)
{
    float a = fabsf(v[0]);
#pragma unroll
    for (int i = 1; i < 8; i++) a = fmaxf(a, fabsf(v[i]));
    a = quad_max(a);
    const float delta = a / 127.0f;
    *d16 = f2h(delta);
    const float scale = delta != 0.0f ? 1.0f / delta : 0.0f;
#pragma unroll
    for (int i = 0; i < 8; i++) q[i] = (int8_t)roundf(v[i] * scale);
}

// Writes v; with BACK, v becomes what is read back.
template <int ADT, bool BACK = false>
__device__ __forceinline__ void act_store8(uint8_t* row, int c, int dofs, float (&v)[8])
{
    if (ADT == Q8) {
        int8_t q[8];
        uint16_t d16;
        q8_quant8(v, q, &d16);
        uint32_t w[2] = {0, 0};
#pragma unroll
        for (int i = 0; i < 8; i++) w[i >> 2] |= (uint32_t)(uint8_t)q[i] << (8 * (i & 3));
        reinterpret_cast<uint2*>(row)[c] = make_uint2(w[0], w[1]);
        if ((c & 3) == 0) reinterpret_cast<uint16_t*>(row + dofs)[c >> 2] = d16;
        if (BACK) {
#pragma unroll
            for (int i = 0; i < 8; i++) v[i] = (float)q[i] * h2f(d16);
        }
    } else if (ADT == F16) {
        uint32_t w[4];
#pragma unroll
        for (int i = 0; i < 4; i++) w[i] = (uint32_t)f2h(v[2 * i]) | (uint32_t)f2h(v[2 * i + 1]) << 16;
        reinterpret_cast<uint4*>(row)[c] = make_uint4(w[0], w[1], w[2], w[3]);
        if (BACK) {
#pragma unroll
            for (int i = 0; i < 8; i++) v[i] = f16_roundtrip(v[i]);
        }
    } else {
#pragma unroll
        for (int h = 0; h < 2; h++)
            reinterpret_cast<float4*>(row)[2 * c + h] = make_float4(v[4 * h], v[4 * h + 1], v[4 * h + 2], v[4 * h + 3]);
    }
}

// act_roundtrip of the eight values.
template <int ADT>
__device__ __forceinline__ void act_round8(float (&v)[8])
{
    if (ADT == Q8) {
        int8_t q[8];
        uint16_t d16;
        q8_quant8(v, q, &d16);
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = (float)q[i] * h2f(d16);
    } else if (ADT == F16) {
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = f16_roundtrip(v[i]);
    }
}

// (x_j, x_{j+d/2}) -> (x_j cos - x_{j+d/2} sin, x_j sin + x_{j+d/2} cos) on
// the first d_r dims of a 64-wide head held one value per lane.
__device__ __forceinline__ float rope_lane(float x, int lane, int d_half, const float2* cs)
{
    const int d_r = 2 * d_half;
    const int partner = lane < d_half ? lane + d_half : (lane < d_r ? lane - d_half : lane);
    const float xp = __shfl(x, partner);
    if (lane < d_half) {
        const float2 t = cs[lane];
        return x * t.x - xp * t.y;
    }
    if (lane < d_r) {
        const float2 t = cs[lane - d_half];
        return xp * t.y + x * t.x;
    }
    return x;
}

// The same with the lane's (cos, sin) pair already loaded (cs[lane] for
// lane < d_half, cs[lane - d_half] for d_half <= lane < 2 d_half).
__device__ __forceinline__ float rope_lane_pair(float x, int lane, int d_half, float2 t)
{
    const int d_r = 2 * d_half;
    const int partner = lane < d_half ? lane + d_half : (lane < d_r ? lane - d_half : lane);
    const float xp = __shfl(x, partner);
    if (lane < d_half) return x * t.x - xp * t.y;
    if (lane < d_r) return xp * t.y + x * t.x;
    return x;
}

// Code of element e (0..31) in a lane-permuted weight block (see
// nc_layout.h): dword index and byte position of the element.
__device__ __forceinline__ int wblock_byte_pos(int e) { return (e & 1) + (((e & 15) >> 3) << 1); }

__device__ __forceinline__ int q4_weight_code(const uint32_t* blk, int e)
{
    const int k = (e & 7) >> 1;
    const uint32_t byte = (blk[k] >> (8 * wblock_byte_pos(e))) & 0xFFu;
    return e < 16 ? (int)(byte >> 4) : (int)(byte & 0x0Fu);
}

__device__ __forceinline__ int q8_weight_code(const uint32_t* blk, int e)
{
    const int k = (e & 7) >> 1;
    const uint32_t dw = blk[2 * k + (e >> 4)];
    return (int)(int8_t)((dw >> (8 * wblock_byte_pos(e))) & 0xFFu);
}

// Index (in uint16 units) of (row, col) in the F16 weight layout.
__device__ __forceinline__ size_t f16_weight_index(int row, int col, int npad)
{
    const int g = col >> 6, m = (col >> 3) & 7, j = col & 7;
    return ((((size_t)g * npad + row) * 8 + j) * 8) + m;
}

}  // namespace nc
