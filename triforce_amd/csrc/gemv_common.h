// What the skinny GEMM forms of gemv.hip and gemv_wide.hip share: activation strides, the rotation's arguments, the norm of an operand, shape checks.
#pragma once
#include "common.h"

enum { SG_PLAIN = 0, SG_GATEUP = 1, SG_F32 = 2, SG_QKV = 3 };

// Element (m, k) of an activation block at base[m * sm + (k / 8) * sk + (k % 8)].
struct SgAct {
    int64_t sm, sk;
};

struct SgRope {                       // arguments of the RoPE + KV-append epilogue (SG_QKV)
    const h16* cosb;                  // [max_pos][D] fp16
    const h16* sinb;
    const int64_t* positions;         // [M]
    h16* q_out;                       // [M][H][D]
    h16* k_cache;                     // layer base, element strides below
    h16* v_cache;
    int64_t stride_t, stride_h;
    const int32_t* slot0_dev;
    int slot0, H, D, rotate_k;
};

// h = w_ln * fp16(x * inv): the cast precedes the weight multiply (modeling_llama.py:141-143); the fp16 product of
// two fp16 values rounded once is the native half multiply.
__device__ __forceinline__ half8 sg_normalise(half8 xv, half8 wv, float inv) {
    half8 o;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = (h16)((float)xv[e] * inv);
    return wv * o;
}

static bool sg_act_ok(const SgAct& s) { return s.sm > 0 && s.sk > 0 && (s.sm % 8) == 0 && (s.sk % 8) == 0; }

static bool sg_shape_ok(int M, int N, int K, const SgAct& xa) {
    return M >= 1 && M <= 32 && N >= 16 && (N % 16) == 0 && K >= 32 && (K % 32) == 0 && sg_act_ok(xa) &&
           xa.sm <= 0x7fffffff && xa.sk <= 0x7fffffff;     // (the kernel takes x's two strides as 32-bit arguments)
}
