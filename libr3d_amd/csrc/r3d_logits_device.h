/* r3d_logits_device.h -- device helpers shared by the two walks of logits_gemm_e4m3
 * (r3d_logits.hip, r3d_logits_wide.h): the exact e4m3 -> bf16 widening, scale elements at
 * every dtype, and the check of the device's header against the host's plan. */
#ifndef R3D_LOGITS_DEVICE_H
#define R3D_LOGITS_DEVICE_H

#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>

#include <stddef.h>

#include "r3d_device.h"
#include "r3d_gemm_any.h"
#include "r3d_plan.h"
#include "rad_planes.h"

namespace r3d {

typedef __bf16 lg_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 lg_bf16x2 __attribute__((ext_vector_type(2)));

/* Eight e4m3 codes (two dwords, byte 0 first) -> eight bf16, exact. */
__device__ __forceinline__ lg_bf16x8 lg_codes8(int w0, int w1) {
    const lg_bf16x2 p0 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((unsigned)w0, 1.0f, false);
    const lg_bf16x2 p1 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((unsigned)w0, 1.0f, true);
    const lg_bf16x2 p2 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((unsigned)w1, 1.0f, false);
    const lg_bf16x2 p3 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((unsigned)w1, 1.0f, true);
    return lg_bf16x8{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
}

/* One scale element (bf16, f16 or f32 by SDT 0/1/2) at byte `off` of the plane, widened
 * exactly; an offset past the plane reads 0. */
template <int SDT>
__device__ __forceinline__ float lg_scale(__amdgpu_buffer_rsrc_t rs, uint32_t off) {
    if (SDT == 2) return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, (int)off, 0, 0));
    const uint32_t v = __builtin_amdgcn_raw_buffer_load_b16(rs, (int)off, 0, 0);
    if (SDT == 0) return __uint_as_float(v << 16);
    return __half2float(__ushort_as_half((unsigned short)v));
}

/* One scale element at any alignment (the dword walk): widened exactly. */
template <int SDT>
__device__ __forceinline__ float lg_scale_any(const AnyBuf& b, uint32_t off) {
    const uint32_t v = any_ld4(b, off);
    if (SDT == 2) return __uint_as_float(v);
    if (SDT == 0) return __uint_as_float(v << 16);
    return __half2float(__ushort_as_half((unsigned short)(v & 0xFFFFu)));
}

/* The device copy of the header still describes the planes the host planned from.  Read
 * by aligned dwords (the blob may start at any byte). */
__device__ __forceinline__ bool lg_header_ok(const LogitsGuard& g) {
    const int ne = (g.ic > g.is ? g.ic : g.is) + 1;
    const uint32_t eb = (uint32_t)sizeof(RadPlanesHeader), es = (uint32_t)sizeof(RadPlanesEntry);
    const AnyBuf hb = any_buf(g.header, eb + es * ne);
    auto u32 = [&](uint32_t o) { return any_ld4(hb, o); };
    auto i64 = [&](uint32_t o) {
        return (int64_t)((uint64_t)any_ld4(hb, o) | ((uint64_t)any_ld4(hb, o + 4) << 32));
    };
    if (u32(offsetof(RadPlanesHeader, magic)) != RAD_PLANES_MAGIC ||
        u32(offsetof(RadPlanesHeader, n_planes)) != 2)
        return false;
    const uint32_t c = eb + es * g.ic, s = eb + es * g.is;
    return u32(c + offsetof(RadPlanesEntry, dtype)) == RAD_F8E4M3 &&
           i64(c + offsetof(RadPlanesEntry, offset)) == g.c_off &&
           i64(c + offsetof(RadPlanesEntry, rows)) == g.c_rows &&
           i64(c + offsetof(RadPlanesEntry, cols)) == g.c_cols &&
           u32(s + offsetof(RadPlanesEntry, dtype)) == g.s_dtype &&
           i64(s + offsetof(RadPlanesEntry, offset)) == g.s_off &&
           i64(s + offsetof(RadPlanesEntry, rows)) == g.s_rows &&
           i64(s + offsetof(RadPlanesEntry, row_bytes)) == g.s_row_bytes &&
           i64(s + offsetof(RadPlanesEntry, block)) == g.s_br;
}

constexpr uint32_t kLgOob = 0x80000000u;     /* past every buffer's num_records: reads 0 */

}  // namespace r3d

#endif /* R3D_LOGITS_DEVICE_H */
