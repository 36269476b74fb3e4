// Pieces shared by the decode-shape kernels (trmoe_skinny.hip, trmoe_decode8.hip).
#pragma once

#include "trmoe_common.h"
#include "trmoe_gemm.h"

namespace trmoe {

// 16x16 MFMA tiles: a K group is 64 bytes of an activation row; lane l
// supplies row l & 15 and the 16-byte chunk l >> 4 of the group (one
// instruction touches 16 rows x 64 contiguous bytes of each operand).
// Output element i of lane l is row 4 * (l >> 4) + i, column l & 15.
__device__ __forceinline__ void mfma16(KindBF16, u32x4 a, u32x4 b, f32x4& acc) {
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), acc,
                                                  0, 0, 0);
}
__device__ __forceinline__ void mfma16(KindF32, u32x4 a, u32x4 b, f32x4& acc) {
    const f32x4 fa = __builtin_bit_cast(f32x4, a);
    const f32x4 fb = __builtin_bit_cast(f32x4, b);
#pragma unroll
    for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[i], fb[i], acc, 0, 0, 0);
}

// One direct buffer -> LDS load of 16 bytes per lane (lane l's bytes land at
// lds + 16 l).  A plain function: the host pass of hipcc rejects a second
// use of a function template specialization that calls the builtin itself.
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t r, char* lds, int off) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, TRMOE_LDS_PTR(lds), 16, off, 0, 0, 0);
}

// Device-scope accesses of split partials: they pass the XCD's own L2, so a
// workgroup of another XCD sees them without a cache write-back.
__device__ __forceinline__ void store_dev(float* p, float v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float load_dev(const float* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// True for every thread of the last of `n` workgroups to arrive at *count,
// after the partials each stored with store_dev (and before reading them).
__device__ __forceinline__ bool last_arrival(int* count, int n) {
    __shared__ int s_last;
    // this wave's partials have reached memory before the count that says so
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0)
        s_last = __hip_atomic_fetch_add(count, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == n - 1;
    __syncthreads();
    return s_last != 0;
}

// red[wave][e][lane] with e = (tm*NU+u)*4+i.
template <int MT, int NU>
__device__ __forceinline__ void skinny_stash(float* red, const f32x4 (&acc)[MT][NU]) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
    for (int tm = 0; tm < MT; ++tm)
#pragma unroll
        for (int u = 0; u < NU; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i) red[((wave * MT * NU + tm * NU + u) * 4 + i) * 64 + lane] = acc[tm][u][i];
}

template <int MT, int NU, int NW>
__device__ __forceinline__ float skinny_sum(const float* red, int tm, int u, int i, int lane) {
    float s = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) s += red[((w * MT * NU + tm * NU + u) * 4 + i) * 64 + lane];
    return s;
}

template <int MT, int NU>
__device__ __forceinline__ void zero_acc16(f32x4 (&acc)[MT][NU]) {
#pragma unroll
    for (int tm = 0; tm < MT; ++tm)
#pragma unroll
        for (int u = 0; u < NU; ++u) acc[tm][u] = f32x4{0.f, 0.f, 0.f, 0.f};
}

// The down epilogue for one output element: row scale, shared scale, the
// route-weighted y rows of the token, the residual.
template <class T>
__device__ __forceinline__ void down_finish(const DownArgs& a, int64_t row, int64_t col, float s) {
    float v = s * a.shared_scale * (a.w_scale ? a.w_scale[col] : 1.0f);
    if (a.y != nullptr) {
        const T* y = static_cast<const T*>(a.y);
        const int64_t last = (int64_t)a.top_k * a.M - 1;
        float racc = 0.f;
        for (int j = 0; j < a.top_k; ++j) {
            int64_t yr = a.inverse[(int64_t)j * a.M + row];
            yr = yr < 0 ? 0 : (yr > last ? last : yr);
            racc += a.rw[j] * to_f32(y[yr * a.ldy + col]);
        }
        v += a.routed_scale * racc;
    }
    if (a.residual != nullptr) v += to_f32(static_cast<const T*>(a.residual)[row * a.ldr + col]);
    static_cast<T*>(a.out)[row * a.ldo + col] = from_f32<T>(v);
}


}  // namespace trmoe
