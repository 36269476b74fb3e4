// Weight re-layout into the K-contiguous packed form (trmoe_pack_weight).
//
// A training step repacks every weight it changed, forward and transposed,
// so the pack is on the step's path: it moves each element once in and once
// out and is bound by HBM.  Three kernels, chosen by the source's strides:
//
//   k_pack_rows   the source is contiguous along K (nn.Linear weights):
//                 16-byte copies along each packed row
//   k_pack_tr     the source is contiguous along the output rows (expert
//                 tensors [E, H, W], the backward's transposes): 128 packed
//                 rows x 64 K values go through an LDS tile, so that both
//                 sides move 16 bytes per lane
//   k_pack        any strides, one element per thread
#include "trmoe_common.h"
#include "trmoe_internal.h"
#include "trmoe_gemm.h"

namespace trmoe {

namespace {

// Feature and source of a packed row: GATE_UP interleaves 32 gate and 32 up
// rows, PLAIN keeps the order.
struct PackedRow {
    int64_t feat;
    bool second;   // the row comes from b
};
__device__ __forceinline__ PackedRow packed_row(const PackArgs& p, int64_t row) {
    if (!p.interleave) return {row, false};
    return {(row >> 6) * 32 + (row & 31), (row & 32) != 0};
}

template <class T>
__device__ __forceinline__ void pack_scale(const PackArgs& p, int64_t g, int64_t row) {
    if constexpr (sizeof(T) == 1) {
        const PackedRow r = packed_row(p, row);
        const float* s = r.second ? p.sb : p.sa;
        p.dst_scale[g * p.dst_scale_group_stride + row] =
            r.feat < p.out_features ? s[g * p.scale_group_stride + r.feat] : 0.0f;
    }
}

template <class T>
__global__ __launch_bounds__(256) void k_pack(PackArgs p) {
    const int64_t total = p.groups * p.dst_rows * p.dst_cols;
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
         idx += (int64_t)gridDim.x * blockDim.x) {
        const int64_t col = idx % p.dst_cols;
        const int64_t rowg = idx / p.dst_cols;
        const int64_t row = rowg % p.dst_rows;
        const int64_t g = rowg / p.dst_rows;
        const PackedRow r = packed_row(p, row);
        const T* src = static_cast<const T*>(r.second ? p.b : p.a);
        const bool valid = r.feat < p.out_features && col < p.in_features;
        static_cast<T*>(p.dst)[g * p.dst_group_stride + row * p.dst_ld + col] =
            valid ? src[g * p.s_group + r.feat * p.s_out + col * p.s_in] : T{};
        if (col == 0) pack_scale<T>(p, g, row);
    }
}

// One wave per packed row (s_in == 1; source and destination rows 16-byte
// aligned).
template <class T>
__global__ __launch_bounds__(256) void k_pack_rows(PackArgs p) {
    constexpr int V = 16 / (int)sizeof(T);
    const int lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= p.dst_rows) return;
    const int64_t g = blockIdx.y;
    const PackedRow r = packed_row(p, row);
    const bool live = r.feat < p.out_features;
    const T* src = static_cast<const T*>(r.second ? p.b : p.a) + g * p.s_group + (live ? r.feat : 0) * p.s_out;
    T* dst = static_cast<T*>(p.dst) + g * p.dst_group_stride + row * p.dst_ld;
    for (int64_t c = (int64_t)lane * V; c < p.dst_cols; c += 64 * V) {
        if (c + V <= p.dst_cols && (!live || c + V <= p.in_features)) {
            const u32x4 zero = {0u, 0u, 0u, 0u};
            *reinterpret_cast<u32x4*>(dst + c) = live ? *reinterpret_cast<const u32x4*>(src + c) : zero;
        } else {
            for (int j = 0; j < V && c + j < p.dst_cols; ++j)
                dst[c + j] = live && c + j < p.in_features ? src[c + j] : T{};
        }
    }
    if (lane == 0) pack_scale<T>(p, g, row);
}

constexpr int kTrRows = 128, kTrCols = 64;

// 128 packed rows x 64 K values through LDS (s_out == 1; destination rows
// 16-byte aligned; SRC16: the source's runs along the output rows are too).
// A GATE_UP tile holds 64 gate and 64 up features, 128 contiguous bytes of
// each bf16 source row.
template <class T, bool SRC16>
__global__ __launch_bounds__(256) void k_pack_tr(PackArgs p) {
    constexpr int V = 16 / (int)sizeof(T);
    constexpr int kLd = kTrCols + 4 / (int)sizeof(T);   // a dword of padding: rows start on different banks
    __shared__ T tile[kTrRows * kLd];
    const int64_t r0 = (int64_t)blockIdx.x * kTrRows, c0 = (int64_t)blockIdx.y * kTrCols;
    const int64_t g = blockIdx.z;
    constexpr int kRuns = kTrRows / V;                   // runs of V rows per K value
    for (int i = threadIdx.x; i < kRuns * kTrCols; i += 256) {
        const int run = i % kRuns, c = i / kRuns;
        // a run never straddles a 32-row half (V divides 32)
        const PackedRow r = packed_row(p, r0 + run * V);
        const int64_t col = c0 + c;
        T v[V];
        if (col < p.in_features && r.feat < p.out_features) {
            const T* src = static_cast<const T*>(r.second ? p.b : p.a) + g * p.s_group + r.feat + col * p.s_in;
            if (SRC16 && r.feat + V <= p.out_features) {
                const u32x4 w = *reinterpret_cast<const u32x4*>(src);
                __builtin_memcpy(v, &w, 16);
            } else {
#pragma unroll
                for (int j = 0; j < V; ++j) v[j] = r.feat + j < p.out_features ? src[j] : T{};
            }
        } else {
#pragma unroll
            for (int j = 0; j < V; ++j) v[j] = T{};
        }
#pragma unroll
        for (int j = 0; j < V; ++j) tile[(run * V + j) * kLd + c] = v[j];
    }
    __syncthreads();
    constexpr int kVecs = kTrCols / V;
    for (int i = threadIdx.x; i < kTrRows * kVecs; i += 256) {
        const int c = (i % kVecs) * V, lr = i / kVecs;
        const int64_t row = r0 + lr, col = c0 + c;
        if (row >= p.dst_rows || col >= p.dst_cols) continue;
        T* dst = static_cast<T*>(p.dst) + g * p.dst_group_stride + row * p.dst_ld + col;
        const T* src = tile + lr * kLd + c;
        if (col + V <= p.dst_cols) {
            T v[V];
#pragma unroll
            for (int j = 0; j < V; ++j) v[j] = src[j];
            u32x4 w;
            __builtin_memcpy(&w, v, 16);
            *reinterpret_cast<u32x4*>(dst) = w;
        } else {
            for (int j = 0; col + j < p.dst_cols; ++j) dst[j] = src[j];
        }
    }
    if (blockIdx.y == 0)
        for (int lr = threadIdx.x; lr < kTrRows && r0 + lr < p.dst_rows; lr += 256) pack_scale<T>(p, g, r0 + lr);
}

bool aligned(const void* p, int64_t ld, int64_t group, int64_t groups, int eb) {
    return (reinterpret_cast<uintptr_t>(p) & 15) == 0 && (ld * eb) % 16 == 0 &&
           (groups == 1 || (group * eb) % 16 == 0);
}

template <class T>
int launch_pack_t(const PackArgs& p, hipStream_t stream) {
    constexpr int eb = (int)sizeof(T);
    const bool dst16 = aligned(p.dst, p.dst_ld, p.dst_group_stride, p.groups, eb);
    const int64_t row_blocks = (p.dst_rows + 3) / 4, tile_cols = (p.dst_cols + kTrCols - 1) / kTrCols;
    // The vector forms need 16-byte rows on the destination; grids past the
    // y / z limits (never met by a layer's weights) take the element form.
    if (dst16 && p.s_in == 1 && p.groups <= 65535 && row_blocks < ((int64_t)1 << 31) &&
        aligned(p.a, p.s_out, p.s_group, p.groups, eb) && aligned(p.b, p.s_out, p.s_group, p.groups, eb)) {
        hipLaunchKernelGGL(k_pack_rows<T>, dim3((unsigned)row_blocks, (unsigned)p.groups), dim3(256), 0, stream, p);
    } else if (dst16 && p.s_out == 1 && p.groups <= 65535 && tile_cols <= 65535 &&
               p.dst_rows < ((int64_t)1 << 31)) {
        const dim3 grid((unsigned)((p.dst_rows + kTrRows - 1) / kTrRows), (unsigned)tile_cols, (unsigned)p.groups);
        const bool src16 = aligned(p.a, p.s_in, p.s_group, p.groups, eb) &&
                           aligned(p.b, p.s_in, p.s_group, p.groups, eb);
        if (src16)
            hipLaunchKernelGGL((k_pack_tr<T, true>), grid, dim3(256), 0, stream, p);
        else
            hipLaunchKernelGGL((k_pack_tr<T, false>), grid, dim3(256), 0, stream, p);
    } else {
        int64_t blocks = (p.groups * p.dst_rows * p.dst_cols + 255) / 256;
        if (blocks > 65536) blocks = 65536;
        if (blocks < 1) blocks = 1;
        hipLaunchKernelGGL(k_pack<T>, dim3((unsigned)blocks), dim3(256), 0, stream, p);
    }
    return check_launch("pack_weight");
}

}  // namespace

int launch_pack(const PackArgs& p, hipStream_t stream) {
    if (p.elem_bytes == 1) return launch_pack_t<uint8_t>(p, stream);
    if (p.elem_bytes == 2) return launch_pack_t<uint16_t>(p, stream);
    return launch_pack_t<uint32_t>(p, stream);
}

}  // namespace trmoe
