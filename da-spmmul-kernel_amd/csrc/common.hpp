// common.hpp -- shared device helpers: vector loads/stores along N,
// BF16 widening, block -> XCD remapping.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "wave64.hpp"

namespace dspmm {

constexpr int kBlock = 256;       // 4 wavefronts per workgroup
constexpr int kNumXcd = 8;        // MI355X: 8 XCDs, workgroups dispatched round-robin

// Workgroup b is dispatched to XCD (b % 8).  Renumber so that each XCD
// works on a contiguous range of logical blocks: neighbouring rows of A
// (which share columns of B in banded/stencil matrices) then hit the same
// L2.  A bijection on [0, nblocks) for any nblocks.
__device__ __forceinline__ int xcd_remap(int b, int nblocks) {
    const int per = nblocks / kNumXcd, rem = nblocks % kNumXcd;
    const int x = b % kNumXcd, i = b / kNumXcd;
    return x * per + (x < rem ? x : rem) + i;
}

// ---- dense FP32 vectors along N ----------------------------------------
template <int VW>
__device__ __forceinline__ void load_vec(float (&r)[VW], const float *p) {
    static_assert(VW == 1 || VW == 2 || VW == 4 || VW == 8, "VW");
    if constexpr (VW == 8) {
        const float4 t0 = reinterpret_cast<const float4 *>(p)[0];
        const float4 t1 = reinterpret_cast<const float4 *>(p)[1];
        r[0] = t0.x; r[1] = t0.y; r[2] = t0.z; r[3] = t0.w;
        r[4] = t1.x; r[5] = t1.y; r[6] = t1.z; r[7] = t1.w;
    } else if constexpr (VW == 4) {
        const float4 t = *reinterpret_cast<const float4 *>(p);
        r[0] = t.x; r[1] = t.y; r[2] = t.z; r[3] = t.w;
    } else if constexpr (VW == 2) {
        const float2 t = *reinterpret_cast<const float2 *>(p);
        r[0] = t.x; r[1] = t.y;
    } else {
        r[0] = *p;
    }
}

template <int VW>
__device__ __forceinline__ void store_vec(float *p, const float (&r)[VW]) {
    if constexpr (VW == 8) {
        reinterpret_cast<float4 *>(p)[0] = make_float4(r[0], r[1], r[2], r[3]);
        reinterpret_cast<float4 *>(p)[1] = make_float4(r[4], r[5], r[6], r[7]);
    } else if constexpr (VW == 4) {
        *reinterpret_cast<float4 *>(p) = make_float4(r[0], r[1], r[2], r[3]);
    } else if constexpr (VW == 2) {
        *reinterpret_cast<float2 *>(p) = make_float2(r[0], r[1]);
    } else {
        *p = r[0];
    }
}

// Streaming store (output is written once and not re-read by the kernel):
// keeps C from evicting the gathered dense input from L2 / MALL.
typedef float nt_f4 __attribute__((ext_vector_type(4)));
typedef float nt_f2 __attribute__((ext_vector_type(2)));
template <int VW>
__device__ __forceinline__ void store_vec_nt(float *p, const float (&r)[VW]) {
    if constexpr (VW == 8) {
        nt_f4 t0 = {r[0], r[1], r[2], r[3]};
        nt_f4 t1 = {r[4], r[5], r[6], r[7]};
        __builtin_nontemporal_store(t0, reinterpret_cast<nt_f4 *>(p));
        __builtin_nontemporal_store(t1, reinterpret_cast<nt_f4 *>(p) + 1);
    } else if constexpr (VW == 4) {
        nt_f4 t = {r[0], r[1], r[2], r[3]};
        __builtin_nontemporal_store(t, reinterpret_cast<nt_f4 *>(p));
    } else if constexpr (VW == 2) {
        nt_f2 t = {r[0], r[1]};
        __builtin_nontemporal_store(t, reinterpret_cast<nt_f2 *>(p));
    } else {
        __builtin_nontemporal_store(r[0], p);
    }
}

// ---- dense BF16 vectors along N (FP32 widening is a 16-bit shift) -------
__device__ __forceinline__ float bf16_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __uint_as_float(w & 0xFFFF0000u); }

template <int VW>
__device__ __forceinline__ void load_vec_bf16(float (&r)[VW], const uint16_t *p) {
    static_assert(VW == 1 || VW == 2 || VW == 4 || VW == 8, "VW");
    if constexpr (VW == 8) {
        const uint4 t = *reinterpret_cast<const uint4 *>(p);
        r[0] = bf16_lo(t.x); r[1] = bf16_hi(t.x); r[2] = bf16_lo(t.y); r[3] = bf16_hi(t.y);
        r[4] = bf16_lo(t.z); r[5] = bf16_hi(t.z); r[6] = bf16_lo(t.w); r[7] = bf16_hi(t.w);
    } else if constexpr (VW == 4) {
        const uint2 t = *reinterpret_cast<const uint2 *>(p);
        r[0] = bf16_lo(t.x); r[1] = bf16_hi(t.x); r[2] = bf16_lo(t.y); r[3] = bf16_hi(t.y);
    } else if constexpr (VW == 2) {
        const uint32_t t = *reinterpret_cast<const uint32_t *>(p);
        r[0] = bf16_lo(t); r[1] = bf16_hi(t);
    } else {
        r[0] = __uint_as_float((uint32_t)(*p) << 16);
    }
}

// Typed dense-input accessor: B element type is float or uint16_t (BF16).
template <typename TB, int VW>
__device__ __forceinline__ void load_b(float (&r)[VW], const TB *p) {
    if constexpr (sizeof(TB) == 4) load_vec<VW>(r, reinterpret_cast<const float *>(p));
    else load_vec_bf16<VW>(r, reinterpret_cast<const uint16_t *>(p));
}

// The same on global memory at any element-aligned address.  Global loads and
// stores of 4 to 16 bytes need no natural alignment on gfx950 (the compiler
// emits one instruction either way), so row-major kernels use the widest
// vectors for every nv and leading dimension; see slab_col.
template <typename T, int N, int ALIGN>
struct VecAt {
    typedef T type __attribute__((ext_vector_type(N), aligned(ALIGN)));
};
template <typename TB, int VW>
__device__ __forceinline__ void load_g(float (&r)[VW], const TB *p) {
    if constexpr (VW == 1) {
        load_b<TB, 1>(r, p);
    } else if constexpr (sizeof(TB) == 4) {
        static_assert(VW <= 4, "VW");
        const auto t = *reinterpret_cast<const typename VecAt<float, VW, 4>::type *>(p);
#pragma unroll
        for (int k = 0; k < VW; k++) r[k] = t[k];
    } else if constexpr (VW == 2) {
        typedef uint32_t u32_at2 __attribute__((aligned(2)));
        const uint32_t t = *reinterpret_cast<const u32_at2 *>(p);
        r[0] = bf16_lo(t); r[1] = bf16_hi(t);
    } else {
        const auto t = *reinterpret_cast<const typename VecAt<uint32_t, VW / 2, 2>::type *>(p);
#pragma unroll
        for (int k = 0; k < VW / 2; k++) { r[2 * k] = bf16_lo(t[k]); r[2 * k + 1] = bf16_hi(t[k]); }
    }
}
template <bool NT, int VW>
__device__ __forceinline__ void store_g(float *p, const float (&r)[VW]) {
    if constexpr (VW == 8) {
        store_g<NT, 4>(p, reinterpret_cast<const float (&)[4]>(r[0]));
        store_g<NT, 4>(p + 4, reinterpret_cast<const float (&)[4]>(r[4]));
    } else if constexpr (VW == 1) {
        if constexpr (NT) __builtin_nontemporal_store(r[0], p); else *p = r[0];
    } else {
        using V = typename VecAt<float, VW, 4>::type;
        V t;
#pragma unroll
        for (int k = 0; k < VW; k++) t[k] = r[k];
        if constexpr (NT) __builtin_nontemporal_store(t, reinterpret_cast<V *>(p));
        else *reinterpret_cast<V *>(p) = t;
    }
}

// Sums of rows in parts (CSR_PARTS): the products of nonzeros p .. p + 7 (< p1),
// values in sv and rows of B in b, four FMAs to a part, the parts to two sums in turn.
template <int VW>
__device__ __forceinline__ void add_parts(float (&even)[VW], float (&odd)[VW], const float (&b)[8][VW],
                                          const float *sv, int p, int p1) {
#pragma unroll
    for (int h = 0; h < 2; h++) {
        float part[VW];
#pragma unroll
        for (int k = 0; k < VW; k++) part[k] = 0.f;
#pragma unroll
        for (int u = 4 * h; u < 4 * h + 4; u++) {
            if (p + u < p1) {
                const float a = sv[p + u];
#pragma unroll
                for (int k = 0; k < VW; k++) part[k] = __builtin_fmaf(a, b[u][k], part[k]);
            }
        }
#pragma unroll
        for (int k = 0; k < VW; k++) {
            if (h == 0) even[k] += part[k];
            else odd[k] += part[k];
        }
    }
}

// First column of a lane's VW columns.  Where fewer than VW are left of the
// row (nv >= VW), the last ones of the row: the lane shares columns with its
// neighbour and both write the same values.
template <int VW>
__device__ __forceinline__ int slab_col(int col, int nv) {
    return VW > 1 && col < nv && col + VW > nv ? nv - VW : col;
}

// Streaming (read-once) scalar loads for the sparse operand.
template <typename T>
__device__ __forceinline__ T ld_stream(const T *p) { return __builtin_nontemporal_load(p); }

}  // namespace dspmm
