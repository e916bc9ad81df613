// Device-side building blocks shared by every kernel of the library: element type
// traits, 16-byte vector access, wave64 lane shifts (DPP), SiLU and per-lane weight
// loading.  Written for gfx950 only (64-lane wavefronts, v_cvt_pk_bf16_f32).
//
// Takes over the roles of csrc/causal_conv1d_common.h:46-98 (BytesToType, Allreduce)
// and csrc/static_switch.h:16-25 of the reference, with a different design: one lane
// always owns one 16-byte vector, and cross-lane traffic is a DPP shift by one lane.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "cc1d.h"

namespace cc1d {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

constexpr int kWave = 64;
constexpr int kBlock = 256;  // 4 wavefronts per workgroup

// A divisor as a factor of the quotient's upper word (device.hpp: divided).  For 2^l < d <= 2^(l+1) the factor is
// 2^(32+l) / d rounded up: below 2^32, and off by less than d / 2^(32+l), so exact for every n < 2^31.
struct FastDiv {
    uint32_t mul, shift;                              // mul 0: a division by one
};
inline FastDiv fast_div(uint32_t d) {
    if (d <= 1) return {0, 0};
    const uint32_t l = 31 - (uint32_t)__builtin_clz(d - 1);
    return {(uint32_t)((((uint64_t)1 << (32 + l)) + d - 1) / d), l};
}

template <typename To, typename From>
__device__ __forceinline__ To bitcast(const From &v) {
    return __builtin_bit_cast(To, v);
}

// ---------------------------------------------------------------------------------
// Element traits.  kVec elements make one 16-byte vector.
// ---------------------------------------------------------------------------------
// SiLU for fp32 tensors.  0 (default): v_exp_f32 + v_rcp_f32 as for 16-bit tensors; against a
// float64 reference the forward's largest error on N(0,1) inputs at (4, 2048, 4096) is 7e-7
// (6e-7 with the precise variant: rounding of the fp32 sums dominates both), inside the
// atol 1e-5 fp32 results are held to, and the fp32 kernels run 6-15 % faster.
// 1: expf and a true division.
#ifndef CC1D_F32_PRECISE_ACT
#define CC1D_F32_PRECISE_ACT 0
#endif

template <int DT> struct Elem;

template <> struct Elem<CC1D_F32> {
    using type = float;
    static constexpr int kVec = 4;
    static constexpr int kBytes = 4;
    static constexpr bool kPreciseAct = CC1D_F32_PRECISE_ACT != 0;
    static __device__ __forceinline__ float to_float(float v) { return v; }
    static __device__ __forceinline__ float from_float(float v) { return v; }
    static __device__ __forceinline__ void unpack(const u32x4 &r, float (&f)[4]) {
        f[0] = bitcast<float>(r.x); f[1] = bitcast<float>(r.y);
        f[2] = bitcast<float>(r.z); f[3] = bitcast<float>(r.w);
    }
    static __device__ __forceinline__ u32x4 pack(const float (&f)[4]) {
        u32x4 r;
        r.x = bitcast<uint32_t>(f[0]); r.y = bitcast<uint32_t>(f[1]);
        r.z = bitcast<uint32_t>(f[2]); r.w = bitcast<uint32_t>(f[3]);
        return r;
    }
};

template <> struct Elem<CC1D_F16> {
    using type = _Float16;
    static constexpr int kVec = 8;
    static constexpr int kBytes = 2;
    static constexpr bool kPreciseAct = false;
    static __device__ __forceinline__ float to_float(_Float16 v) { return (float)v; }
    static __device__ __forceinline__ _Float16 from_float(float v) {
        asm("" : "+v"(v));                  // no fused round-to-fp16 multiply (see Pack::pack)
        return (_Float16)v;
    }
    static __device__ __forceinline__ void unpack(const u32x4 &r, float (&f)[8]) {
        const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            f16x2 h = bitcast<f16x2>(w[i]);
            f[2 * i] = (float)h.x;
            f[2 * i + 1] = (float)h.y;
        }
    }
    static __device__ __forceinline__ u32x4 pack(const float (&f)[8]) {
        uint32_t w[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float lo = f[2 * i], hi = f[2 * i + 1];
            asm("" : "+v"(lo), "+v"(hi));     // no fused round-to-fp16 multiply (see Pack::pack)
            f16x2 h;
            h.x = (_Float16)lo;
            h.y = (_Float16)hi;
            w[i] = bitcast<uint32_t>(h);
        }
        u32x4 r; r.x = w[0]; r.y = w[1]; r.z = w[2]; r.w = w[3];
        return r;
    }
};

template <> struct Elem<CC1D_BF16> {
    using type = __bf16;
    static constexpr int kVec = 8;
    static constexpr int kBytes = 2;
    static constexpr bool kPreciseAct = false;
    static __device__ __forceinline__ float to_float(__bf16 v) { return (float)v; }
    static __device__ __forceinline__ __bf16 from_float(float v) { return (__bf16)v; }
    static __device__ __forceinline__ void unpack(const u32x4 &r, float (&f)[8]) {
        const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            f[2 * i] = bitcast<float>(w[i] << 16);
            f[2 * i + 1] = bitcast<float>(w[i] & 0xffff0000u);
        }
    }
    static __device__ __forceinline__ u32x4 pack(const float (&f)[8]) {
        uint32_t w[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            bf16x2 h;                       // round-to-nearest-even: v_cvt_pk_bf16_f32
            h.x = (__bf16)f[2 * i];
            h.y = (__bf16)f[2 * i + 1];
            w[i] = bitcast<uint32_t>(h);
        }
        u32x4 r; r.x = w[0]; r.y = w[1]; r.z = w[2]; r.w = w[3];
        return r;
    }
};

// ---------------------------------------------------------------------------------
// CH channels of one row held by one lane: a 16-byte or an 8-byte register vector.
// ---------------------------------------------------------------------------------
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x1 __attribute__((ext_vector_type(1)));
template <int BYTES> struct RawBytes;
template <> struct RawBytes<16> { using type = u32x4; };
template <> struct RawBytes<8> { using type = u32x2; };
template <> struct RawBytes<4> { using type = u32x1; };

template <int DT, int CH>
struct Pack {
    static constexpr int kBytes = CH * Elem<DT>::kBytes;
    static constexpr int kDwords = kBytes / 4;
    using raw_t = typename RawBytes<kBytes>::type;

    static __device__ __forceinline__ raw_t zero() {
        raw_t r;
#pragma unroll
        for (int i = 0; i < kDwords; ++i) r[i] = 0u;
        return r;
    }
    static __device__ __forceinline__ void unpack(const raw_t &r, float (&f)[CH]) {
        if constexpr (DT == CC1D_F32) {
#pragma unroll
            for (int i = 0; i < kDwords; ++i) f[i] = bitcast<float>(r[i]);
        } else if constexpr (DT == CC1D_BF16) {
#pragma unroll
            for (int i = 0; i < kDwords; ++i) {
                f[2 * i] = bitcast<float>(r[i] << 16);
                f[2 * i + 1] = bitcast<float>(r[i] & 0xffff0000u);
            }
        } else {
#pragma unroll
            for (int i = 0; i < kDwords; ++i) {
                const f16x2 h = bitcast<f16x2>(r[i]);
                f[2 * i] = (float)h.x;
                f[2 * i + 1] = (float)h.y;
            }
        }
    }
    static __device__ __forceinline__ raw_t pack(const float (&f)[CH]) {
        raw_t r;
        if constexpr (DT == CC1D_F32) {
#pragma unroll
            for (int i = 0; i < kDwords; ++i) r[i] = bitcast<uint32_t>(f[i]);
        } else if constexpr (DT == CC1D_BF16) {
#pragma unroll
            for (int i = 0; i < kDwords; ++i) {
                bf16x2 h;                   // round-to-nearest-even: v_cvt_pk_bf16_f32
                h.x = (__bf16)f[2 * i];
                h.y = (__bf16)f[2 * i + 1];
                r[i] = bitcast<uint32_t>(h);
            }
        } else {
#pragma unroll
            for (int i = 0; i < kDwords; ++i) {
                // The empty asm keeps the compiler from folding the producing multiply
                // into a mixed-precision fma that rounds to fp16 in one step: with it every
                // code path rounds fp32 -> fp16 the same way and gives the same bits.
                float lo = f[2 * i], hi = f[2 * i + 1];
                asm("" : "+v"(lo), "+v"(hi));
                f16x2 h;
                h.x = (_Float16)lo;
                h.y = (_Float16)hi;
                r[i] = bitcast<uint32_t>(h);
            }
        }
        return r;
    }
};

// ---------------------------------------------------------------------------------
// Global memory access.  Offsets are element offsets, always 64-bit.
// ---------------------------------------------------------------------------------
template <int DT>
__device__ __forceinline__ u32x4 ld_vec(const void *base, int64_t elem_off) {
    using T = typename Elem<DT>::type;
    return *reinterpret_cast<const u32x4 *>(reinterpret_cast<const T *>(base) + elem_off);
}
template <int DT>
__device__ __forceinline__ void st_vec(void *base, int64_t elem_off, const u32x4 &v) {
    using T = typename Elem<DT>::type;
    *reinterpret_cast<u32x4 *>(reinterpret_cast<T *>(base) + elem_off) = v;
}
// Streaming variants: data that is touched once should not displace the L2 contents.
template <int DT>
__device__ __forceinline__ u32x4 ld_vec_nt(const void *base, int64_t elem_off) {
    using T = typename Elem<DT>::type;
    return __builtin_nontemporal_load(
        reinterpret_cast<const u32x4 *>(reinterpret_cast<const T *>(base) + elem_off));
}
template <int DT>
__device__ __forceinline__ void st_vec_nt(void *base, int64_t elem_off, const u32x4 &v) {
    using T = typename Elem<DT>::type;
    __builtin_nontemporal_store(
        v, reinterpret_cast<u32x4 *>(reinterpret_cast<T *>(base) + elem_off));
}
// How the short-row kernels (channel-first rows of at most 64 vectors) move a row: as whole vectors on the 16-byte
// grid, as vectors of any address (rows of a vector and more), or element by element.
enum ShortRows : int { kWhole, kAnywhere, kElements };
// A vector that starts at any element: one access wherever the address lies.
typedef uint32_t u32x4_on2 __attribute__((ext_vector_type(4), aligned(2)));
typedef uint32_t u32x4_on4 __attribute__((ext_vector_type(4), aligned(4)));
template <int DT>
__device__ __forceinline__ u32x4 ld_vec_any(const void *base, int64_t elem_off) {
    using T = typename Elem<DT>::type;
    const T *at = reinterpret_cast<const T *>(base) + elem_off;
    if constexpr (sizeof(T) == 2) return *reinterpret_cast<const u32x4_on2 *>(at);
    else return *reinterpret_cast<const u32x4_on4 *>(at);
}
// The first n elements (a whole vector or fewer) of v to any element: a vector's front part as one store each
// of 8, 4 and 2 bytes.  n_front is the same for every lane that stores a front part, so its bits are branches of
// the wavefront.
template <int DT>
__device__ __forceinline__ void st_front_any(void *base, int64_t elem_off, const u32x4 &v, bool whole, int n_front) {
    using T = typename Elem<DT>::type;
    typedef uint32_t u32_on2 __attribute__((aligned(2)));
    typedef uint32_t u32x2_on2 __attribute__((ext_vector_type(2), aligned(2)));
    T *at = reinterpret_cast<T *>(base) + elem_off;
    if (whole) {
        if constexpr (sizeof(T) == 2) *reinterpret_cast<u32x4_on2 *>(at) = v;
        else *reinterpret_cast<u32x4_on4 *>(at) = v;
        return;
    }
    const int bytes = n_front * (int)sizeof(T);
    char *to = reinterpret_cast<char *>(at);
    uint32_t next = v.x, after = v.y;
    if (bytes & 8) {
        *reinterpret_cast<u32x2_on2 *>(to) = u32x2_on2{v.x, v.y};
        to += 8;
        next = v.z;
        after = v.w;
    }
    if (bytes & 4) {
        *reinterpret_cast<u32_on2 *>(to) = next;
        to += 4;
        next = after;
    }
    if (sizeof(T) == 2 && (bytes & 2)) *reinterpret_cast<uint16_t *>(to) = (uint16_t)next;
}
// v without its first `bytes` bytes (0 .. 14, even), zeros behind the rest.
__device__ __forceinline__ u32x4 without_front(const u32x4 &v, int bytes) {
    const uint32_t x = v.x, y = v.y, z = v.z, w = v.w;   // values: an array here would be chosen from by address, in memory
    const bool two = (bytes & 8) != 0, one = (bytes & 4) != 0, half = (bytes & 2) != 0;
    const uint32_t a0 = two ? z : x, a1 = two ? w : y, a2 = two ? 0u : z, a3 = two ? 0u : w;
    const uint32_t b0 = one ? a1 : a0, b1 = one ? a2 : a1, b2 = one ? a3 : a2, b3 = one ? 0u : a3;
    return u32x4{half ? __builtin_amdgcn_alignbit(b1, b0, 16) : b0, half ? __builtin_amdgcn_alignbit(b2, b1, 16) : b1,
                 half ? __builtin_amdgcn_alignbit(b3, b2, 16) : b2, half ? b3 >> 16 : b3};
}
template <int DT>
__device__ __forceinline__ float ld_elem(const void *base, int64_t elem_off) {
    using T = typename Elem<DT>::type;
    return Elem<DT>::to_float(reinterpret_cast<const T *>(base)[elem_off]);
}
template <int DT>
__device__ __forceinline__ void st_elem(void *base, int64_t elem_off, float v) {
    using T = typename Elem<DT>::type;
    reinterpret_cast<T *>(base)[elem_off] = Elem<DT>::from_float(v);
}
// Bit-preserving element copy (state shifts and gathers must be exact).
template <int DT>
__device__ __forceinline__ typename Elem<DT>::type ld_raw(const void *base, int64_t elem_off) {
    using T = typename Elem<DT>::type;
    return reinterpret_cast<const T *>(base)[elem_off];
}
template <int DT>
__device__ __forceinline__ void st_raw(void *base, int64_t elem_off, typename Elem<DT>::type v) {
    using T = typename Elem<DT>::type;
    reinterpret_cast<T *>(base)[elem_off] = v;
}

// Weight / bias element of runtime type `w_dtype`, as fp32.
__device__ __forceinline__ float ld_weight(const void *base, int w_dtype, int64_t elem_off) {
    if (w_dtype == CC1D_F32) return reinterpret_cast<const float *>(base)[elem_off];
    if (w_dtype == CC1D_F16) return (float)reinterpret_cast<const _Float16 *>(base)[elem_off];
    return (float)reinterpret_cast<const __bf16 *>(base)[elem_off];
}

// Weights and bias of NCH consecutive channels starting at c0 into registers.
// contiguous_f32 is a host-checked promise: fp32, strides (W, 1), 16-byte aligned base;
// then NCH*W consecutive floats are fetched as 16-byte vectors.
template <int W, int NCH>
__device__ __forceinline__ void load_weights(const void *weight, const void *bias, int w_dtype,
                                             int64_t stride_c, int64_t stride_w,
                                             bool contiguous_f32, int c0,
                                             float (&wv)[NCH][W], float (&bv)[NCH]) {
    if (contiguous_f32) {
        // NCH*W consecutive floats starting at a multiple of NCH floats: the compiler
        // merges them into the widest loads the alignment allows.
        constexpr int kAlign = NCH * 4 > 16 ? 16 : NCH * 4;
        const float *src = static_cast<const float *>(__builtin_assume_aligned(
            reinterpret_cast<const float *>(weight) + (int64_t)c0 * W, kAlign));
        float flat[NCH * W];
#pragma unroll
        for (int i = 0; i < NCH * W; ++i) flat[i] = src[i];
#pragma unroll
        for (int j = 0; j < NCH; ++j)
#pragma unroll
            for (int w = 0; w < W; ++w) wv[j][w] = flat[j * W + w];
    } else {
#pragma unroll
        for (int j = 0; j < NCH; ++j)
#pragma unroll
            for (int w = 0; w < W; ++w)
                wv[j][w] = ld_weight(weight, w_dtype, (int64_t)(c0 + j) * stride_c + w * stride_w);
    }
#pragma unroll
    for (int j = 0; j < NCH; ++j)
        bv[j] = bias == nullptr ? 0.f : ld_weight(bias, w_dtype, c0 + j);
}

// Taps and bias of NCH adjacent channels stored packed (dim, W) / (dim,) with element type
// WDT, base pointers 16-byte aligned (a host-checked promise).  request() issues plain vector
// loads into raw registers and uses none of the values, so a caller can queue further loads
// behind it; finish() turns the raw bits into fp32.
template <int W, int NCH, int WDT>
struct PackedTaps {
    static constexpr int kN = NCH * W;
    static constexpr bool k32 = WDT == CC1D_F32;
    static constexpr int kWords = k32 ? kN : kN / 2;
    static constexpr int kBiasWords = k32 ? NCH : NCH / 2;
    uint32_t wraw[kWords];
    uint32_t braw[kBiasWords];
    static_assert(k32 || NCH % 2 == 0, "two 16-bit taps per word");

    static constexpr int pow2_align(int bytes) { return bytes % 16 == 0 ? 16 : bytes % 8 == 0 ? 8 : 4; }

    __device__ __forceinline__ void request(const void *weight, const void *bias, int c0) {
        constexpr int kElem = k32 ? 4 : 2;
        const char *wbase = reinterpret_cast<const char *>(weight) + (int64_t)c0 * W * kElem;
        const uint32_t *src = static_cast<const uint32_t *>(__builtin_assume_aligned(wbase, pow2_align(kN * kElem)));
#pragma unroll
        for (int i = 0; i < kWords; ++i) wraw[i] = src[i];
        // Without a bias the taps are read a second time in its place: the load stays
        // unconditional; finish() discards it.
        const char *bbase = bias != nullptr ? reinterpret_cast<const char *>(bias) + (int64_t)c0 * kElem : wbase;
        const uint32_t *bsrc = static_cast<const uint32_t *>(__builtin_assume_aligned(bbase, pow2_align(NCH * kElem)));
#pragma unroll
        for (int j = 0; j < kBiasWords; ++j) braw[j] = bsrc[j];
    }

    static __device__ __forceinline__ float element(const uint32_t *words, int i) {
        if constexpr (k32) {
            return bitcast<float>(words[i]);
        } else if constexpr (WDT == CC1D_BF16) {
            return bitcast<float>(i % 2 ? (words[i / 2] & 0xffff0000u) : (words[i / 2] << 16));
        } else {
            const f16x2 h = bitcast<f16x2>(words[i / 2]);
            return i % 2 ? (float)h.y : (float)h.x;
        }
    }

    __device__ __forceinline__ void finish(bool has_bias, float (&wv)[NCH][W], float (&bv)[NCH]) {
        // Pins the first use of the raw words to this point of the program: without it the
        // compiler converts them right behind their loads and waits there.
#pragma unroll
        for (int i = 0; i < kWords; ++i) asm volatile("" : "+v"(wraw[i]));
#pragma unroll
        for (int j = 0; j < kBiasWords; ++j) asm volatile("" : "+v"(braw[j]));
#pragma unroll
        for (int i = 0; i < kN; ++i) wv[i / W][i % W] = element(wraw, i);
#pragma unroll
        for (int j = 0; j < NCH; ++j) bv[j] = has_bias ? element(braw, j) : 0.f;
    }
};

// The same two-phase protocol for taps of any stride and of runtime element type (fp32, fp16,
// bf16): request() fetches each tap and bias element as raw bits (one 4- or 2-byte load each,
// under a branch on the type that is uniform for the launch) and uses none of them; finish()
// converts.
template <int W, int NCH>
struct StridedTaps {
    uint32_t wraw[NCH * W];
    uint32_t braw[NCH];

    __device__ __forceinline__ void request(const void *weight, const void *bias, int w_dtype, int64_t stride_c,
                                            int64_t stride_w, int c0) {
        if (w_dtype == CC1D_F32) {
            const uint32_t *wp = reinterpret_cast<const uint32_t *>(weight);
            const uint32_t *bp = reinterpret_cast<const uint32_t *>(bias != nullptr ? bias : weight);
#pragma unroll
            for (int j = 0; j < NCH; ++j) {
#pragma unroll
                for (int w = 0; w < W; ++w) wraw[j * W + w] = wp[(int64_t)(c0 + j) * stride_c + w * stride_w];
                braw[j] = bias != nullptr ? bp[c0 + j] : 0u;
            }
        } else {
            const uint16_t *wp = reinterpret_cast<const uint16_t *>(weight);
            const uint16_t *bp = reinterpret_cast<const uint16_t *>(bias != nullptr ? bias : weight);
#pragma unroll
            for (int j = 0; j < NCH; ++j) {
#pragma unroll
                for (int w = 0; w < W; ++w) wraw[j * W + w] = wp[(int64_t)(c0 + j) * stride_c + w * stride_w];
                braw[j] = bias != nullptr ? bp[c0 + j] : 0u;
            }
        }
    }
    static __device__ __forceinline__ float as_float(uint32_t bits, int w_dtype) {
        if (w_dtype == CC1D_F32) return bitcast<float>(bits);
        if (w_dtype == CC1D_BF16) return bitcast<float>(bits << 16);
        return (float)bitcast<_Float16>((uint16_t)bits);
    }
    __device__ __forceinline__ void finish(int w_dtype, bool has_bias, float (&wv)[NCH][W], float (&bv)[NCH]) {
#pragma unroll
        for (int i = 0; i < NCH * W; ++i) asm volatile("" : "+v"(wraw[i]));
#pragma unroll
        for (int j = 0; j < NCH; ++j) asm volatile("" : "+v"(braw[j]));
#pragma unroll
        for (int i = 0; i < NCH * W; ++i) wv[i / W][i % W] = as_float(wraw[i], w_dtype);
#pragma unroll
        for (int j = 0; j < NCH; ++j) bv[j] = has_bias ? as_float(braw[j], w_dtype) : 0.f;
    }
};

// Taps and bias of one channel as fp32, any strides and type.  One branch on the type for all of them:
// with a branch per element each load waits for everything in flight before the next is issued, five
// waits in a row.  Taps of 16 bits, bf16 data, channel-first: backward (16, 4096, 1001) 116 -> 82 us,
// see cc1d_fwd_channelfirst_tile.hip for the forward.
template <int W>
__device__ __forceinline__ void channel_taps(const void *weight, const void *bias, int w_dtype, int64_t stride_c,
                                             int64_t stride_w, int c, float (&wv)[W], float &bv) {
    if (w_dtype == CC1D_F32) {
        const float *wp = reinterpret_cast<const float *>(weight) + (int64_t)c * stride_c;
#pragma unroll
        for (int w = 0; w < W; ++w) wv[w] = wp[(int64_t)w * stride_w];
        bv = bias != nullptr ? reinterpret_cast<const float *>(bias)[c] : 0.f;
    } else {
        uint16_t raw[W + 1];
        const uint16_t *wp = reinterpret_cast<const uint16_t *>(weight) + (int64_t)c * stride_c;
#pragma unroll
        for (int w = 0; w < W; ++w) raw[w] = wp[(int64_t)w * stride_w];
        raw[W] = bias != nullptr ? reinterpret_cast<const uint16_t *>(bias)[c] : (uint16_t)0;
        const bool bf16 = w_dtype == CC1D_BF16;
#pragma unroll
        for (int w = 0; w < W; ++w) wv[w] = bf16 ? bitcast<float>((uint32_t)raw[w] << 16) : (float)bitcast<_Float16>(raw[w]);
        bv = bf16 ? bitcast<float>((uint32_t)raw[W] << 16) : (float)bitcast<_Float16>(raw[W]);
    }
}
// The same for a channel that all lanes of the wavefront share: the values end in scalar registers.
template <int W>
__device__ __forceinline__ void uniform_taps(const void *weight, const void *bias, int w_dtype, int64_t stride_c,
                                             int64_t stride_w, int c, float (&wv)[W], float &bv) {
    channel_taps<W>(weight, bias, w_dtype, stride_c, stride_w, c, wv, bv);
#pragma unroll
    for (int w = 0; w < W; ++w) wv[w] = bitcast<float>(__builtin_amdgcn_readfirstlane(bitcast<int>(wv[w])));
    bv = bitcast<float>(__builtin_amdgcn_readfirstlane(bitcast<int>(bv)));
}

// ---------------------------------------------------------------------------------
// Wave64 lane shifts through DPP (no LDS, no memory).  All 64 lanes must be active.
//   from_prev_lane: lane i receives lane i-1's value, lane 0 receives `lane0_fill`.
//   from_next_lane: lane i receives lane i+1's value, lane 63 receives `lane63_fill`.
// ---------------------------------------------------------------------------------
__device__ __forceinline__ float from_prev_lane(float v, float lane0_fill) {
    return bitcast<float>(__builtin_amdgcn_update_dpp(
        bitcast<int>(lane0_fill), bitcast<int>(v), 0x138 /* wave_shr:1 */, 0xf, 0xf, false));
}
__device__ __forceinline__ float from_next_lane(float v, float lane63_fill) {
    return bitcast<float>(__builtin_amdgcn_update_dpp(
        bitcast<int>(lane63_fill), bitcast<int>(v), 0x130 /* wave_shl:1 */, 0xf, 0xf, false));
}
__device__ __forceinline__ float read_lane(float v, int lane) {
    return bitcast<float>(__builtin_amdgcn_readlane(bitcast<int>(v), lane));
}
// Every vector-memory load this wavefront has issued so far has returned.  Used in front of the
// final_states stores of the forward kernels: final_states may be the very buffer initial_states
// were read from (a chunked prefill that keeps one state tensor), the wavefront that reads a
// row's initial_states is the one that writes its final_states, and with this wait the reads are
// complete before the first such store is issued.
__device__ __forceinline__ void wait_for_loads() {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// Sum over the 64 lanes of a wave in a fixed butterfly order (deterministic).
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, kWave);
    return v;
}

// The W + 1 sums of a channel (dweight's terms and dbias') over the 64 lanes, all at once: lane w < W ends
// with the total of dW[w], lane 4 with dB's.  Values that share a register from a step on halve the work
// that is left, 19 instructions for five sums where one after the other takes 47, and the results lie in
// lanes of their own, so one store writes them all.  Fixed order: bit-reproducible.  Backward, us before /
// after: rows of one wavefront (16, 512, 256) bf16 5.9 / 5.4, (8, 1536, 64) fp16 5.3 / 4.9, (4, 1024, 300) 8.1 / 7.8 (their sums went
// through LDS lane by lane); tiles (16, 4096, 1025) 76.9 / 75.4, (16, 4096, 1001) 74.1 / 73.7.
template <int CTRL>
__device__ __forceinline__ float dpp_moved(float v) {
    return bitcast<float>(__builtin_amdgcn_update_dpp(0, bitcast<int>(v), CTRL, 0xf, 0xf, true));
}
// Lanes with `second` set go on with b, the others with a, each plus what the lane at the other end of the DPP move has of it.
template <int CTRL>
__device__ __forceinline__ float folded(float a, float b, bool second) {
    return (second ? b : a) + dpp_moved<CTRL>(second ? a : b);
}
template <int W>
__device__ __forceinline__ float wave_sums(const float (&dW)[W], float dB, int lane) {
    constexpr int kXor1 = 0xB1, kXor2 = 0x4E, kRor4 = 0x124, kRor8 = 0x128;      // quad_perm, quad_perm, row_ror, row_ror
    const float low = folded<kXor1>(dW[0], dW[1], (lane & 1) != 0);
    const float high = W > 2 ? folded<kXor1>(dW[W > 2 ? 2 : 0], W > 3 ? dW[W > 3 ? 3 : 0] : 0.f, (lane & 1) != 0) : 0.f;
    const float four = folded<kXor2>(low, high, (lane & 2) != 0);                // lane & 3: which of dW, over quads
    dB += dpp_moved<kXor1>(dB);
    dB += dpp_moved<kXor2>(dB);
    float v = folded<kRor4>(four, dB, (lane & 4) != 0);                          // in a row of 16 lanes 4 away is the other kind
    v += dpp_moved<kRor8>(v);
    const auto rows = __builtin_amdgcn_permlane16_swap(bitcast<uint32_t>(v), bitcast<uint32_t>(v), false, false);
    v = bitcast<float>((uint32_t)rows[0]) + bitcast<float>((uint32_t)rows[1]);
    const auto halves = __builtin_amdgcn_permlane32_swap(bitcast<uint32_t>(v), bitcast<uint32_t>(v), false, false);
    return bitcast<float>((uint32_t)halves[0]) + bitcast<float>((uint32_t)halves[1]);
}

// n / d for a d that the host knows (fast_div): two scalar instructions for wave-uniform numbers instead of
// two dozen with a reciprocal among them, in front of a wavefront's first request.  n < 2^31.
__device__ __forceinline__ uint32_t divided(uint32_t n, const FastDiv &d) {
    return d.mul == 0 ? n : __umulhi(n, d.mul) >> d.shift;
}

// ---------------------------------------------------------------------------------
// Activation.
// ---------------------------------------------------------------------------------
template <bool PRECISE>
__device__ __forceinline__ float sigmoid(float z) {
    if (PRECISE) {
        return 1.0f / (1.0f + expf(-z));
    } else {
        // v_exp_f32 + v_rcp_f32: about 2 ulp, far inside the 16-bit output rounding.
        return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(z * -1.4426950408889634f));
    }
}
template <bool PRECISE>
__device__ __forceinline__ float silu(float z) {
    if (PRECISE) {
        return z / (1.0f + expf(-z));
    } else {
        return z * sigmoid<false>(z);
    }
}
// SiLU of z given y = -log2(e) * z (the caller folds that factor into the taps and the bias,
// which saves one multiply per element):  z sigmoid(z) = y / (c + c 2^y),  c = -log2(e).
__device__ __forceinline__ float silu_from_scaled(float y) {
    constexpr float c = -1.4426950408889634f;
    return y * __builtin_amdgcn_rcpf(fmaf(__builtin_amdgcn_exp2f(y), c, c));
}
constexpr float kSiluPrescale = -1.4426950408889634f;

// d silu(z) / dz = s (1 + z (1 - s)),  s = sigmoid(z)  (csrc/causal_conv1d_bwd.cu:168-170)
template <bool PRECISE>
__device__ __forceinline__ float silu_grad(float z) {
    const float s = sigmoid<PRECISE>(z);
    return s * (1.0f + z * (1.0f - s));
}
// The same derivative given y = -log2(e) z, the pre-activation formed with taps and bias that
// carry that factor (one multiply per element less than forming z and scaling it):
//   s = 1 / (1 + 2^y),   z (1 - s) = y k (1 - s) with k = -ln 2,   k (1 - s) = k - k s.
__device__ __forceinline__ float silu_grad_from_scaled(float y) {
    constexpr float k = -0.6931471805599453f;
    const float s = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(y));
    return s * fmaf(y, fmaf(-k, s, k), 1.0f);
}
// The derivative divided by c = -log2(e), for kernels that keep only the prescaled taps c w:
// with g' = dout act'(z) / c, dx = sum (c w) g' is the true dx, and the sums of g' x and of g'
// are dweight / c and dbias / c (multiplied by c once, at the end).  1 / c = -ln 2 = k.
__device__ __forceinline__ float silu_grad_from_scaled_over_c(float y) {
    constexpr float k = -0.6931471805599453f, kk = 0.4804530139182014f;   // kk = k^2
    const float s = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(y));
    return s * fmaf(y, fmaf(-kk, s, kk), k);
}
// d silu / dz at z = bias + sum_w wv[w] xwin[w].  The fast variant takes the taps and bias
// prescaled by -log2(e) (wvs, bias_s); the precise one the plain ones.
template <int W, bool PRECISE>
__device__ __forceinline__ float silu_grad_of_window(const float (&wv)[W], float bias_v, const float (&wvs)[W],
                                                     float bias_s, const float *xwin) {
    if constexpr (PRECISE) {
        float z = bias_v;
#pragma unroll
        for (int w = 0; w < W; ++w) z = fmaf(wv[w], xwin[w], z);
        return silu_grad<true>(z);
    } else {
        float y = bias_s;
#pragma unroll
        for (int w = 0; w < W; ++w) y = fmaf(wvs[w], xwin[w], y);
        return silu_grad_from_scaled(y);
    }
}

// How the sums of dweight / dbias are handed over (cc1d_bwd_params::overwrite_dweight): added into what is
// there, stored in fp32, or stored rounded to the parameters' 16-bit type.  The last spares the caller a
// conversion of each, two launches of about 4.5 us of host time that a short training step of 16-bit
// parameters is bound by: forward and backward of (2, 64, 512) bf16 92.7 -> 83.3 us, (2, 1024, 512) 95.7 -> 84.5
// (parameters in fp32: 82.6 and 85.3).
enum SumStore : int { kAddF32 = 0, kStoreF32 = 1, kStoreF16 = 2, kStoreBf16 = 3 };
__host__ __device__ inline int sum_store(const cc1d_bwd_params &p) {
    if (p.overwrite_dweight == CC1D_STORE_IN_W_DTYPE && p.w_dtype != CC1D_F32) return p.w_dtype == CC1D_F16 ? kStoreF16 : kStoreBf16;
    return p.overwrite_dweight != 0 ? kStoreF32 : kAddF32;
}
__device__ __forceinline__ void put_sum(void *base, int64_t off, float v, int how) {
    if (how == kStoreF16) reinterpret_cast<_Float16 *>(base)[off] = Elem<CC1D_F16>::from_float(v);
    else if (how == kStoreBf16) reinterpret_cast<__bf16 *>(base)[off] = Elem<CC1D_BF16>::from_float(v);
    else {
        float *dst = reinterpret_cast<float *>(base) + off;
        *dst = how == kStoreF32 ? v : *dst + v;
    }
}

template <int DT, int CH>
struct alignas(CH * Elem<DT>::kBytes) RawElems {
    typename Elem<DT>::type v[CH];
};

// CH channels of one (batch, l) row of a (batch, dim, k) states tensor.
template <int DT, int CH>
__device__ __forceinline__ typename Pack<DT, CH>::raw_t
load_state_row(const void *base, int64_t sb, int64_t sc, int64_t sl, int b, int c0, int l) {
    using T = typename Elem<DT>::type;
    using raw_t = typename Pack<DT, CH>::raw_t;
    const T *row = reinterpret_cast<const T *>(base) + (int64_t)b * sb + (int64_t)l * sl;
    if (sc == 1 && (reinterpret_cast<uintptr_t>(row + c0) % sizeof(raw_t)) == 0)
        return *reinterpret_cast<const raw_t *>(row + c0);
    RawElems<DT, CH> r;
#pragma unroll
    for (int j = 0; j < CH; ++j) r.v[j] = row[(int64_t)(c0 + j) * sc];
    return bitcast<raw_t>(r);
}
template <int DT, int CH>
__device__ __forceinline__ void store_state_row(void *base, int64_t sb, int64_t sc, int64_t sl,
                                                int b, int c0, int l,
                                                const typename Pack<DT, CH>::raw_t &v) {
    using T = typename Elem<DT>::type;
    using raw_t = typename Pack<DT, CH>::raw_t;
    T *row = reinterpret_cast<T *>(base) + (int64_t)b * sb + (int64_t)l * sl;
    if (sc == 1 && (reinterpret_cast<uintptr_t>(row + c0) % sizeof(raw_t)) == 0) {
        *reinterpret_cast<raw_t *>(row + c0) = v;
        return;
    }
    const RawElems<DT, CH> r = bitcast<RawElems<DT, CH>>(v);
#pragma unroll
    for (int j = 0; j < CH; ++j) row[(int64_t)(c0 + j) * sc] = r.v[j];
}

}  // namespace cc1d
