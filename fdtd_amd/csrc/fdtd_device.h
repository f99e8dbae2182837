// Device helpers shared by the step kernels: element access in the storage
// types and the two forms of the Debye update.
#pragma once

#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <type_traits>

namespace {

__device__ inline float e_update(float c, float d, float a, double g1, double g2, double g3, float e0, float e1,
                                 float dn1, float dn, float dm1)
{
    const float fe = d * e0 - a * e1;
    double s = (double)fe + g1 * (double)dn1;
    s = s - g2 * (double)dn;
    s = s + g3 * (double)dm1;
    return (float)((double)c * s);
}

// Element access at a 32-bit byte offset from a scalar base, for the three
// storage types.  fp32 values pass through; fp16/bf16 convert to and from
// fp32 with round-to-nearest-even.  The _nt forms are the streaming
// (nontemporal) variants for data a launch touches once: the ring levels n
// and n-1 of D, level n-1 of E and every store.
template <typename T> struct Elem;

template <> struct Elem<float> {
    static __device__ __forceinline__ float rnd(float v) { return v; }
    static __device__ __forceinline__ float ld(const float *p, uint32_t b) { return *(const float *)((const char *)p + b); }
    static __device__ __forceinline__ float ld_nt(const float *p, uint32_t b)
    {
        return __builtin_nontemporal_load((const float *)((const char *)p + b));
    }
    static __device__ __forceinline__ void st(float *p, uint32_t b, float v) { *(float *)((char *)p + b) = v; }
    static __device__ __forceinline__ void st_nt(float *p, uint32_t b, float v)
    {
        __builtin_nontemporal_store(v, (float *)((char *)p + b));
    }
};

template <> struct Elem<__half> {
    static __device__ __forceinline__ float cvt(unsigned short u) { return __half2float(__ushort_as_half(u)); }
    static __device__ __forceinline__ unsigned short enc(float v) { return __half_as_ushort(__float2half_rn(v)); }
    static __device__ __forceinline__ float rnd(float v) { return cvt(enc(v)); }
    static __device__ __forceinline__ float ld(const __half *p, uint32_t b)
    {
        return cvt(*(const unsigned short *)((const char *)p + b));
    }
    static __device__ __forceinline__ float ld_nt(const __half *p, uint32_t b)
    {
        return cvt(__builtin_nontemporal_load((const unsigned short *)((const char *)p + b)));
    }
    static __device__ __forceinline__ void st(__half *p, uint32_t b, float v) { *(unsigned short *)((char *)p + b) = enc(v); }
    static __device__ __forceinline__ void st_nt(__half *p, uint32_t b, float v)
    {
        __builtin_nontemporal_store(enc(v), (unsigned short *)((char *)p + b));
    }
};

template <> struct Elem<__hip_bfloat16> {
    static __device__ __forceinline__ float cvt(unsigned short u) { return __uint_as_float((uint32_t)u << 16); }
    // Round to nearest even by the conversion instruction: all 2^32 floats, NaNs
    // too, give what the shifts and adds it replaces gave, about six vector
    // instructions a value (us a step: 130x156x150 42.0 -> 39.4, 256^3 195 -> 186,
    // 400x400x1000 in tiles 2048 -> 1959).
    static __device__ __forceinline__ unsigned short enc(float v)
    {
        return __builtin_bit_cast(unsigned short, (__bf16)v);
    }
    static __device__ __forceinline__ float rnd(float v) { return cvt(enc(v)); }
    static __device__ __forceinline__ float ld(const __hip_bfloat16 *p, uint32_t b)
    {
        return cvt(*(const unsigned short *)((const char *)p + b));
    }
    static __device__ __forceinline__ float ld_nt(const __hip_bfloat16 *p, uint32_t b)
    {
        return cvt(__builtin_nontemporal_load((const unsigned short *)((const char *)p + b)));
    }
    static __device__ __forceinline__ void st(__hip_bfloat16 *p, uint32_t b, float v)
    {
        *(unsigned short *)((char *)p + b) = enc(v);
    }
    static __device__ __forceinline__ void st_nt(__hip_bfloat16 *p, uint32_t b, float v)
    {
        __builtin_nontemporal_store(enc(v), (unsigned short *)((char *)p + b));
    }
};

// A Mur face's new value, the product q * x, as storage type T takes it.  A
// compiler may round such a product and its conversion to fp16 together
// (v_fma_mixlo_f16) or one after the other, so for fp16 both are spelled out:
// mur_once rounds once, as the face kernels' faces do; mur_twice by way of fp32,
// as the x faces do that a tile updates.  The other types know one way.
template <typename T>
__device__ __forceinline__ float mur_once(float q, float x)
{
    if constexpr (std::is_same<T, __half>::value) {
        uint32_t r = 0;
        asm("v_fma_mixlo_f16 %0, %1, %2, 0" : "+v"(r) : "v"(q), "v"(x));
        return Elem<T>::cvt((unsigned short)r);
    } else {
        return q * x;
    }
}
template <typename T>
__device__ __forceinline__ float mur_twice(float q, float x)
{
    float v = q * x;
    if constexpr (std::is_same<T, __half>::value) asm("" : "+v"(v));
    return v;
}

// E^{n+1} in scaled units (16-bit storage): fp32 throughout.
__device__ inline float e_update_scaled(float k1, float k2, float k3, float k5, float e0, float e1, float dn1,
                                        float dn, float dm1)
{
    const float d1 = dn1 - dn;
    const float d2 = d1 - (dn - dm1);
    return k1 * e0 - k2 * e1 + k3 * d1 + k5 * d2;
}

}  // namespace
