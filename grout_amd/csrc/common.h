// Shared device helpers for the gfx950 attention kernels: vector types, MFMA
// wrappers, 16-byte global/LDS moves and wave-level exchanges.
//
// Lane layouts (verified on gfx950):
//  * v_mfma_f32_32x32x16_f16: A lane l holds row l%32, k = 8*(l/32)+i;
//    B lane l holds column l%32, k = 8*(l/32)+i; C register r of lane l is
//    row 8*(r/4) + 4*(l/32) + r%4, column l%32.
//  * v_mfma_f32_16x16x32_f16: A lane l holds row l%16, k = 8*(l/16)+i;
//    B lane l holds column l%16, k = 8*(l/16)+i; C register r of lane l is
//    row 4*(l/16) + r, column l%16.
//  * ds_read_b64_tr_b16: within each 16-lane group, lane i receives element
//    (i%4) of the 8-byte chunk addressed by lane 4*j + i/4, as element j.
//  * v_permlane32_swap(a, b): returns {a with lanes 32..63 replaced by b's
//    lanes 0..31, b with lanes 0..31 replaced by a's lanes 32..63}.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace grout {

typedef _Float16 half_t;
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef short short4_t __attribute__((ext_vector_type(4)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef float float16_t __attribute__((ext_vector_type(16)));
typedef uint32_t uint4_t __attribute__((ext_vector_type(4)));

constexpr int kHeadDim = 128;
constexpr int kWave = 64;

__device__ __forceinline__ float16_t mfma32x32x16(half8_t a, half8_t b, float16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ float4_t mfma16x16x32(half8_t a, half8_t b, float4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// 16-byte global load / store of 8 halves.
__device__ __forceinline__ half8_t load_half8(const uint16_t* p) {
    return *reinterpret_cast<const half8_t*>(p);
}
__device__ __forceinline__ void store_half8(uint16_t* p, half8_t v) {
    *reinterpret_cast<half8_t*>(p) = v;
}
__device__ __forceinline__ uint4_t load_u128(const void* p) {
    return *reinterpret_cast<const uint4_t*>(p);
}
__device__ __forceinline__ void store_u128(void* p, uint4_t v) {
    *reinterpret_cast<uint4_t*>(p) = v;
}

typedef __attribute__((address_space(3))) short4_t lds_short4_t;

// Transposing LDS read of 4 halves (see the layout note at the top).
__device__ __forceinline__ half4_t lds_read_tr16(const half_t* lds_ptr) {
    short4_t v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (lds_short4_t*)(lds_ptr));
    return __builtin_bit_cast(half4_t, v);
}

// Value of lane l^32 for every lane l.
__device__ __forceinline__ float swap_halves(float x) {
    int xi = __builtin_bit_cast(int, x);
    auto r = __builtin_amdgcn_permlane32_swap(xi, xi, false, false);
    int lane = __lane_id();
    return __builtin_bit_cast(float, lane < 32 ? (int)r[1] : (int)r[0]);
}

// Value of lane l ^ 16: v_permlane16_swap exchanges 16-lane rows 2i and 2i+1
// between its two operands; with both equal, an odd row's partner arrives in
// the first result, an even row's in the second.
__device__ __forceinline__ float swap_rows16(float x) {
    int xi = __builtin_bit_cast(int, x);
    auto r = __builtin_amdgcn_permlane16_swap(xi, xi, false, false);
    int lane = __lane_id();
    return __builtin_bit_cast(float, (lane & 16) ? (int)r[0] : (int)r[1]);
}

// Value of lane l ^ 1, l ^ 2, and the sum over each aligned group of 8 lanes by
// DPP moves (quad swaps, then the mirror of 8, which pairs quads that already
// hold their sums): the adds of three xor shuffles, without their LDS trips.
__device__ __forceinline__ float sum8_dpp(float x) {
    const auto move = [](float v, auto ctrl) {
        return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v),
                                                                     decltype(ctrl)::value, 0xf, 0xf, false));
    };
    x += move(x, std::integral_constant<int, 0xB1>{});   // quad_perm [1,0,3,2]
    x += move(x, std::integral_constant<int, 0x4E>{});   // quad_perm [2,3,0,1]
    x += move(x, std::integral_constant<int, 0x141>{});  // row_half_mirror
    return x;
}

constexpr double inv_factorial_of(int n) { return n <= 1 ? 1.0 : inv_factorial_of(n - 1) / n; }
template <int n>
constexpr double kInvFact = inv_factorial_of(n);

// sin and cos of an f32 angle, each rounded once to f32 from an f64 value good
// to ~1e-16.  Cody and Waite's two-term reduction, theta = n pi/2 + r with |r| <=
// pi/4: pi/2's f64 value is a multiple of 2^-52, so x - n hi is exact in one FMA,
// and the second FMA takes n times the rest of pi/2.  Taylor series in r^2 to r^17 and r^16 (the terms left out are
// below 2e-18), summed pairwise: a launch waits for one such chain, and the
// library's sincos is ~1600 cycles long.  Angles of 2^30 and more, infinities and
// NaN take the library's.
__device__ __forceinline__ void sincos_f32(float theta, float* sn, float* cs) {
    const double x = static_cast<double>(theta);
    double sv, cv;
    if (__builtin_expect(fabsf(theta) < 1073741824.0f, 1)) {
        constexpr double kTwoOverPi = 0.63661977236758134308;
        constexpr double kPio2Hi = 1.57079632679489655800;
        constexpr double kPio2Lo = 6.12323399573676603587e-17;
        const double n = __builtin_rint(x * kTwoOverPi);
        const double r = fma(-n, kPio2Lo, fma(-n, kPio2Hi, x));
        const int q = static_cast<int>(n);
        const double z = r * r, z2 = z * z, z4 = z2 * z2;
        const double p = fma(z4, fma(z2, fma(kInvFact<17>, z, -kInvFact<15>), fma(kInvFact<13>, z, -kInvFact<11>)),
                             fma(z2, fma(kInvFact<9>, z, -kInvFact<7>), fma(kInvFact<5>, z, -kInvFact<3>)));
        const double c = fma(z4, fma(z2, kInvFact<16>, fma(-kInvFact<14>, z, kInvFact<12>)),
                             fma(z2, fma(-kInvFact<10>, z, kInvFact<8>), fma(-kInvFact<6>, z, kInvFact<4>)));
        const double sr = fma(r * z, p, r);
        const double cr = fma(z2, c, fma(-0.5, z, 1.0));
        sv = (q & 1) ? cr : sr;
        cv = (q & 1) ? sr : cr;
        if (q & 2) sv = -sv;
        if ((q + 1) & 2) cv = -cv;
    } else {
        sincos(x, &sv, &cv);
    }
    *sn = static_cast<float>(sv);
    *cs = static_cast<float>(cv);
}

// Orders LDS traffic of one wavefront (lanes exchange data through LDS
// without a workgroup barrier).
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ half8_t cat(half4_t a, half4_t b) {
    return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
}

}  // namespace grout
