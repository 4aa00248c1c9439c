// fft_core.hpp -- register/LDS building blocks of the gfx950 batched C2C FFT.
//
// Arithmetic is fp32 for both storage types (float2 and half2): half inputs
// are widened on load and rounded once, round-to-nearest-even, on store.
//
// Transform convention (include/thunderfft/thunderfft.cuh:129-141 of the
// reference): forward X[k] = sum_n x[n] exp(-2*pi*i*n*k/N), inverse uses
// exp(+...), neither is normalized; natural order in and out.
//
// Algorithm: self-sorting (Stockham) decimation-in-time passes.  A pass of
// radix R after sub-transforms of length L have been formed treats butterfly
// b (0 <= b < N/R): k = b mod L, inputs x[b + j*N/R] (j < R) are multiplied
// by W_{L*R}^{j*k}, an R-point DFT gives outputs y_m written to
// (b - k)*R + k + m*L.  Inputs of every pass are unit-stride across
// threads, so pass 0 reads global memory coalesced and the last pass
// (L*R = N) writes y[b + m*N/R], also coalesced.
#pragma once

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <type_traits>

namespace thff {

struct cpx {
    float re, im;
};

__device__ __forceinline__ cpx cadd(cpx a, cpx b) { return {a.re + b.re, a.im + b.im}; }
__device__ __forceinline__ cpx csub(cpx a, cpx b) { return {a.re - b.re, a.im - b.im}; }

// a * w  (w = c + i s)
__device__ __forceinline__ cpx cmul(cpx a, cpx w) {
    return {a.re * w.re - a.im * w.im, a.re * w.im + a.im * w.re};
}
// a * conj(w)
__device__ __forceinline__ cpx cmulc(cpx a, cpx w) {
    return {a.re * w.re + a.im * w.im, a.im * w.re - a.re * w.im};
}

template <int B, int E, class F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (B < E) {
        f(std::integral_constant<int, B>{});
        static_for<B + 1, E>(f);
    }
}

// cos(2*pi*e/16), sin(2*pi*e/16), e = 0..15 (correctly rounded constants)
constexpr float kCos16[16] = {
    1.0f, 0.92387953251128675613f, 0.70710678118654752440f, 0.38268343236508977173f,
    0.0f, -0.38268343236508977173f, -0.70710678118654752440f, -0.92387953251128675613f,
    -1.0f, -0.92387953251128675613f, -0.70710678118654752440f, -0.38268343236508977173f,
    0.0f, 0.38268343236508977173f, 0.70710678118654752440f, 0.92387953251128675613f};
constexpr float kSin16[16] = {
    0.0f, 0.38268343236508977173f, 0.70710678118654752440f, 0.92387953251128675613f,
    1.0f, 0.92387953251128675613f, 0.70710678118654752440f, 0.38268343236508977173f,
    0.0f, -0.38268343236508977173f, -0.70710678118654752440f, -0.92387953251128675613f,
    -1.0f, -0.92387953251128675613f, -0.70710678118654752440f, -0.38268343236508977173f};

// (cos, sin)(2 pi num / den) for a power-of-two den, computed with the
// hardware transcendentals (v_cos_f32 / v_sin_f32, whose argument is in
// revolutions) with no memory access: num is reduced mod den first, so the
// argument num/den in [0, 1) is exact.  Within 1.1e-7 for every multiple of
// 1/4096 of a revolution.  Used where the result is rounded to
// f16 or applied to data that is (the device API's fp16 coefficients): the
// table of ThunderFFTInitialize stays the source of every fp32 twiddle.
__device__ __forceinline__ cpx cis_rev(int num, int den) {
    const float r = static_cast<float>(num & (den - 1)) / static_cast<float>(den);
    return {__builtin_amdgcn_cosf(r), __builtin_amdgcn_sinf(r)};
}

// a * W_R^E with W_R = exp(-2*pi*i/R) (forward) or exp(+2*pi*i/R) (inverse).
// R divides 16; multiplications by +-1 and +-i cost no multiplies.
template <int R, int E, bool FWD>
__device__ __forceinline__ cpx rot(cpx a) {
    constexpr int e = ((E % R) + R) % R;
    constexpr int e16 = e * (16 / R);
    if constexpr (e16 == 0) {
        return a;
    } else if constexpr (e16 == 8) {
        return {-a.re, -a.im};
    } else if constexpr (e16 == 4) {  // forward: * (-i)
        return FWD ? cpx{a.im, -a.re} : cpx{-a.im, a.re};
    } else if constexpr (e16 == 12) {  // forward: * (+i)
        return FWD ? cpx{-a.im, a.re} : cpx{a.im, -a.re};
    } else {
        constexpr float c = kCos16[e16], s = kSin16[e16];
        if constexpr (FWD)
            return {a.re * c + a.im * s, a.im * c - a.re * s};
        else
            return {a.re * c - a.im * s, a.im * c + a.re * s};
    }
}

// In-register R-point DFT, natural order in and out, R in {1,2,4,8,16}.
template <int R, bool FWD>
struct Dft {
    // R = P * Q four-step: n = Q*n1 + n2, k = k1 + P*k2.
    static constexpr int Q = 4;
    static constexpr int P = R / Q;
    static_assert(R == 8 || R == 16, "Dft: unsupported radix");
    __device__ __forceinline__ static void run(cpx* x) {
        cpx a[Q][P];
        static_for<0, Q>([&](auto n2) {
            constexpr int N2 = decltype(n2)::value;
            static_for<0, P>([&](auto n1) { a[N2][decltype(n1)::value] = x[Q * decltype(n1)::value + N2]; });
            Dft<P, FWD>::run(a[N2]);
            static_for<0, P>([&](auto k1) {
                constexpr int K1 = decltype(k1)::value;
                a[N2][K1] = rot<R, N2 * K1, FWD>(a[N2][K1]);
            });
        });
        static_for<0, P>([&](auto k1) {
            constexpr int K1 = decltype(k1)::value;
            cpx b[Q];
            static_for<0, Q>([&](auto n2) { b[decltype(n2)::value] = a[decltype(n2)::value][K1]; });
            Dft<Q, FWD>::run(b);
            static_for<0, Q>([&](auto k2) { x[K1 + P * decltype(k2)::value] = b[decltype(k2)::value]; });
        });
    }
};

template <bool FWD>
struct Dft<1, FWD> {
    __device__ __forceinline__ static void run(cpx*) {}
};

template <bool FWD>
struct Dft<2, FWD> {
    __device__ __forceinline__ static void run(cpx* x) {
        const cpx a = x[0], b = x[1];
        x[0] = cadd(a, b);
        x[1] = csub(a, b);
    }
};

template <bool FWD>
struct Dft<4, FWD> {
    __device__ __forceinline__ static void run(cpx* x) {
        const cpx t0 = cadd(x[0], x[2]), t1 = csub(x[0], x[2]);
        const cpx t2 = cadd(x[1], x[3]), t3 = rot<4, 1, FWD>(csub(x[1], x[3]));
        x[0] = cadd(t0, t2);
        x[2] = csub(t0, t2);
        x[1] = cadd(t1, t3);
        x[3] = csub(t1, t3);
    }
};

// ---------------------------------------------------------------------------
// Storage types.  float2 holds (re, im); __half2 holds low = re, high = im
// (the reference's vec2_t<half>, include/thunderfft/detail/util_cuda.h:46-49).
// ---------------------------------------------------------------------------
using u32x2 = unsigned __attribute__((ext_vector_type(2)));
using u32x4 = unsigned __attribute__((ext_vector_type(4)));

// Non-temporal global accesses (streamed data, touched once).
template <class W>
__device__ __forceinline__ W ld_nt(const W* p) {
    return __builtin_nontemporal_load(p);
}
template <class W>
__device__ __forceinline__ void st_nt(W* p, W w) {
    __builtin_nontemporal_store(w, p);
}

// The `bytes` bytes at `base` (both uniform over the wave) as a buffer for
// streamed stores; stores at offset v (per lane) past the end are dropped by
// the hardware's range check.  A constant step s goes into the scalar offset,
// which the check may leave out or take off the size first: for steps below
// `bytes` of lanes whose v is past the end whenever v + s is.  Other steps are
// part of v, based on step_base().  kThrough also writes through the
// XCD's L2 (agent scope) instead of leaving lines for the write-back at the
// kernel's end.  For whole lines from workgroups that each store once it is
// mostly the faster form: a copy of 512 MiB takes 162.4 against 165.0 us, the fp32
// C2C of 2^26 values 171.2 against 173.6 (N = 1024) and 174.8 against 177.0
// (N = 128), 2^20 values at N = 128 ... 1024 4.3-5.5 against 4.8-5.9; around
// 2^23 values, where the arrays just fit the memory-side cache, it is level to
// 2% slower (N = 1024: 26.0 against 25.6 us).  VALU kernels that walk their
// tiles gain too (C2C N = 2048 178.3 against 180.1, shared-filter conv1d N =
// 512 100.3 against 104.4 at 2^25 values), but not at every size; the half2
// walks on the matrix cores and the real convolutions measured 1-6% slower
// with it and do without.  Which calls use it, and what both forms take around
// each line, stands at the launches (c2c_instance.hip).  Partial lines each
// cost a write to memory (an unaligned half2 C2C: 12.1 against 6.5 us).
template <bool kThrough>
struct StreamOut {
    static constexpr int kPolicy = kThrough ? 18 : 2;  // nt, sc1
    __amdgpu_buffer_rsrc_t rs;
    __device__ __forceinline__ StreamOut(void* base, int bytes)
        : rs(__builtin_amdgcn_make_buffer_rsrc(base, 0, bytes, 0x00020000)) {}
    __device__ __forceinline__ void store(u32x4 w, int v, int s = 0) const {
        __builtin_amdgcn_raw_buffer_store_b128(w, rs, v, s, kPolicy);
    }
    __device__ __forceinline__ void store(u32x2 w, int v, int s = 0) const {
        __builtin_amdgcn_raw_buffer_store_b64(w, rs, v, s, kPolicy);
    }
};

// v as the base of a buffer access's constant steps: opaque here, so that the
// steps (up to 4095) become the instructions' immediate offsets; sums known
// outside a loop are computed there and kept, a register for each step.
__device__ __forceinline__ int step_base(int v) {
    asm volatile("" : "+v"(v));
    return v;
}

// Bit casts taken on plain scalars: clang mis-evaluates __builtin_bit_cast
// applied directly to an ext-vector element (w.y read as w.x), so elements
// are always passed by value first.
__device__ __forceinline__ float as_f32(unsigned u) { return __builtin_bit_cast(float, u); }
__device__ __forceinline__ unsigned as_u32(float f) { return __builtin_bit_cast(unsigned, f); }

template <class IO>
struct Io;

// W1 holds one complex value, W4 one 16-byte vector of kVec values; A4 is a W4
// in memory at its element's alignment (16-byte global accesses need no more).
template <>
struct Io<float2> {
    static constexpr int kVec = 2;
    using W1 = u32x2;
    using W4 = u32x4;
    typedef unsigned A4 __attribute__((ext_vector_type(4), aligned(8)));
    __device__ __forceinline__ static cpx decode1(W1 w) { return {as_f32(w.x), as_f32(w.y)}; }
    __device__ __forceinline__ static W1 encode1(cpx v) { return W1{as_u32(v.re), as_u32(v.im)}; }
    __device__ __forceinline__ static void decode4(W4 w, cpx* v) {
        v[0] = {as_f32(w.x), as_f32(w.y)};
        v[1] = {as_f32(w.z), as_f32(w.w)};
    }
    __device__ __forceinline__ static W4 encode4(const cpx* v) {
        return W4{as_u32(v[0].re), as_u32(v[0].im), as_u32(v[1].re), as_u32(v[1].im)};
    }
};

template <>
struct Io<__half2> {
    static constexpr int kVec = 4;
    using W1 = unsigned;
    using W4 = u32x4;
    typedef unsigned A4 __attribute__((ext_vector_type(4), aligned(4)));
    __device__ __forceinline__ static cpx unpack(unsigned w) {
        const float2 f = __half22float2(__builtin_bit_cast(__half2, w));
        return {f.x, f.y};
    }
    // Round to nearest even, low half = real.
    __device__ __forceinline__ static unsigned pack(cpx v) {
        return __builtin_bit_cast(unsigned, __floats2half2_rn(v.re, v.im));
    }
    __device__ __forceinline__ static cpx decode1(W1 w) { return unpack(w); }
    __device__ __forceinline__ static W1 encode1(cpx v) { return pack(v); }
    __device__ __forceinline__ static void decode4(W4 w, cpx* v) {
        v[0] = unpack(w.x);
        v[1] = unpack(w.y);
        v[2] = unpack(w.z);
        v[3] = unpack(w.w);
    }
    __device__ __forceinline__ static W4 encode4(const cpx* v) {
        return W4{pack(v[0]), pack(v[1]), pack(v[2]), pack(v[3])};
    }
};

// Synchronisation of an LDS region that only one wavefront touches.  LDS
// operations of one wavefront are performed in program order, so only the
// compiler must be kept from moving LDS accesses across this point.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// s_waitcnt vmcnt(0) (expcnt and lgkmcnt left at their maxima, gfx9
// encoding): every vector memory access of the wave has completed.  Placed
// inside a rarely taken branch that loads, it keeps the compiler from
// waiting for everything at the branch's join on every pass: after the join
// it counts only the accesses the common path issued.
__device__ __forceinline__ void wait_vmem_all() { __builtin_amdgcn_s_waitcnt(0x0F70); }

}  // namespace thff
