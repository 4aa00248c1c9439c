// fft_fir.hpp -- valid 1-D correlation with a short filter as a banded matrix
// product on the matrix cores (no transform).
#pragma once

#include "fft_mfma.hpp"

namespace thff {

// ---------------------------------------------------------------------------
// y[b][i] = sum_{k < F} x[b][i + k] * f[k],  i < L - F + 1,  1 <= F <= 64,
// complex x, f, no conjugation (the reference's conv1d_direct_fft_kernel,
// sample/conv1d/main.cu:38-128, computes it through 64-point FFT windows).
//
// A signal is cut into 64-byte chunks (8 float2 or 16 half2 values).  Output
// chunk c is a fixed real matrix times the input chunks c, c + 1, ..., c +
// A - 1, A = ceil((chunk - 1 + F) / chunk): the taps on its diagonals, each
// complex tap a 2 x 2 block.  The data is the B operand, one column per
// output chunk, so 16 consecutive chunks (1 KiB) make one group and step a of
// the product reads them shifted by a columns; the matrix is the A operand,
// built once per wave and kept in registers.
//   float2: v_mfma_f32_16x16x4_f32, exact fp32 products and sums.  Lane
//     (n, q) holds the 16 bytes q of its chunk, which feed four
//     instructions (any order of the reals within a chunk will do, as long as
//     both operands use it), and receives the 16 bytes q of output chunk n.
//   half2: v_mfma_f32_16x16x32_f16, one instruction per chunk and output
//     half.  A tap enters as the sum of two f16 values (scaled by a power of
//     two so that the largest has exponent 10: within 2^-23 of itself or 2^-35
//     of the largest, whichever is more), the sums are fp32, and outputs are
//     rounded once.
// What bounds it: HBM up to F of about 30 (float2) and for every F in half2;
// beyond that the fp32 matrix rate, 4 A instructions of 32 cycles per 128
// outputs.  Against overlap-save transforms (float2 64-point windows, of which
// 65 - F outputs are valid, half2 256-point), which this replaced:
//   float2, 2^26 values, F = 9:    183 us against 224 (5.9 TB/s; a copy 165)
//   float2, 2^24 values, F = 17:    50 against  93;  F = 64: 85 against 2447
//   half2,  2^26 values, F = 9:     93 against 113;  F = 64: 101 against 149
//   half2,  64 x 100003, F = 41:    13 against  25 (setting up the matrix from
//     global memory in each wave instead of the workgroup's table: 22)
// with smaller errors: rel L2 0.6e-7 to 1.1e-7 against 1.4e-7 (float2), 2.1e-4
// (one rounding) against 4.8e-4 (half2, data rounded at each DFT16 stage).
//
// A wave takes spans of 4 groups (its chunks and A - 1 more) grid-stride,
// loading the next span while it works on the current one (2 groups: 199 us
// for 2^26 float2 values, 8 groups: 190-194).  The span passes
// through LDS in four planes, one for each quarter of a chunk, so that a
// step's reads (lane n of a quarter: chunk n + a) and the reordering of the
// outputs for contiguous 1 KiB stores are free of bank conflicts (the plane
// stride is 4 mod 16 sixteen-byte slots).  Global accesses are 16 bytes at
// the element's alignment, so signals of any length move as vectors.
// Zeros stand for values past a signal's end; no valid output uses them.
// ---------------------------------------------------------------------------
template <class IO, int A>
struct FirPlan {
    static constexpr int kVec = Io<IO>::kVec;                   // values per 16 bytes
    static constexpr int kChunk = 4 * kVec;                     // values per chunk
    static constexpr int kGroups = 4;                 // groups per span
    static constexpr int kGroup = 16 * kChunk;                  // outputs per group
    static constexpr int kSpan = kGroups * kGroup;              // outputs per span
    static constexpr int kRead = kSpan + (A - 1) * kChunk;      // inputs per span
    static constexpr int kPlane = 16 * kGroups + A - 1 <= 68 ? 68 : 84;  // slots per plane
    static constexpr int kLoads = kGroups + (A > 1 ? 1 : 0);
    static constexpr int steps(int ntaps) { return (2 * kChunk - 2 + ntaps) / kChunk; }  // A
    static constexpr int kMaxSteps = steps(64);
};

// The matrix of a wave's lanes, (row, k) = (lane mod 16, lane / 16), read from
// two tables of the taps with zeros on both sides: entry d of table p is the
// pair that multiplies a value's (real, imaginary) for output part p.  The
// reals of a lane's quarter of chunk a are consecutive entries, so a table
// costs one pass over the taps per workgroup and the matrix a few LDS reads.
template <class IO, int A>
struct FirMatrix;

template <int A>
struct FirMatrix<float2, A> {
    static constexpr int kFirst = -7;               // entries d = -7 ... 8 A - 1
    static constexpr int kEntries = 8 * A - kFirst;
    struct Table {
        float2 t[2][kEntries];
    };
    float m[A][4];

    __device__ __forceinline__ static void fill(Table& table, const float2* __restrict__ taps,
                                                int ntaps, int tid) {
        if (tid < kEntries) {
            const int d = tid + kFirst;
            float2 f = make_float2(0.f, 0.f);
            if (d >= 0 && d < ntaps) f = taps[d];
            table.t[0][tid] = make_float2(f.x, -f.y);
            table.t[1][tid] = make_float2(f.y, f.x);
        }
    }
    __device__ __forceinline__ FirMatrix(const Table& table, int lane) {
        const int row = lane & 15, k = lane >> 4;
        const float2* const t = table.t[row & 1] + 2 * k - row / 2 - kFirst;
#pragma unroll
        for (int a = 0; a < A; ++a)
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                m[a][2 * c] = t[8 * a + c].x;
                m[a][2 * c + 1] = t[8 * a + c].y;
            }
    }
    // Four chains of sums, added at the end: the error stays below that of
    // the 64-point transforms for every F (one chain: 2.1e-7 at F = 64).
    __device__ __forceinline__ u32x4 run(const u32x4 (&b)[A]) const {
        f32x4 acc[4] = {};
#pragma unroll
        for (int a = 0; a < A; ++a) {
            const f32x4 v = __builtin_bit_cast(f32x4, b[a]);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                acc[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(m[a][e], v[e], acc[e], 0, 0, 0);
        }
        return __builtin_bit_cast(u32x4, (acc[0] + acc[1]) + (acc[2] + acc[3]));
    }
};

template <int A>
struct FirMatrix<__half2, A> {
    static constexpr int kFirst = -15;              // entries d = -15 ... 16 A - 1
    static constexpr int kEntries = 16 * A - kFirst;
    struct Table {
        unsigned t[2][2][kEntries];                 // [part][hi, lo]
        float unscale;
    };
    f16x8 hi[A][2], lo[A][2];  // rows 4 q + r of half h give real 8 q + 4 h + r of the chunk
    float unscale;

    __device__ __forceinline__ static void fill(Table& table, const float2* __restrict__ taps,
                                                int ntaps, int tid) {
        // The largest component's exponent (64 taps at most, one per lane).
        const int lane = tid & 63;
        float big = 0.0f;
        if (lane < ntaps) big = fmaxf(fabsf(taps[lane].x), fabsf(taps[lane].y));
#pragma unroll
        for (int s = 32; s > 0; s >>= 1) big = fmaxf(big, __shfl_xor(big, s));
        int shift = 10 + 127 - static_cast<int>(as_u32(big) >> 23);
        shift = shift < -126 ? -126 : shift > 126 ? 126 : shift;
        const float scale = as_f32(static_cast<unsigned>(127 + shift) << 23);
        if (tid < kEntries) {
            const int d = tid + kFirst;
            float2 f = make_float2(0.f, 0.f);
            if (d >= 0 && d < ntaps) f = taps[d];
            const cpx v{f.x * scale, f.y * scale};
            const cpx high = Io<__half2>::unpack(Io<__half2>::pack(v));
            const cpx low = csub(v, high);
            table.t[0][0][tid] = Io<__half2>::pack({high.re, -high.im});
            table.t[0][1][tid] = Io<__half2>::pack({low.re, -low.im});
            table.t[1][0][tid] = Io<__half2>::pack({high.im, high.re});
            table.t[1][1][tid] = Io<__half2>::pack({low.im, low.re});
        }
        if (tid == 0) table.unscale = as_f32(static_cast<unsigned>(127 - shift) << 23);
    }
    __device__ __forceinline__ FirMatrix(const Table& table, int lane) : unscale(table.unscale) {
        const int row = lane & 15, k = lane >> 4;
        // row -> real 8 (row / 4) + row % 4 (+ 4 for h = 1): value 4 (row / 4) + (row % 4) / 2 + 2 h
        const int at = 4 * k - 4 * (row / 4) - (row % 4) / 2 - kFirst;
        const unsigned* const thi = table.t[row & 1][0] + at;
        const unsigned* const tlo = table.t[row & 1][1] + at;
#pragma unroll
        for (int a = 0; a < A; ++a)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                u32x4 vh, vl;
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    vh[c] = thi[16 * a - 2 * h + c];
                    vl[c] = tlo[16 * a - 2 * h + c];
                }
                hi[a][h] = __builtin_bit_cast(f16x8, vh);
                lo[a][h] = __builtin_bit_cast(f16x8, vl);
            }
    }
    __device__ __forceinline__ u32x4 run(const u32x4 (&b)[A]) const {
        f32x4 acc[2] = {};
#pragma unroll
        for (int a = 0; a < A; ++a) {
            const f16x8 v = __builtin_bit_cast(f16x8, b[a]);
#pragma unroll
            for (int h = 0; h < 2; ++h)
                acc[h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo[a][h], v, acc[h], 0, 0, 0);
#pragma unroll
            for (int h = 0; h < 2; ++h)
                acc[h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi[a][h], v, acc[h], 0, 0, 0);
        }
        cpx o[4];
#pragma unroll
        for (int c = 0; c < 4; ++c)
            o[c] = {acc[c / 2][2 * (c % 2)] * unscale, acc[c / 2][2 * (c % 2) + 1] * unscale};
        return Io<__half2>::encode4(o);
    }
};

// Workgroups per CU of the grid (3, 4, 6 and one span per wave were timed):
// 4 for float2 (2^26 values, F = 9: 183 us, 3 185, 6 199, one span per wave
// 201), the occupancy for half2, which the matrix's registers set (A = 3, F <=
// 33: 4 waves per SIMD, above that 3; bounded there, since the compiler's own
// choice of 158 to 174 registers left a fourth workgroup for a second round:
// 64 signals of 100003, F = 41, 12.8 against 14.7 us).
template <class IO, int A>
inline constexpr int kFirPerCu = std::is_same_v<IO, __half2> && A > 3 ? 3 : 4;
template <class IO, int A>
inline constexpr int kFirMinWavesPerEU = std::is_same_v<IO, __half2> ? kFirPerCu<IO, A> : 1;

template <class IO, int A>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(kFirMinWavesPerEU<IO, A>))) void
conv1d_fir_kernel(const IO* __restrict__ x, const float2* __restrict__ taps, IO* __restrict__ y,
                  long long len, int ntaps, int batch) {
    using P = FirPlan<IO, A>;
    using Vec = typename Io<IO>::A4;
    using W1 = typename Io<IO>::W1;
    constexpr int kVec = P::kVec;
    __shared__ u32x4 lds[4 * 4 * P::kPlane];
    __shared__ typename FirMatrix<IO, A>::Table table;
    const int lane = threadIdx.x & 63, n = lane & 15, q = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    u32x4* const region = lds + wave * 4 * P::kPlane;
    u32x4* const linear = region + (lane & 3) * P::kPlane + (lane >> 2);  // 16 bytes `lane` of a group
    u32x4* const column = region + q * P::kPlane + n;                     // quarter q of chunk n

    const long long out_len = len - ntaps + 1;
    const long long spans = (out_len + P::kSpan - 1) / P::kSpan;  // per signal
    const long long total = spans * batch;
    const long long step = 4LL * gridDim.x;
    long long s = 4LL * blockIdx.x + wave;
    const DivWalk walk(step, spans);

    // The inputs of a span, zero past the signal's end.
    auto load = [&](DivPos at, u32x4 (&r)[P::kLoads]) {
        const long long start = at.r * P::kSpan;
        const IO* const src = x + at.q * len + start + kVec * lane;
        const long long left = len - start;
        if (left >= P::kRead) {
#pragma unroll
            for (int g = 0; g < P::kGroups; ++g)
                r[g] = ld_nt(reinterpret_cast<const Vec*>(src + g * P::kGroup));
            if constexpr (A > 1)
                if (lane < 4 * (A - 1))
                    r[P::kGroups] = ld_nt(reinterpret_cast<const Vec*>(src + P::kSpan));
        } else {
#pragma unroll
            for (int g = 0; g < P::kLoads; ++g) {
                W1 w[kVec];
#pragma unroll
                for (int c = 0; c < kVec; ++c) {
                    const int e = g * P::kGroup + kVec * lane + c;
                    w[c] = W1{};
                    if (e < left) w[c] = *reinterpret_cast<const W1*>(src + g * P::kGroup + c);
                }
                __builtin_memcpy(&r[g], w, 16);
            }
        }
    };

    u32x4 next[P::kLoads] = {};
    DivPos pos = walk.at(s);
    if (s < total) load(pos, next);
    FirMatrix<IO, A>::fill(table, taps, ntaps, threadIdx.x);
    __syncthreads();
    const FirMatrix<IO, A> matrix(table, lane);
    for (; s < total; s += step) {
        const DivPos at = pos;
        pos = walk.advance(pos);
        wave_lds_sync();  // the previous span's outputs have been read
#pragma unroll
        for (int g = 0; g < P::kGroups; ++g) linear[16 * g] = next[g];
        if constexpr (A > 1)
            if (lane < 4 * (A - 1)) linear[16 * P::kGroups] = next[P::kGroups];
        if (s + step < total) load(pos, next);
        wave_lds_sync();

        // A group's outputs take the place of its chunks, which later groups
        // do not read.
#pragma unroll 1
        for (int g = 0; g < P::kGroups; ++g) {
            u32x4 b[A];
#pragma unroll
            for (int a = 0; a < A; ++a) b[a] = column[16 * g + a];
            const u32x4 out = matrix.run(b);
            wave_lds_sync();
            column[16 * g] = out;
            wave_lds_sync();
        }
        const long long start = at.r * P::kSpan;
        const long long left = out_len - start;
        IO* const span = y + at.q * out_len + start;
        IO* const dst = span + kVec * lane;
        const StreamOut<false> whole(span, P::kSpan * static_cast<int>(sizeof(IO)));
#pragma unroll
        for (int g = 0; g < P::kGroups; ++g) {
            const u32x4 v = linear[16 * g];
            if (left >= P::kSpan) {
                whole.store(v, 16 * lane, 1024 * g);
            } else {
                W1 w[kVec];
                __builtin_memcpy(w, &v, 16);
#pragma unroll
                for (int c = 0; c < kVec; ++c)
                    if (g * P::kGroup + kVec * lane + c < left)
                        *reinterpret_cast<W1*>(dst + g * P::kGroup + c) = w[c];
            }
        }
    }
}

}  // namespace thff
