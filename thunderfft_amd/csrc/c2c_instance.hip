// c2c_instance.hip -- instantiates the C2C kernels of one length THFF_N
// (compiled once per length, -DTHFF_N=64 ... 4096, so the lengths build in
// parallel).
#include "thunderfft/detail/fft_c2c.hpp"
#include "thunderfft/detail/fft_conv.hpp"
#include "thunderfft/detail/fft_conv_mfma.hpp"
#include "thunderfft/detail/fft_fir.hpp"
#include "thunderfft/detail/fft_image.hpp"
#include "thunderfft/detail/fft_mfma.hpp"
#include "launch.hpp"

#include <type_traits>

#ifndef THFF_N
#error "compile with -DTHFF_N=<transform length>"
#endif

namespace thff {

// Grids.  per_cu = 0: one workgroup per tile.  per_cu = k: min(ntiles, k x
// CUs) workgroups walking the tiles grid-stride (tiles_per_block = 0,
// tile_walk in fft_tile.hpp), so the workgroups resident at any moment work
// on neighbouring tiles and one workgroup's set-up (twiddles, DFT operands, a
// shared filter's transform) serves many tiles.  The k of each kernel below
// is the fastest of 1, 2, 3, 4, 6, 8 and 16 on MI355X at 2^25-2^26 values
// per array (usually the kernel's occupancy in workgroups per CU).
struct Grid {
    unsigned blocks;
    int tiles_per_block;
};

inline Grid make_grid(long long ntiles, int per_cu, int num_cus) {
    if (per_cu <= 0) return {static_cast<unsigned>(ntiles), 1};
    const long long g = static_cast<long long>(per_cu) * (num_cus > 0 ? num_cus : 256);
    return {static_cast<unsigned>(ntiles < g ? ntiles : g), 0};
}

// C2C launch shape per (N, precision): workgroups per CU (make_grid) and
// whether the next tile's loads are issued before the current tile is
// transformed.  Measured at batch = 2^26/N:
//   fp32 N <= 1024: one tile per workgroup, 172-177 us (device grids: 181+).
//   fp32 N = 2048, 4096: 16 per CU (fewer for few tiles: launch_c2c) with
//     prefetch, 184 us (one or two tiles per workgroup: 188-194 us); with
//     direct movement, same box: 178 / 180 us
//     against 12 per CU 181 / 179, 8 per CU 184 / 180, 4 per CU 189 / 181,
//     8 per CU without prefetch 186 / 186, one tile per workgroup 181 / 186.
//     fp32 N = 2048 as one transform per 128-lane workgroup (each pass
//     barrier then spans the transform's 2 waves, not 4): 172.6 us at 32
//     per CU, 180.8 at 16, against 173.3 us (same box).
//   fp16 N = 2048 (three-stage MFMA, two transforms per tile): 2 per CU with
//     prefetch 88.2-88.5 us, against 90.6 at 3 per CU and 105.6 without
//     prefetch (the two-stage one-transform-per-wave kernel it replaced:
//     93-95 us at 2 per CU).
//   fp16 N = 64 (VALU): one tile per workgroup.
//   fp16 N = 128 (MFMA, c2c_mfma128_kernel): 2 per CU with prefetch 87.3 us,
//     against 90.0 at 3 per CU, 99.5 with one tile per workgroup and 90.3-91.1
//     for the VALU kernel (one tile per workgroup; device grids 93).
//   fp16 N = 256 ... 1024: the one-shot kernel (below), whose shape is fixed there.
//   fp16 N = 4096 (the walk): 2 per CU with prefetch, 89 us; 3 per CU is
//     ahead by up to 10% for 1000 to 2000 transforms (13.1 against 14.5 us)
//     and 8% behind for 16384.  Runs
//     of contiguous tiles per workgroup, which leave the balancing to the
//     dispatcher, are slower: 2 tiles 87-98 us, 4-32 tiles 93-110 us (the
//     grid-stride walk keeps all workgroups on neighbouring tiles).
// `direct` (VALU kernel): tiles move between HBM and the first pass's
// registers with no LDS staging (DirectIO, fft_tile.hpp).  fp32, same box:
// N = 256 170 vs 175 us, 512 172 vs 174, 2048 180 vs 184, 4096 179 vs 183;
// 1024 174 vs 173; 64 and 128 244 / 192 vs 172 us (a wave instruction then
// covers 16 or 8 transforms with 32- or 64-byte pieces).
struct LaunchShape {
    int per_cu;
    bool prefetch;
    bool direct = false;
};

template <int N>
constexpr LaunchShape launch_shape(int precision) {
    if (precision == 0)
        return N <= 1024 ? LaunchShape{0, false, N == 256 || N == 512}
                         : LaunchShape{16, true, true};
    if (N == 128) return {2, true};
    return N == 64 ? LaunchShape{0, false} : LaunchShape{2, true};
}

// half2 lengths whose radix-16 stages run on MFMA (fft_mfma.hpp): N = 256*C
// (two stages), N = 2048, 4096 (three stages across a workgroup) and N = 128
// (a DFT16 and a DFT8 pair within a wave).
template <int N>
inline constexpr bool kHalfOnMfma = N >= 256 && N <= 1024;
template <int N>
inline constexpr bool kHalfOnMfma3 = N == 2048 || N == 4096;
template <int N>
inline constexpr bool kHalfOnMfma128 = N == 128;

// Only the launch shape in use is instantiated.
template <class IO, int N, bool FWD>
void enqueue(Grid g, const IO* x, IO* y, int batch, const float2* tw, int num_cus,
             hipStream_t stream) {
    constexpr LaunchShape kShape = launch_shape<N>(std::is_same_v<IO, float2> ? 0 : 1);
    // Whole lines, written through (fp32 N = 256 172.4 against 174.7 us, 2048
    // 178.5 against 180.9, 1024 171.2 against 173.6; half2 N = 64 84.9 against
    // 86.6), but for fp32 N = 64 (2^22 values 12.4 against 10.8 us) and 4096
    // (1025 signals 5% slower).
    constexpr bool kThrough = !std::is_same_v<IO, float2> || (N > 64 && N < 4096);
    // fp32 N = 128, 512 and 1024 leave the lines in the L2 for mid-size batches.
    // Above 2^21 values, where the two arrays are more than the 32 MiB of the
    // eight L2s (N = 128: 16384 signals 6.3 us, written through 6.1).  N = 128
    // and 512 below 3 * 2^22 values, 192 of the memory-side cache's 256 MiB
    // (N = 128: 18820 signals 7.6, 8.0; 32768 12.8, 13.1; 65536 24.5, 24.8;
    // 131072 45.5, 44.9; N = 512: 5042 signals 8.7, 9.9; 8192 13.8, 14.1; 16384
    // 25.3, 25.5).  N = 1024 as long as every tile runs at once, 3 per CU (2702
    // signals 8.4, 8.6; 3104, with a second round, 12.1, 11.5).  N = 256 gains
    // from the write-through there too (10809 signals 10.1, 9.6; the cause is
    // not known: N = 512 stores the same way).
    // Small fp32 calls leave them too: N = 256 and 2048 below a whole tile (4
    // signals of 256 2.93 us, written through 3.23; 16 3.57, 3.54; 1 of 2048
    // 4.54, 4.73, 2 4.98, 4.94), N = 512 up to 2^16 values (2 signals 3.57,
    // 3.74; 128 4.28, 4.30; 512 4.43, 4.33), N = 1024 up to 2^19 (8 signals
    // 4.55, 4.66; 128 4.81, 4.93; 512 5.07, 5.10; 768 5.47, 5.33).
    if constexpr (std::is_same_v<IO, float2> && N >= 128 && N <= 2048) {
        constexpr long long kSmall = N == 1024  ? 1LL << 19
                                     : N == 512 ? 1LL << 16
                                     : N == 128 ? 0
                                                : C2CPlan<N>::kTile - 1;
        constexpr bool kBand = N == 128 || N == 512 || N == 1024;
        const long long end = N == 1024 ? 3LL * num_cus * C2CPlan<N>::kTile : 3LL << 22;
        const long long values = static_cast<long long>(batch) * N;
        if (values <= kSmall || (kBand && values > 1LL << 21 && values < end)) {
            c2c_kernel<IO, N, FWD, kShape.prefetch, kShape.direct><<<g.blocks, 256, 0, stream>>>(
                x, y, batch, tw, g.tiles_per_block);
            return;
        }
    }
    c2c_kernel<IO, N, FWD, kShape.prefetch, kShape.direct, kThrough><<<g.blocks, 256, 0, stream>>>(
        x, y, batch, tw, g.tiles_per_block);
}

// fp16 N = 256 ... 1024 run the one-shot kernel (c2c_mfma_wave_kernel: one
// tile per wave, its coefficients computed, no LDS table, no workgroup
// barrier).  Against a persistent 2-per-CU grid-stride kernel with LDS
// tables: N = 1024 86.6-87.0 against 88.4-89.1 us for 2^26 values, and
// 86.9-88.4 us over 8 output placements (bench.py's placement leg) against
// 90.0-102.0: the dispatcher keeps the CUs evenly fed, as for a streaming
// copy, and the time does not depend on where the output lies.  Workgroups
// of 1 or 2 such waves: 86.4-87.0 and 87.1-87.2 us at N = 1024, slower at 256
// and 512.  One tile per workgroup for the three-stage kernels (N = 2048,
// 4096) takes 118 and 96.6 us against 91.2 and 88.9 us for the walk.
// Waves per SIMD: more than fit at once, 6, and HBM serves fewer of them
// faster, the more so the shorter a wave's computing is (us at 4 per SIMD and
// uncapped, means over 8 layouts of three pairs of buffers: N = 256 16.1, 19.7
// for 40342 signals, 34.2, 43.8 for 99334, 83.5, 95.1 for 262144; N = 1024 35.1,
// 41.7 for 24833, 83.8, 89.4 for 65536; 3 per SIMD 86.1 and 84.9 for 2^26 values);
// below that one round of all the waves is ahead (N = 256 9.1 against 9.9 for
// 21618; N = 512 9.3 against 10.7 for 10809).
inline constexpr int kHalfOneShotWaves = 4;  // waves (tiles) per workgroup

template <int N, bool FWD>
void enqueue_mfma(const __half2* x, __half2* y, int batch, int num_cus, hipStream_t stream) {
    constexpr int kW = kHalfOneShotWaves, C = N / 256;
    constexpr long long kPerBlock = static_cast<long long>(kW) * MfmaPlan<C>::kFPW;
    const long long blocks = (static_cast<long long>(batch) + kPerBlock - 1) / kPerBlock;
    if (blocks <= 0) return;
    const unsigned grid = static_cast<unsigned>(blocks);
    if (blocks * kW > 4 * 6LL * num_cus)
        c2c_mfma_wave_kernel<C, FWD, kW, 4><<<grid, 64 * kW, 0, stream>>>(x, y, batch);
    else
        c2c_mfma_wave_kernel<C, FWD, kW, 0><<<grid, 64 * kW, 0, stream>>>(x, y, batch);
}

template <bool FWD>
void enqueue_mfma128(Grid g, const __half2* x, __half2* y, int batch, hipStream_t stream) {
    constexpr bool kPf = launch_shape<128>(1).prefetch;
    c2c_mfma128_kernel<FWD, kPf><<<g.blocks, 256, 0, stream>>>(x, y, batch, g.tiles_per_block);
}

template <int N, bool FWD>
void enqueue_mfma3(Grid g, const __half2* x, __half2* y, int batch, hipStream_t stream) {
    constexpr bool kPf = launch_shape<N>(1).prefetch;
    if constexpr (N == 2048)
        c2c_mfma2048_kernel<FWD, kPf><<<g.blocks, 256, 0, stream>>>(x, y, batch, g.tiles_per_block);
    else
        c2c_mfma4096_kernel<FWD, kPf><<<g.blocks, 256, 0, stream>>>(x, y, batch, g.tiles_per_block);
}

// Buffers that are element-aligned but not 16-byte aligned (any vec2_t<T>
// pointer, the reference's contract): the VALU kernel, one tile per workgroup,
// either staged, with 16-byte accesses at the element's alignment, or with
// direct movement, one element per lane and access.  Direct movement covers
// 64 N / 1024 consecutive values at a time, so short transforms are staged
// (2^26 values, half2 N = 64 91.8 against 525 us, 128 94.6 against 225; fp32
// N = 64 188 against 313 us); it saves the staging's latency in small calls
// (fp32 N = 1024, 1023 signals: 5.8 against 6.2 us), and for half2 from
// N = 512 on the staging costs more than the accesses (N = 1024, 2^26 values:
// 111 against 125 us).  Staged are
//   N = 64 from a whole tile on (64 signals: fp32 3.64 against 3.69 us, half2
//     3.54, 3.64; 16 signals 3.41, 2.85 and 3.28, 2.80);
//   N = 128 from 2^19 values (fp32: 2048 signals 4.34, 4.10, 4096 4.64, 4.64,
//     8192 5.52, 5.77; half2: 4.08, 3.90, 4.18, 4.18, 4.48, 4.85);
//   the rest above 2^21 values (fp32 N = 1024, 2895 signals: 9.7, 12.1; 2048
//     7.90, 7.57; half2 N = 256, 16383: 8.1, 11.1; 8192 5.96, 5.73).
template <class IO, int N, bool kDirect>
void enqueue_unaligned(bool forward, const IO* x, IO* y, int batch, const float2* tw,
                       hipStream_t stream) {
    const unsigned blocks =
        static_cast<unsigned>((static_cast<long long>(batch) + C2CPlan<N>::kFPB - 1) /
                              C2CPlan<N>::kFPB);
    if (forward)
        c2c_kernel<IO, N, true, false, kDirect><<<blocks, 256, 0, stream>>>(x, y, batch, tw, 1);
    else
        c2c_kernel<IO, N, false, false, kDirect><<<blocks, 256, 0, stream>>>(x, y, batch, tw, 1);
}

template <class IO, int N>
void enqueue_unaligned(bool forward, const IO* x, IO* y, int batch, const float2* tw,
                       hipStream_t stream) {
    if constexpr (std::is_same_v<IO, float2> || N <= 256) {
        constexpr long long kStaged = N == 64 ? C2CPlan<N>::kTile : N == 128 ? 1LL << 19 : (1LL << 21) + 1;
        if (static_cast<long long>(batch) * N >= kStaged) {
            enqueue_unaligned<IO, N, false>(forward, x, y, batch, tw, stream);
            return;
        }
    }
    enqueue_unaligned<IO, N, true>(forward, x, y, batch, tw, stream);
}

template <int N>
hipError_t launch_c2c(int precision, bool forward, bool aligned16, const void* in, void* out,
                      int batch, const float2* tw, int num_cus, hipStream_t stream) {
    if (!aligned16) {
        if (precision == 0)
            enqueue_unaligned<float2, N>(forward, static_cast<const float2*>(in),
                                         static_cast<float2*>(out), batch, tw, stream);
        else
            enqueue_unaligned<__half2, N>(forward, static_cast<const __half2*>(in),
                                          static_cast<__half2*>(out), batch, tw, stream);
        return hipGetLastError();
    }
    const bool mfma = precision != 0 && kHalfOnMfma<N>;
    long long fpb = C2CPlan<N>::kFPB;  // 2 for N = 2048 and 1 for N = 4096 on either kernel
    if constexpr (kHalfOnMfma<N>)
        if (mfma) fpb = MfmaPlan<N / 256>::kFPB;
    const long long ntiles = (static_cast<long long>(batch) + fpb - 1) / fpb;
    int per_cu = launch_shape<N>(precision).per_cu;
    if (precision == 0 && N >= 2048) {
        // Many tiles: the 16 per CU of launch_shape; below, fewer workgroups
        // that each prefetch what 16 per CU would start afresh: up to 5 tiles
        // per CU 2 (N = 2048: 1448 signals 10.0 against 12.2 us, 2048 13.2
        // against 15.6; N = 4096: 1024 signals 14.4 against 16.6), then 4, N =
        // 2048 up to 8 (4096 signals 26.5 against 27.5; beyond, a third and
        // fourth round are uneven: 5042 33.8, 32.1; 6653 43.6, 40.7), N = 4096
        // up to 16 (2048 27.4, 29.3; 3821 47.1, 48.5; at 2^26 values 4 per CU
        // takes 183-185 us, 16 per CU 179-181).
        if (ntiles <= 5LL * num_cus)
            per_cu = 2;
        else if (ntiles <= (N == 2048 ? 8LL : 16LL) * num_cus)
            per_cu = 4;
    }
    // The half2 walks take a third workgroup per CU between 5 and 10 tiles per
    // CU: N = 128, 46341 signals 9.8 against 10.6 us, 65537 13.2 against 13.9;
    // N = 2048, 2897 signals 11.9 against 12.5; N = 4096, 2049 signals 13.3
    // against 14.0.  Outside it the third is even or behind (N = 4096, 1025
    // signals 7.9 against 7.6; N = 2048, 1449 8.8 against 7.9, 32769 99
    // against 91).
    if (precision != 0 && per_cu == 2 && ntiles > 5LL * num_cus && ntiles <= 10LL * num_cus)
        per_cu = 3;
    const Grid g = make_grid(ntiles, per_cu, num_cus);
    if (precision == 0) {
        const auto* x = static_cast<const float2*>(in);
        auto* y = static_cast<float2*>(out);
        if (forward)
            enqueue<float2, N, true>(g, x, y, batch, tw, num_cus, stream);
        else
            enqueue<float2, N, false>(g, x, y, batch, tw, num_cus, stream);
    } else {
        const auto* x = static_cast<const __half2*>(in);
        auto* y = static_cast<__half2*>(out);
        if constexpr (kHalfOnMfma<N>) {
            if (forward)
                enqueue_mfma<N, true>(x, y, batch, num_cus, stream);
            else
                enqueue_mfma<N, false>(x, y, batch, num_cus, stream);
        } else if constexpr (kHalfOnMfma3<N>) {
            if (forward)
                enqueue_mfma3<N, true>(g, x, y, batch, stream);
            else
                enqueue_mfma3<N, false>(g, x, y, batch, stream);
        } else if constexpr (kHalfOnMfma128<N>) {
            if (forward)
                enqueue_mfma128<true>(g, x, y, batch, stream);
            else
                enqueue_mfma128<false>(g, x, y, batch, stream);
        } else if (forward) {
            enqueue<__half2, N, true>(g, x, y, batch, tw, num_cus, stream);
        } else {
            enqueue<__half2, N, false>(g, x, y, batch, tw, num_cus, stream);
        }
    }
    return hipGetLastError();
}

// Launch shapes of the VALU convolutions (conv1d_kernel, conv1d_real_kernel):
// workgroups per CU (make_grid; 0 = one tile per workgroup) and next-tile
// prefetch.  Measured on MI355X (complex: 2^25 values per array; real: 2^26
// samples, 64 channels):
//   complex fp32, per-signal filters: one tile per workgroup up to N = 256
//     (130-133 us against 135-152 us for device grids); N = 512 ... 2048 3 per
//     CU below 20 tiles per CU (N = 1024: 4097 signals 22.0, 10086 46.3 us; one
//     tile per workgroup 23.7, 49.7; N = 2048: 6 per CU 2-4% behind, at 8192
//     signals 78.8 against 74.6, at 9410 89.0 against 87.6), from there on
//     (N = 2048: 11585 signals 106.2 against 106.9, 14263 126.4 against 135.1)
//     6 per CU, so that a finished workgroup's place is taken at once
//     (N = 512 136.9, 1024 140.0 us, one tile per workgroup 140.0, 145.6;
//     N = 2048 146.3, 3 per CU 149.3);
//     N = 4096 2 per CU (167 us; prefetch 192).
//   complex fp32, shared filter (transformed once per workgroup): up to N =
//     256 one tile per workgroup (93-97 us, 3 per CU the same), except
//     between 4 and 16 tiles per CU, where 3 per CU is ahead (2^22.7 values
//     22.7-23.7 against 24.3-25.0 us; at 600 tiles N = 128 is behind, 13.0
//     against 9.9); N = 512 2
//     per CU with early prefetch (101 us, one tile per workgroup 122);
//     N = 1024, 2048 3 per CU (102 and 107 us; one tile per workgroup 127);
//     N = 4096 2 per CU with early prefetch (113 us against 121).
//   real fp32: 2 per CU with prefetch, late up to N = 512 and early above:
//     97-116 us for N = 64 ... 512 (one tile per workgroup 110-153) and
//     112/121/115 us for N = 1024/2048/4096 (168-176 without prefetch).
//   fp16 on VALU (N = 64, 128 only): 4 per CU, the occupancy: real 62-64 us
//     (prefetch 62-74); complex shared filter 56.8 / 61.2 us for N = 64 / 128
//     (16 per CU 62.9 / 68.9, 5 69 / 74, 3 61 / 65; 2^24 values 30.8 / 33.7
//     against 38.1 / 41.7), per-signal 78.4 / 83.0 us (16 per CU 83.0 / 87.7).
struct ConvShape {
    int per_cu;
    Prefetch prefetch;
};

template <int N>
constexpr ConvShape valu_conv_shape(int precision, bool real, bool per_signal,
                                    long long tiles_per_cu) {
    if (precision != 0) return {4, Prefetch::kNone};
    if (real) return {2, N <= 512 ? Prefetch::kLate : Prefetch::kEarly};
    if (per_signal) return {N <= 256 ? 0 : N == 4096 ? 2 : tiles_per_cu >= 20 ? 6 : 3,
                             Prefetch::kNone};
    if (N <= 256) return {tiles_per_cu >= 4 && tiles_per_cu < 16 ? 3 : 0, Prefetch::kNone};
    if (N == 512 || N == 4096) return {2, Prefetch::kEarly};
    return {3, Prefetch::kNone};
}

// Whether a shared-filter fp32 conv1d of `tiles` tiles stores through the L2:
// always up to N = 512 (2^14 values 6.08 us, without 6.45; 2^23 26.8, 28.0 at N =
// 128; 2^25 100.3, 104.4 at 512). N = 1024 and 2048 do not just above 2^21 values,
// where input and output are more than the L2s' 32 MiB together (N = 1024 up to
// 2^22: 2194 signals 14.5, 13.9; 3565 18.6, 17.6; outside 2048 11.0, 11.3, 4705
// 20.7, 21.5; N = 2048 while every tile runs at once, 3 per CU: 1260 16.6, 15.7;
// outside 1024 13.1, 13.2, 1782 17.9, 18.7), nor N = 2048 from 2^23 values on
// (5792 42.9, 41.9; 16384 107.7, 106.0), nor N = 4096 from 3 tiles per CU on (724
// 17.2, 17.4; 1663 30.5, 29.4; 5792 84.7, 83.7).
template <int N>
bool shared_conv_through(long long tiles, int num_cus) {
    constexpr long long kLine = (1LL << 21) / C2CPlan<N>::kTile;
    if (N == 1024) return tiles <= kLine || tiles > 2 * kLine;
    if (N == 2048) return tiles <= kLine || (tiles > 3LL * num_cus && tiles < 4 * kLine);
    return N < 1024 || tiles < 3LL * num_cus;
}

// half2 (N = 64, 128) always stores through the L2; float2 with per-signal
// filters never does (N = 64, 128: 2% slower).
template <class IO, int N>
void enqueue_conv1d(bool per_signal, Grid g, Prefetch pf, const IO* x, const IO* h, IO* y,
                    int batch, const float2* tw, int num_cus, hipStream_t stream) {
    constexpr bool kHalf = std::is_same_v<IO, __half2>;
    const auto shared = [&](auto through) {
        constexpr bool kThrough = decltype(through)::value;
        if (pf == Prefetch::kEarly)
            conv1d_kernel<IO, N, false, Prefetch::kEarly, false, kThrough>
                <<<g.blocks, 256, 0, stream>>>(x, h, y, batch, tw, g.tiles_per_block);
        else
            conv1d_kernel<IO, N, false, Prefetch::kNone, false, kThrough>
                <<<g.blocks, 256, 0, stream>>>(x, h, y, batch, tw, g.tiles_per_block);
    };
    if (per_signal) {
        conv1d_kernel<IO, N, true, Prefetch::kNone, (N >= 256), kHalf>
            <<<g.blocks, 256, 0, stream>>>(x, h, y, batch, tw, g.tiles_per_block);
        return;
    }
    if constexpr (!kHalf && N >= 1024) {
        const long long tiles =
            (static_cast<long long>(batch) + C2CPlan<N>::kFPB - 1) / C2CPlan<N>::kFPB;
        if (!shared_conv_through<N>(tiles, num_cus)) {
            shared(std::false_type{});
            return;
        }
    }
    shared(std::true_type{});
}

template <int N>
hipError_t launch_conv1d(int precision, bool per_signal_filter, const void* x, const void* h,
                         void* y, int batch, const float2* tw, int num_cus, hipStream_t stream) {
    // fp16 N = 256 ... 2048: all three transforms on MFMA (fft_conv_mfma.hpp);
    // per-signal filters, 2^25 values, against the VALU path on MI355X:
    // 77 vs 90 us (N=256), 83 vs 116 (512), 91 vs 122 (1024), 107 vs 138 (2048).
    // Grid: the occupancy, 3 workgroups per CU (2 for N = 2048), 6% faster
    // than 4 tiles per workgroup.
    if constexpr (N >= 256 && N <= 2048) {
        if (precision != 0) {
            constexpr int C = N / 256;
            using M = MfmaPlan<C>;
            const long long ntiles = (static_cast<long long>(batch) + M::kFPB - 1) / M::kFPB;
            const Grid g = make_grid(ntiles, C == 8 ? 2 : 3, num_cus);
            const auto* xx = static_cast<const __half2*>(x);
            const auto* hh = static_cast<const __half2*>(h);
            auto* yy = static_cast<__half2*>(y);
            if (per_signal_filter)
                conv1d_mfma_kernel<C, true><<<g.blocks, 256, 0, stream>>>(xx, hh, yy, batch,
                                                                          g.tiles_per_block);
            else
                conv1d_mfma_kernel<C, false><<<g.blocks, 256, 0, stream>>>(xx, hh, yy, batch,
                                                                           g.tiles_per_block);
            return hipGetLastError();
        }
    }
    // fp16 N = 4096: the three-stage MFMA transform, one signal per tile, the
    // grid at the kernel's occupancy (per-signal filters: 3 workgroups per CU;
    // a shared filter keeps its spectrum live across the loop, 2 per CU).
    // 2^25 values on MI355X: 103 vs 162 us per-signal, 76 vs 125 us shared,
    // against the VALU path.
    if constexpr (N == 4096) {
        if (precision != 0) {
            const Grid g = make_grid(batch, per_signal_filter ? 3 : 2, num_cus);
            const auto* xx = static_cast<const __half2*>(x);
            const auto* hh = static_cast<const __half2*>(h);
            auto* yy = static_cast<__half2*>(y);
            if (per_signal_filter)
                conv1d_mfma4096_kernel<N, true><<<g.blocks, 256, 0, stream>>>(xx, hh, yy, batch);
            else
                conv1d_mfma4096_kernel<N, false><<<g.blocks, 256, 0, stream>>>(xx, hh, yy, batch);
            return hipGetLastError();
        }
    }
    using P = C2CPlan<N>;
    const long long ntiles = (static_cast<long long>(batch) + P::kFPB - 1) / P::kFPB;
    const ConvShape shape =
        valu_conv_shape<N>(precision, false, per_signal_filter, ntiles / (num_cus > 0 ? num_cus : 256));
    const Grid g = make_grid(ntiles, shape.per_cu, num_cus);
    if (precision == 0)
        enqueue_conv1d<float2, N>(per_signal_filter, g, shape.prefetch,
                                  static_cast<const float2*>(x), static_cast<const float2*>(h),
                                  static_cast<float2*>(y), batch, tw, num_cus, stream);
    else if constexpr (N < 256)  // fp16 N >= 256 returned above (MFMA)
        enqueue_conv1d<__half2, N>(per_signal_filter, g, Prefetch::kNone,
                                   static_cast<const __half2*>(x), static_cast<const __half2*>(h),
                                   static_cast<__half2*>(y), batch, tw, num_cus, stream);
    return hipGetLastError();
}

template <int N>
hipError_t launch_conv1d_real_filter(const float* h, float2* spectrum, int channels, float scale,
                                     const float2* tw, hipStream_t stream) {
    const unsigned grid =
        static_cast<unsigned>((channels + C2CPlan<N>::kFPB - 1) / C2CPlan<N>::kFPB);
    conv1d_real_filter_kernel<N><<<grid, 256, 0, stream>>>(h, spectrum, channels, scale, tw);
    return hipGetLastError();
}

template <int N>
hipError_t launch_conv1d_real(int precision, const void* x, const float2* spectrum, void* y,
                              int batch, int channels, const float2* tw, int num_cus,
                              hipStream_t stream) {
    using P = C2CPlan<N>;
    const long long transforms = (static_cast<long long>(batch) + 1) / 2 * channels;
    // fp16 N = 256 ... 2048: both transforms on MFMA (fft_conv_mfma.hpp);
    // measured against this VALU path at 2^26 samples: 61 vs 68 us (N=256),
    // 60 vs 87 (512), 64 vs 87 (1024).  Grid: the occupancy, 3 workgroups per
    // CU (N = 256: 51.5 against 57.0 us for 2), 2 for N = 2048; up to N = 1024 the channels' spectra
    // stay in registers (5-9% over reloading them per tile).
    if constexpr (N >= 256 && N <= 2048) {
        if (precision != 0) {
            using M = MfmaPlan<N / 256>;
            const long long ntiles = (transforms + M::kFPB - 1) / M::kFPB;
            const Grid g = make_grid(ntiles, N == 2048 ? 2 : 3, num_cus);
            if (real_buffer_fits<N / 256>(channels))
                conv1d_real_mfma_kernel<N / 256, true><<<g.blocks, 256, 0, stream>>>(
                    static_cast<const __half*>(x), spectrum, static_cast<__half*>(y), batch,
                    channels, g.tiles_per_block);
            else
                conv1d_real_mfma_kernel<N / 256, false><<<g.blocks, 256, 0, stream>>>(
                    static_cast<const __half*>(x), spectrum, static_cast<__half*>(y), batch,
                    channels, g.tiles_per_block);
            return hipGetLastError();
        }
    }
    // fp16 N = 4096: the three-stage MFMA transform, both directions; 2
    // workgroups per CU: 77 us against 87-84 us for 3 or 4 (2^26 samples);
    // the channel's spectrum stays in registers (84 us reloading it per tile).
    if constexpr (N == 4096) {
        if (precision != 0) {
            const Grid g = make_grid(transforms, 2, num_cus);
            if (channels <= kReal4096BufferMaxChannels)
                conv1d_real_mfma4096_kernel<N, true><<<g.blocks, 256, 0, stream>>>(
                    static_cast<const __half*>(x), spectrum, static_cast<__half*>(y), batch,
                    channels, g.tiles_per_block);
            else
                conv1d_real_mfma4096_kernel<N, false><<<g.blocks, 256, 0, stream>>>(
                    static_cast<const __half*>(x), spectrum, static_cast<__half*>(y), batch,
                    channels, g.tiles_per_block);
            return hipGetLastError();
        }
    }
    const long long ntiles = (transforms + P::kFPB - 1) / P::kFPB;
    const ConvShape shape = valu_conv_shape<N>(precision, true, false, 0);
    const Grid g = make_grid(ntiles, shape.per_cu, num_cus);
    constexpr Prefetch kF32 = valu_conv_shape<N>(0, true, false, 0).prefetch;
    // fp32 N >= 2048 moves samples straight between HBM and registers
    // (conv1d_real_kernel's kDirect): N = 4096 108-114 us against 115-117,
    // 2048 115-119 against 120-123; at N = 1024 it measured slower (125 vs 113).
    if (precision == 0) {
        const auto launch = [&](auto early) {
            conv1d_real_kernel<float2, N, kF32, (N >= 2048), decltype(early)::value>
                <<<g.blocks, 256, 0, stream>>>(static_cast<const float*>(x), spectrum,
                                               static_cast<float*>(y), batch, channels, tw,
                                               g.tiles_per_block);
        };
        // The channel's spectrum, early (in flight during the forward
        // transform) or after it; 16 channels, tiles in rounds of 2 per CU:
        //   N <= 256: after it while every workgroup has one tile (N = 128, 0.7
        //     rounds 7.45 against 7.58 us, 1.0 8.02 against 8.14), early from the
        //     second on (1.1 rounds 11.4 against 12.2, 4.0 28.5 against 29.2);
        //   above: early while a CU has one tile (0.25 rounds, N = 512 7.82 against
        //     7.88, 2048 7.88 against 7.96) and from 2 rounds on (2.2, N = 512 21.6
        //     against 22.8; 4.0, N = 1024 32.3 against 34.0), N = 2048 from 2.5 (2.2
        //     rounds 22.0 late, 22.3 early; 2.8 26.2, 25.7), after it between
        //     (0.7 rounds, N = 512 9.98 against 10.16, 1024 9.51 against 9.73).
        if constexpr (N <= 2048) {
            const long long round = 2LL * num_cus;
            const bool early = N <= 256 ? ntiles > round
                                        : 2 * ntiles < round ||
                                              2 * ntiles >= (N == 2048 ? 5 : 4) * round;
            if (!early) {
                launch(std::false_type{});
                return hipGetLastError();
            }
        }
        launch(std::true_type{});
    } else if constexpr (N < 256) {  // fp16 N >= 256 returned above (MFMA)
        conv1d_real_kernel<__half2, N><<<g.blocks, 256, 0, stream>>>(
            static_cast<const __half*>(x), spectrum, static_cast<__half*>(y), batch, channels, tw,
            g.tiles_per_block);
    }
    return hipGetLastError();
}

#if THFF_N == 64
template <class IO, int A = 1>
void enqueue_conv1d_fir(int steps, const IO* x, const float2* taps, IO* y, long long len, int ntaps,
                        int batch, int num_cus, hipStream_t stream) {
    using P = FirPlan<IO, A>;
    if constexpr (A < P::kMaxSteps) {
        if (steps > A) {
            enqueue_conv1d_fir<IO, A + 1>(steps, x, taps, y, len, ntaps, batch, num_cus, stream);
            return;
        }
    }
    const long long spans = (len - ntaps + P::kSpan) / P::kSpan * batch;
    const Grid g = make_grid((spans + 3) / 4, kFirPerCu<IO, A>, num_cus);
    conv1d_fir_kernel<IO, A><<<g.blocks, 256, 0, stream>>>(x, taps, y, len, ntaps, batch);
}

hipError_t launch_conv1d_valid(int precision, const void* x, long long len, const float2* taps,
                               int ntaps, void* y, int batch, int num_cus, hipStream_t stream) {
    if (precision == 0)
        enqueue_conv1d_fir<float2>(FirPlan<float2, 1>::steps(ntaps), static_cast<const float2*>(x),
                                   taps, static_cast<float2*>(y), len, ntaps, batch, num_cus,
                                   stream);
    else
        enqueue_conv1d_fir<__half2>(FirPlan<__half2, 1>::steps(ntaps),
                                    static_cast<const __half2*>(x), taps, static_cast<__half2*>(y),
                                    len, ntaps, batch, num_cus, stream);
    return hipGetLastError();
}

hipError_t launch_conv2d64(int precision, const void* x, const void* h, void* y, int batch,
                           const float2* tw, int num_cus, hipStream_t stream) {
    // One image per tile; a device grid at the kernel's occupancy walks the
    // images grid-stride, and each workgroup transforms the filter once.
    // fp32: the VALU kernel, 4 workgroups per CU.  fp16: the MFMA kernel
    // (conv2d64_mfma_kernel), kConv2dMfmaPerCu per CU.
    if (precision == 0) {
        const Grid g = make_grid(batch, 4, num_cus);
        conv2d64_kernel<float2><<<g.blocks, 256, 0, stream>>>(
            static_cast<const float2*>(x), static_cast<const float2*>(h), static_cast<float2*>(y),
            batch, tw, g.tiles_per_block);
    } else {
        constexpr int kConv2dMfmaPerCu = 3;
        const Grid g = make_grid(batch, kConv2dMfmaPerCu, num_cus);
        conv2d64_mfma_kernel<kConv2dMfmaPerCu><<<g.blocks, 256, 0, stream>>>(
            static_cast<const __half2*>(x), static_cast<const __half2*>(h),
            static_cast<__half2*>(y), batch, g.tiles_per_block);
    }
    return hipGetLastError();
}
#endif

#if THFF_N == 128
hipError_t launch_conv2d128(int precision, const void* x, const void* h, void* y, int batch,
                            const float2* tw, int num_cus, hipStream_t stream) {
    // One image per workgroup: fp32 on VALU (conv2d128_lanes_kernel: 1024
    // lanes, a 129 KiB exchange buffer), fp16 on MFMA (conv2d128_mfma_kernel:
    // 512 lanes, 146 KiB of LDS); one workgroup per CU either way, so a device
    // grid of one per CU walks the images grid-stride.
    const Grid g = make_grid(batch, 1, num_cus);
    if (precision == 0)
        conv2d128_lanes_kernel<><<<g.blocks, 1024, 0, stream>>>(
            static_cast<const float2*>(x), static_cast<const float2*>(h), static_cast<float2*>(y),
            batch, tw);
    else
        conv2d128_mfma_kernel<1><<<g.blocks, 512, 0, stream>>>(
            static_cast<const __half2*>(x), static_cast<const __half2*>(h),
            static_cast<__half2*>(y), batch, g.tiles_per_block);
    return hipGetLastError();
}
#endif

#if THFF_N == 1024
namespace {
template <class IO>
void enqueue_conv2d1024(const IO* x, const IO* h, IO* y, float2* workspace, int batch,
                        const float2* tw, int num_cus, hipStream_t stream) {
    using P = ImagePlan<IO>;
    static_assert(sizeof(float2) * P::kImage + P::kMarkImages * P::kMarks == kConv2d1024WorkspaceBytes,
                  "workspace: the filter and the marks");
    auto* const marks = reinterpret_cast<unsigned char*>(workspace + P::kImage);
    const int wanted = kImageColsPerCu * num_cus / P::kBlocks;  // images in flight
    const int round = P::kMarked ? P::kMarkImages : batch;
    for (int first = 0; first < batch; first += round) {  // first < 2^16
        const int n = batch - first < round ? batch - first : round;
        const unsigned groups = static_cast<unsigned>(n) * P::kLen;
        const int images = wanted < 1 ? 1 : wanted < n ? wanted : n;
        IO* const out = y + first * P::kImage;
        image_rows_kernel<IO, true><<<groups + (first == 0 ? P::kLen : 0), P::kRowLanes, 0, stream>>>(
            x + first * P::kImage, out, h, workspace, groups, nullptr, tw);
        image_cols_kernel<IO><<<P::kBlocks * images, 256, 0, stream>>>(
            out, workspace, marks, n, P::kScale * P::kQuiet / (1024.0f * 1024.0f), tw);
        image_rows_kernel<IO, false><<<groups, P::kRowLanes, 0, stream>>>(out, out, nullptr, nullptr,
                                                                          groups, marks, tw);
    }
}
}  // namespace

hipError_t launch_conv2d1024(int precision, const void* x, const void* h, void* y,
                             float2* workspace, int batch, const float2* tw, int num_cus,
                             hipStream_t stream) {
    if (precision == 0)
        enqueue_conv2d1024(static_cast<const float2*>(x), static_cast<const float2*>(h),
                           static_cast<float2*>(y), workspace, batch, tw, num_cus, stream);
    else
        enqueue_conv2d1024(static_cast<const __half2*>(x), static_cast<const __half2*>(h),
                           static_cast<__half2*>(y), workspace, batch, tw, num_cus, stream);
    return hipGetLastError();
}
#endif

template hipError_t launch_c2c<THFF_N>(int, bool, bool, const void*, void*, int, const float2*,
                                       int, hipStream_t);
template hipError_t launch_conv1d<THFF_N>(int, bool, const void*, const void*, void*, int,
                                          const float2*, int, hipStream_t);
template hipError_t launch_conv1d_real_filter<THFF_N>(const float*, float2*, int, float,
                                                      const float2*, hipStream_t);
template hipError_t launch_conv1d_real<THFF_N>(int, const void*, const float2*, void*, int, int,
                                               const float2*, int, hipStream_t);

}  // namespace thff
