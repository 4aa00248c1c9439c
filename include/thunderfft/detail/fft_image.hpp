// fft_image.hpp -- the passes of the 1024 x 1024 convolution
//   y = IFFT2(FFT2(x) * FFT2(h)) / 2^20
// (the reference's sample runs it as row FFT, column FFT x H x IFFT, inverse
// row FFT, sample/conv2d/thunder.cu:70-207).  Here the row passes also do the
// first radix of the column transforms, and the last of their inverse:
//   rows:    FFTs of rows r0 + kLen m (m < kRadix) of x, then across them
//              Z_k2[r0] = W_1024^(r0 k2) sum_m X[r0 + kLen m] W_kRadix^(m k2),
//            stored as row r0 + kLen k2 of y; h likewise into a workspace (fp32)
//   columns: for each k2 and column, FFT of kLen over r0, product with H,
//            inverse FFT, in place in y; each workgroup transforms its columns
//            of the filter first
//   rows:    inverse row FFTs, then the inverse across the rows k2, in place
//
// Why.  Every pass reads and writes the images once, so three copies bound a
// large batch (32 float2 images: 3 x 83 us at the rate of a copy).  A row pass
// alone leaves the arithmetic units idle half of the time, while a column pass
// has two transforms to do.  With the radix of 8 moved to the row passes the
// columns are transforms of 128, with one exchange instead of two, and a
// workgroup that holds 4096 values takes 32 adjacent columns: whole lines of
// every row (256 bytes float2, 128 half2), moved straight between HBM and
// registers.  The filter's rows ride in the first launch and its columns in
// the column pass, three launches instead of five.
//
// Measured, whole calls, against row passes by the C2C kernels, column units
// of 8 or 16 columns staged through LDS (64 bytes of each row) and the
// filter's two passes in launches of their own:
//   float2: 32 images 278 us against 362, 9 images 89 against 136, 1 image 29
//     (24 on the GPU) against 49
//   half2:  32 images 182 us against 215 (a column pass on MFMA), 8 images 57
//     against 84, 1 image 25 to 29 against 41; rel L2 3.6e-4 against 5.3e-4
//     (7.0e-4 from 8 images on): the values are rounded when stored, not
//     between the stages of a transform
// Tried: groups of 4 (8) rows stored column by column instead of the radix
// (4-column units, 128-byte pieces): 292 and 184 us; a radix of 4 for float2:
// within 1%; half2 rows on MFMA: 182 for 32 images, but the filter's rows in a
// launch of their own; non-temporal accesses as in the C2C kernels: 295 and
// 188 us for 32 images (the next pass then finds less in the caches), non-
// temporal reads of x alone: 271 float2, but 185 half2 and 4% slower up to 8
// images.
#pragma once

#include "fft_tile.hpp"

namespace thff {

template <class IO>
struct ImagePlan {
    static constexpr int kN = 1024;
    static constexpr int kRadix = 8;              // rows of a row workgroup
    static constexpr int kLen = kN / kRadix;      // column transform
    static constexpr int kCols = 4096 / kLen;     // columns of a column workgroup
    static constexpr int kRowLanes = 64 * kRadix;
    static constexpr int kBlocks = kRadix * (kN / kCols);              // column workgroups per image
    // The forward row pass's results are 1 / kScale of Z (image_rows_kernel).
    static constexpr float kScale = std::is_same_v<IO, float2> ? 1.0f : kRadix;
    static constexpr long long kImage = static_cast<long long>(kN) * kN;
    // half2: the column pass stores the values of a wave (32 columns of 32
    // rows) times kQuiet where that leaves all of them below 65504, and marks
    // the waves where it does not.  Before the last radix the values are a
    // third of the size that the rows' spectra have after it, and stored as
    // they are they meet the f16 subnormals earlier than those would (rel L2 at
    // an output rms of 1e-3 2.5e-3, 9.9e-4 for a whole column transform
    // stored; marked 3.6e-4, as at an rms of 1, down to 2e-4); a fixed factor
    // would take as much from the largest outputs.  The marks are one byte
    // (kQuiet times the factor to apply) for each wave of each column
    // workgroup, behind the filter's spectra in the workspace.  Without them
    // one image takes 24.0 us against 24.8, 8 images 55.9 against 57.3;
    // multiplying every value on both sides, instead of the loud waves' alone,
    // 25.2 and 57.3.
    static constexpr bool kMarked = !std::is_same_v<IO, float2>;
    static constexpr int kQuiet = kMarked ? 128 : 1;
    static constexpr int kMarks = 4 * kBlocks;    // bytes per image
    static constexpr int kMarkImages = 256;       // images per round of passes
    // Slots of the column transforms: equal positions of the 32 columns of a
    // half-wave fall on different 8-byte banks.
    static constexpr int kColSlot = C2CPlan<kLen>::kSlot + 1;
    static_assert(kColSlot % 2 == 1 && kCols == 32, "slots on different banks");
};

// The radix across the rows of a row workgroup, for one column: z[m] is row m's
// value; w[k] = W_1024^(r0 k) times `scale`.  The forward pass multiplies the
// sums k, the inverse the inputs k.
template <int R, bool FWD>
__device__ __forceinline__ void image_across(cpx (&z)[R], const cpx (&w)[R], float scale) {
    if constexpr (FWD) {
        Dft<R, true>::run(z);
        z[0] = {z[0].re * scale, z[0].im * scale};
#pragma unroll
        for (int k = 1; k < R; ++k) z[k] = cmulc(z[k], w[k]);
    } else {
        z[0] = {z[0].re * scale, z[0].im * scale};
#pragma unroll
        for (int k = 1; k < R; ++k) z[k] = cmul(z[k], w[k]);
        Dft<R, false>::run(z);
    }
}

// Where the mark of wave w and column workgroup `block` of an image lies: a row
// workgroup's lane finds the marks of its 16 columns in 16 adjacent bytes.
__device__ __forceinline__ int image_mark(int w, int block) {
    const int cols = block % 32;
    return 256 * w + 32 * (block / 32) + 16 * (cols % 2) + cols / 2;
}

// Two adjacent values of one row as one vector.
template <class IO>
__device__ __forceinline__ void image_store_pair(IO* dst, cpx a, cpx b) {
    using W1 = typename Io<IO>::W1;
    using Pair = std::conditional_t<sizeof(IO) == 8, u32x4, u32x2>;
    const W1 o[2] = {Io<IO>::encode1(a), Io<IO>::encode1(b)};
    Pair p;
    __builtin_memcpy(&p, o, sizeof(p));
    *reinterpret_cast<Pair*>(dst) = p;
}

// Row pass, one row per wave: workgroup r0 of an image; workgroups from `split`
// on work on the filter, whose results stay float2.  It may run in place: a
// workgroup writes the rows that it has read.  `marks`: the column pass's, for
// the inverse.
template <class IO, bool FWD>
__global__ __launch_bounds__(ImagePlan<IO>::kRowLanes) __attribute__((amdgpu_waves_per_eu(4))) void
image_rows_kernel(const IO* image, IO* out, const IO* filter, float2* filter_out, unsigned split,
                  const unsigned char* __restrict__ marks, const float2* __restrict__ tw) {
    using Plan = ImagePlan<IO>;
    constexpr int N = Plan::kN, R = Plan::kRadix, kLen = Plan::kLen;
    constexpr int kPairs = N / 2 / Plan::kRowLanes;  // column pairs per lane
    constexpr int kSlot = C2CPlan<N>::kSlot;
    using W1 = typename Io<IO>::W1;
    __shared__ cpx lds[R * kSlot];
    const int tid = threadIdx.x, t = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool is_filter = FWD && blockIdx.x >= split;
    const unsigned block = is_filter ? blockIdx.x - split : blockIdx.x;
    const int r0 = static_cast<int>(block % kLen);
    const long long first = block / kLen * Plan::kImage + r0 * N;  // row r0 of the image
    const IO* const src = (is_filter ? filter : image) + first + wave * kLen * N;
    cpx* const slot = lds + wave * kSlot;

    W1 raw[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) raw[j] = reinterpret_cast<const W1*>(src + t)[64 * j];
    [[maybe_unused]] u32x4 mark{};  // byte j: column t + 64 j, column workgroup 2 j + t / 32
    if constexpr (Plan::kMarked && !FWD)
        mark = *reinterpret_cast<const u32x4*>(marks + static_cast<long long>(block / kLen) * Plan::kMarks +
                                               image_mark(r0 % 8 / 2, 32 * wave + t / 32));
    LaneTwiddles<N> w;
    w.load(t, tw);
    // 1 / kScale where a forward result is half2: the sums across the rows
    // then stay as far from overflow as the rows' spectra.
    const float scale = !FWD ? 1.0f / Plan::kQuiet : is_filter ? 1.0f : 1.0f / Plan::kScale;
    cpx across[R];
#pragma unroll
    for (int k = 1; k < R; ++k) {
        const float2 f = tw[r0 * k & (N - 1)];
        across[k] = {f.x * scale, f.y * scale};
    }
    cpx v[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) v[j] = Io<IO>::decode1(raw[j]);
    if constexpr (Plan::kMarked && !FWD) {
        if (__ballot((mark.x & mark.y & mark.z & mark.w) != 0x01010101u)) {  // mostly not
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                const float f = static_cast<float>(mark[j / 4] >> (8 * (j % 4)) & 255u);
                v[j] = {v[j].re * f, v[j].im * f};
            }
        }
    }
    fft_registers<N, FWD>(v, slot, t, w);
    wave_lds_sync();
#pragma unroll
    for (int j = 0; j < 16; ++j) slot[lds_pad(t + 64 * j)] = v[j];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kPairs; ++i) {
        const int c = 2 * (tid + Plan::kRowLanes * i);
        cpx z[2][R];
#pragma unroll
        for (int m = 0; m < R; ++m)
#pragma unroll
            for (int e = 0; e < 2; ++e) z[e][m] = lds[m * kSlot + lds_pad(c) + e];
#pragma unroll
        for (int e = 0; e < 2; ++e) image_across<R, FWD>(z[e], across, scale);
        if (is_filter) {
#pragma unroll
            for (int k = 0; k < R; ++k)
                image_store_pair(filter_out + first + k * kLen * N + c, z[0][k], z[1][k]);
        } else {
#pragma unroll
            for (int k = 0; k < R; ++k)
                image_store_pair(out + first + k * kLen * N + c, z[0][k], z[1][k]);
        }
    }
}

// Column workgroups per CU (4 without spills needs the next image's values not
// to be loaded ahead: 1-2% slower).
inline constexpr int kImageColsPerCu = 3;

// Column pass: a workgroup keeps kCols columns of one k2 for all the images
// that it takes, image blockIdx / kBlocks onwards in steps of gridDim /
// kBlocks (the grid is a multiple of kBlocks).  It transforms the filter's
// columns first (`filter`: the row pass's output) and holds H in registers.
// Lane (column, t) moves row t + kLen / 16 j straight between HBM and its
// registers; a column's lanes are spread over the four waves (so that a wave
// moves whole lines), and the passes synchronise the workgroup.  half2: kMarks
// marks per image, and `scale` includes kQuiet.
template <class IO>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(kImageColsPerCu))) void image_cols_kernel(
    IO* image, const float2* __restrict__ filter, unsigned char* __restrict__ marks, int images,
    float scale, const float2* __restrict__ tw) {
    using P = ImagePlan<IO>;
    using I = Io<IO>;
    using W1 = typename I::W1;
    constexpr int N = P::kN, kLen = P::kLen, kCols = P::kCols;
    constexpr int kT = kLen / 16;  // lanes of a transform
    __shared__ cpx lds[kCols * P::kColSlot];
    const int tid = threadIdx.x, c = tid % kCols, t = tid / kCols;
    const int block = static_cast<int>(blockIdx.x % P::kBlocks);
    const int row0 = block / (N / kCols) * kLen, col0 = block % (N / kCols) * kCols;
    const SharedSlot slot{lds + c * P::kColSlot};
    const int step = static_cast<int>(gridDim.x / P::kBlocks);
    int img = static_cast<int>(blockIdx.x / P::kBlocks);

    // Through a buffer resource for each image: the lane's offset is one
    // register and j's a scalar (16 64-bit addresses otherwise).
    constexpr int kSize = static_cast<int>(sizeof(IO));
    const int at = (row0 + t) * N + col0 + c;
    auto resource = [&](int im) {
        return __builtin_amdgcn_make_buffer_rsrc(image + im * P::kImage, 0,
                                                 static_cast<int>(P::kImage) * kSize, 0x00020000);
    };
    cpx H[16];
    {
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<float2*>(filter), 0, static_cast<int>(P::kImage) * 8, 0x00020000);
#pragma unroll
        for (int j = 0; j < 16; ++j)
            H[j] = Io<float2>::decode1(__builtin_bit_cast(
                u32x2, __builtin_amdgcn_raw_buffer_load_b64(rs, 8 * at, 8 * kT * N * j, 0)));
    }
    W1 next[16];
    auto load = [&](int im) {
        const __amdgpu_buffer_rsrc_t rs = resource(im);
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            if constexpr (kSize == 8)
                next[j] = __builtin_bit_cast(
                    W1, __builtin_amdgcn_raw_buffer_load_b64(rs, kSize * at, kSize * kT * N * j, 0));
            else
                next[j] = __builtin_bit_cast(
                    W1, __builtin_amdgcn_raw_buffer_load_b32(rs, kSize * at, kSize * kT * N * j, 0));
        }
    };
    load(img);
    LaneTwiddles<kLen> w;
    {   // W_kLen^m = W_1024^(kRadix m)
#pragma unroll
        for (int k = 0; k < w.p1.kStored; ++k) {
            const int j = w.p1.kCompact && k >= 3 ? 4 * (k - 2) : k + 1;
            const float2 f = tw[j * t * P::kRadix & (N - 1)];
            w.p1.b[k] = {f.x, f.y};
        }
    }
    fft_registers<kLen, true>(H, slot, t, w);
#pragma unroll
    for (int j = 0; j < 16; ++j) H[j] = {H[j].re * scale, H[j].im * scale};

    for (; img < images; img += step) {
        cpx v[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) v[j] = I::decode1(next[j]);
        if (img + step < images) load(img + step);
        fft_registers<kLen, true>(v, slot, t, w);
#pragma unroll
        for (int j = 0; j < 16; ++j) v[j] = cmul(v[j], H[j]);
        fft_registers<kLen, false>(v, slot, t, w);
        if constexpr (P::kMarked) {
            float big = 0.0f;
#pragma unroll
            for (int j = 0; j < 16; ++j) big = fmaxf(big, fmaxf(fabsf(v[j].re), fabsf(v[j].im)));
            const bool loud = __ballot(!(big < 65504.0f)) != 0;
            if (loud) {
#pragma unroll
                for (int j = 0; j < 16; ++j) v[j] = {v[j].re / P::kQuiet, v[j].im / P::kQuiet};
            }
            if ((tid & 63) == 0)
                marks[static_cast<long long>(img) * P::kMarks + image_mark(tid >> 6, block)] =
                    loud ? P::kQuiet : 1;
        }
        const __amdgpu_buffer_rsrc_t rs = resource(img);
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            if constexpr (kSize == 8)
                __builtin_amdgcn_raw_buffer_store_b64(I::encode1(v[j]), rs, kSize * at, kSize * kT * N * j, 0);
            else
                __builtin_amdgcn_raw_buffer_store_b32(I::encode1(v[j]), rs, kSize * at, kSize * kT * N * j, 0);
        }
    }
}

}  // namespace thff
