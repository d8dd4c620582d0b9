// Device code for contractions of floats on the bf16 matrix instruction, as source text for hipRTC.
#pragma once

namespace tc {
namespace hip {

// A float as the sum of three bf16 values: its nearest bf16, the nearest bf16 of what is left, and the rest, which
// has at most 8 bits; the differences are exact, so the sum is the float.  A product of floats is six products of such parts
// (high * high, the two of high * middle, middle * middle, the two of high * low); each is exact in float, and what
// the other three would add is below 2^-26 of the product, less than half the rounding of one float addition.
// v_mfma_f32_16x16x32_bf16 does 16 times the work of v_mfma_f32_16x16x4_f32 a cycle, so six of them still are 2.7
// times as fast; an output's chain of additions gets shorter as well (32 products to an instruction), and the five small
// products have an accumulator of their own, whose roundings are those of a sum 2^-8 as large.  Error against 64 bits, normal
// deviates, 2-norm: 96, 992 and 4096 terms 0.6e-7, 1.8e-7, 3.9e-7 (float instruction 1.8e-7, 5.6e-7, 11.5e-7).
//
// What the parts cannot hold is computed again with float arithmetic, block by block (see `SplitRange`):
//  - a value from 2^-100 down, other than zero, whose low part may be below the smallest normal bf16;
//  - an infinity, or a value that rounds to one: a middle part of infinity minus infinity.  These, and sums that overflow,
//    are seen by a result that is not finite.
constexpr const char* kDeviceSplitParts = R"HIP(
namespace __tc {
typedef __attribute__((address_space(3))) char ldschar;
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) bf16x8 ldsbf16x8;
struct SplitParts { bf16x8 part[3]; };
// The smallest magnitude but zero that was split: twice the bits of a float order it by magnitude, less one zero comes last.
struct SplitRange {
  unsigned least = ~0u;
  __device__ __forceinline__ void see(float a, float b) {
    least = __builtin_elementwise_min(least, __builtin_elementwise_min(2 * __builtin_bit_cast(unsigned, a) - 1, 2 * __builtin_bit_cast(unsigned, b) - 1));
  }
  __device__ __forceinline__ bool isTooSmall() const { return least < 2u * (27u << 23) - 1; }
};
__device__ __forceinline__ SplitParts splitFloats(const float (&v)[8], SplitRange& range) {
  typedef float floatx2 __attribute__((ext_vector_type(2)));
  SplitParts s;
#pragma unroll
  for (int j = 0; j < 8; j += 2) {
    float a = v[j], b = v[j + 1];
    range.see(a, b);
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      const bf16x2 h = __builtin_convertvector((floatx2{a, b}), bf16x2);
      s.part[q][j] = h[0];
      s.part[q][j + 1] = h[1];
      const unsigned u = __builtin_bit_cast(unsigned, h);
      a -= __builtin_bit_cast(float, u << 16);
      b -= __builtin_bit_cast(float, u & 0xffff0000u);
    }
  }
  return s;
}
// (by the bits: fast math takes every float for finite)
__device__ __forceinline__ bool isFiniteFloat(float x) { return (__builtin_bit_cast(unsigned, x) & 0x7f800000u) != 0x7f800000u; }
// The six products of the parts of 16 rows and 16 columns, 32 terms each, in the order of `q`; the last one is high * high.
constexpr int kSplitProducts = 6;
__device__ __forceinline__ constexpr int splitPartA(int q) { return q == 0 ? 2 : q == 1 || q == 3 ? 1 : 0; }
__device__ __forceinline__ constexpr int splitPartB(int q) { return q == 2 ? 2 : q == 1 || q == 4 ? 1 : 0; }
}
)HIP";

// A convolution in kernels the mapper gives to it (split_convolution.h), stride 1, no padding:
//
//   O(n, g, f, h, w) = sum over c, kh, kw of I(n, g, c, h + kh, w + kw) * W1(g, f, c, kh, kw)  [+ B(g, f)]
//
// A block computes 16 * PT consecutive pixels of one image's plane for 16 * FB filters of a group.  It goes through the
// channels CC at a time: the window of the input rows below those pixels and the filters' weights are read from memory in
// registers while the chunk before is multiplied, split once each, and laid down in LDS with eight channels of a pixel, or of
// a weight's place in the window, in 16 bytes, three such planes.  A step of the matrix instruction multiplies
// four of those: a lane group reads its eight channels of a pixel at its own place of the window, whatever place that
// is.  WF x WP wavefronts divide the filters and the pixels; a lane ends up with four consecutive pixels of a filter.
// Rows of pixels and of weights are an odd number of 16-byte units apart: no bank conflicts.
//
// What bounds it, at 16 x 64 x 57 x 57, 64 filters 3 x 3 (24 x 2 tiles, chunks of 16, 1 x 8 wavefronts, one block a compute
// unit): 28 to 30 us (on the float instruction 41 to 44, whose matrix cores alone take 23): 14.4 us of matrix instructions (an eighth of them
// for steps that do not exist: 18 places of eight channels in five steps), 9 of LDS reads, 3 of splitting, in turn at the
// barriers of a chunk, one block being all that fits.  Two smaller blocks a compute unit instead 33 to 37 us, a chunk of 8
// channels 33 (a third of its steps do not exist), four wavefronts 31 to 35, operands requested a step ahead by hand 32 and more (spills).
constexpr const char* kDeviceSplitConvolution = R"HIP(
namespace __tc {
template <bool Bias, int N, int G, int C, int F, int H, int W, int KH, int KW, int PT, int FB, int CC, int WF, int WP> struct SplitConvolution {
  static constexpr int OH = H - KH + 1, OW = W - KW + 1, kPlane = OH * OW, kPlaces = KH * KW, kOctets = CC / 8;
  static constexpr int kThreads = 64 * WF * WP, kPixelsOfBlock = 16 * PT, kFiltersOfBlock = 16 * FB;
  static constexpr int kBands = (kPlane + kPixelsOfBlock - 1) / kPixelsOfBlock, kFilterBlocks = (F + kFiltersOfBlock - 1) / kFiltersOfBlock;
  static constexpr int kLines = (kPixelsOfBlock + OW - 2) / OW + 1, kRows = (kLines < OH ? kLines : OH) + KH - 1, kPixels = kRows * W; // of the window
  static constexpr int kSlots = kPlaces * kOctets, kSteps = (kSlots + 3) / 4; // (a slot: eight channels at one place)
  static constexpr int kPitchI = 16 * (kOctets | 1), kPartI = kPixels * kPitchI;
  static constexpr int kPitchW = 16 * ((4 * kSteps) | 1), kPartW = kFiltersOfBlock * kPitchW;
  static constexpr int kItemsI = kPixels * kOctets, kTurnsI = (kItemsI + kThreads - 1) / kThreads;
  static constexpr int kItemsW = kFiltersOfBlock * kSlots, kTurnsW = (kItemsW + kThreads - 1) / kThreads;
  static constexpr int kChunks = (C + CC - 1) / CC;
  static constexpr int FT = FB / WF, PW = PT / WP; // tiles of a wavefront

  static __device__ __forceinline__ void run(float* pO, const float* pI, const float* pW, const float* pB, ldschar* lds) {
    const int lane = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(threadIdx.y), tid = lane + 64 * wave;
    int block = blockIdx.x;
    const int band = block % kBands;
    block /= kBands;
    const int f0 = block % kFilterBlocks * kFiltersOfBlock;
    block /= kFilterBlocks;
    const int group = block % G, n = block / G;
    const int p0 = band * kPixelsOfBlock, row0 = tmin(p0 / OW, H - kRows);
    const float* const image = pI + (n * G + group) * (C * H * W);
    const float* const weights = pW + group * (F * C * kPlaces);
    ldschar *li = lds, *lw = lds + 3 * kPartI;
    // What a thread stages: eight channels of a pixel, or of a place of a filter (threads without an item repeat the last one).
    int fromI[kTurnsI], toI[kTurnsI], fromW[kTurnsW], toW[kTurnsW];
#pragma unroll
    for (int i = 0; i < kTurnsI; ++i) {
      const int item = tmin(i * kThreads + tid, kItemsI - 1), octet = item / kPixels, px = item % kPixels;
      fromI[i] = (8 * octet * H * W + row0 * W + px) * 4;
      toI[i] = px * kPitchI + 16 * octet;
    }
#pragma unroll
    for (int i = 0; i < kTurnsW; ++i) {
      const int item = tmin(i * kThreads + tid, kItemsW - 1), f = item / kSlots, octet = item % kSlots / kPlaces, place = item % kPlaces;
      fromW[i] = ((tmin(f0 + f, F - 1) * C + 8 * octet) * kPlaces + place) * 4;
      toW[i] = f * kPitchW + 16 * (place * kOctets + octet);
    }
    float rawI[kTurnsI][8], rawW[kTurnsW][8];
    auto load = [&](int c0) __attribute__((always_inline)) {
      // (the descriptors begin at the chunk and end with the operand: what lies behind reads zeros)
      const __amdgpu_buffer_rsrc_t rsI = __builtin_amdgcn_make_buffer_rsrc((void*)(image + c0 * H * W), 0, (C - c0) * H * W * 4, 0x00020000);
      const __amdgpu_buffer_rsrc_t rsW = __builtin_amdgcn_make_buffer_rsrc((void*)(weights + c0 * kPlaces), 0, (F * C - c0) * kPlaces * 4, 0x00020000);
#pragma unroll
      for (int i = 0; i < kTurnsI; ++i)
#pragma unroll
        for (int e = 0; e < 8; ++e) rawI[i][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsI, fromI[i] + e * H * W * 4, 0, 0));
#pragma unroll
      for (int i = 0; i < kTurnsW; ++i)
#pragma unroll
        for (int e = 0; e < 8; ++e) rawW[i][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsW, fromW[i] + e * kPlaces * 4, 0, 0));
    };
    SplitRange range;
    auto lay = [&](float (&v)[8], int firstChannel, ldschar* to, int part) __attribute__((always_inline)) {
      if constexpr (C % CC != 0) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = firstChannel + e < C ? v[e] : 0.0f;
      }
      const SplitParts s = splitFloats(v, range);
#pragma unroll
      for (int q = 0; q < 3; ++q) *(ldsbf16x8*)(to + q * part) = s.part[q];
    };
    load(0);
    if constexpr (kSlots % 4 != 0) { // the weights of slots that do not exist; the input is read at some other place there
      constexpr int kMissing = 4 * kSteps - kSlots;
      for (int i = tid; i < 3 * kFiltersOfBlock * kMissing; i += kThreads) {
        *(ldsbf16x8*)(lw + i / kMissing * kPitchW + 16 * (kSlots + i % kMissing)) = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
      }
    }
    // Where this lane reads: its pixel of each tile, its slot of each step, its filter.
    const int r = lane & 15, g = lane >> 4, wf = wave % WF, wp = wave / WF;
    int atI[PW], slotI[kSteps];
#pragma unroll
    for (int t = 0; t < PW; ++t) {
      const int p = tmin(p0 + 16 * (wp * PW + t) + r, kPlane - 1);
      atI[t] = ((p / OW - row0) * W + p % OW) * kPitchI;
    }
#pragma unroll
    for (int j = 0; j < kSteps; ++j) {
      const int slot = 4 * j + g < kSlots ? 4 * j + g : 0, place = slot / kOctets;
      slotI[j] = (place / KW * W + place % KW) * kPitchI + 16 * (slot % kOctets);
    }
    const int atW = (16 * wf * FT + r) * kPitchW + 16 * g;
    floatx4 large[PW][FT], small[PW][FT];
#pragma unroll
    for (int t = 0; t < PW; ++t)
#pragma unroll
      for (int f = 0; f < FT; ++f) large[t][f] = small[t][f] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
    for (int c = 0; c < kChunks; ++c) {
#pragma unroll
      for (int i = 0; i < kTurnsI; ++i) lay(rawI[i], c * CC + 8 * (tmin(i * kThreads + tid, kItemsI - 1) / kPixels), li + toI[i], kPartI);
#pragma unroll
      for (int i = 0; i < kTurnsW; ++i) lay(rawW[i], c * CC + 8 * (tmin(i * kThreads + tid, kItemsW - 1) % kSlots / kPlaces), lw + toW[i], kPartW);
      __syncthreads();
      load(tmin(c + 1, kChunks - 1) * CC);
#pragma unroll
      for (int j = 0; j < kSteps; ++j) {
        bf16x8 vw[FT][3], vi[PW][3];
#pragma unroll
        for (int f = 0; f < FT; ++f)
#pragma unroll
          for (int q = 0; q < 3; ++q) vw[f][q] = *(const ldsbf16x8*)(lw + atW + f * 16 * kPitchW + 64 * j + q * kPartW);
#pragma unroll
        for (int t = 0; t < PW; ++t)
#pragma unroll
          for (int q = 0; q < 3; ++q) vi[t][q] = *(const ldsbf16x8*)(li + atI[t] + slotI[j] + q * kPartI);
#pragma unroll
        for (int q = 0; q < kSplitProducts; ++q)
#pragma unroll
          for (int t = 0; t < PW; ++t)
#pragma unroll
            for (int f = 0; f < FT; ++f) {
              floatx4& sum = q == kSplitProducts - 1 ? large[t][f] : small[t][f];
              sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vi[t][splitPartA(q)], vw[f][splitPartB(q)], sum, 0, 0, 0);
            }
      }
      __syncthreads();
    }
    bool again = range.isTooSmall();
#pragma unroll
    for (int t = 0; t < PW; ++t)
#pragma unroll
      for (int f = 0; f < FT; ++f) {
        large[t][f] += small[t][f];
#pragma unroll
        for (int e = 0; e < 4; ++e) again |= !isFiniteFloat(large[t][f][e]);
      }
    if (__syncthreads_or(again)) { // (what the parts cannot hold: rare, and slow)
#pragma unroll 1
      for (int i = tid; i < kFiltersOfBlock * kPixelsOfBlock; i += kThreads) {
        const int filter = f0 + i / kPixelsOfBlock, p = p0 + i % kPixelsOfBlock;
        if (filter >= F || p >= kPlane) continue;
        float sum = 0.0f;
#pragma unroll 1
        for (int k = 0; k < C * kPlaces; ++k) {
          const int place = k % kPlaces;
          sum = __builtin_fmaf(image[k / kPlaces * (H * W) + (p / OW + place / KW) * W + p % OW + place % KW], weights[filter * (C * kPlaces) + k], sum);
        }
        if constexpr (Bias) sum += pB[group * F + filter];
        pO[((n * G + group) * F + filter) * kPlane + p] = sum;
      }
      return;
    }
    typedef unsigned uintx4 __attribute__((ext_vector_type(4)));
    const __amdgpu_buffer_rsrc_t rsO = __builtin_amdgcn_make_buffer_rsrc((void*)pO, 0, N * G * F * kPlane * 4, 0x00020000);
#pragma unroll
    for (int f = 0; f < FT; ++f) {
      const int filter = f0 + 16 * (wf * FT + f) + r;
      if (F % kFiltersOfBlock != 0 && filter >= F) continue;
      float bias = 0.0f;
      if constexpr (Bias) bias = pB[group * F + filter];
#pragma unroll
      for (int t = 0; t < PW; ++t) {
        const int p = p0 + 16 * (wp * PW + t) + 4 * g, at = ((n * G + group) * F + filter) * kPlane + p;
        floatx4 v = large[t][f];
        if constexpr (Bias) v += floatx4{bias, bias, bias, bias};
        if (kPlane % kPixelsOfBlock == 0 || p + 4 <= kPlane) {
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(uintx4, v), rsO, at * 4, 0, 16);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if (p + e < kPlane) __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, (float)v[e]), rsO, (at + e) * 4, 0, 16);
          }
        }
      }
    }
  }
};
}
)HIP";

} // namespace hip
} // namespace tc
