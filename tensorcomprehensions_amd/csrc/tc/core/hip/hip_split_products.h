// Device code for contractions of floats on the bf16 matrix instruction, as source text for hipRTC.
#pragma once

namespace tc {
namespace hip {

// A float as the sum of three bf16 values: its nearest bf16, the nearest bf16 of what is left, and the rest, which
// has at most 8 bits; the differences are exact, so the sum is the float (Henry, Tang, Heinecke, "Leveraging the bfloat16 Artificial Intelligence
// Datatype For Higher-Precision Computations", ARITH 2019).  A product of floats is six products of such parts
// (high * high, the two of high * middle, middle * middle, the two of high * low), each exact in float.  What the other three would
// add is at most 2^-24 of the product (both factors just above a power of two, as 0x1.00ff8p0), a rounding of it; for normal deviates it is 6e-9 of a sum
// of 1000 terms, a thirtieth of the roundings below.
// v_mfma_f32_16x16x32_bf16 does 16 times the work of v_mfma_f32_16x16x4_f32 a cycle, so six of them still are 2.7
// times as fast; an output's chain of additions gets shorter as well (32 products to an instruction), and in convolutions and in products of fewer than 16 tiles
// a wavefront the five small products have an accumulator of their own, whose roundings are those of a sum 2^-8 as large.
// Error against 64 bits, normal deviates, 2-norm: convolutions of 111, 576 and 837 terms 0.7e-7, 1.4e-7 and 1.7e-7; products of 1500 terms in eight slices 1.0e-7; with
// one accumulator 1.6e-7 (1000 terms, eight slices) and 2.9e-7 (768 terms, two slices).  (Float instruction: 96, 992 and 4096 terms 1.8e-7, 5.6e-7, 11.5e-7.)
//
// What the parts cannot hold is computed again on the float instruction, block by block, from the same tiles (one infinity: 1000^3 16.5 -> 39.2 us,
// the convolution below 30.3 -> 61.9):
//  - infinities, and values that round to one (a middle part of infinity minus infinity), and sums that overflow: seen by a
//    result that is not finite;
//  - small values.  A bf16 has the exponents of a float, denormal ones included, so the parts are exact from 2^-110 on, and below it
//    less than 2^-134 is left out of a value: of a sum of up to 65536 terms less than 2^-117 of the largest value that is in it, nothing
//    beside the rounding of a sum from 2^-92 of that value on, nor of a sum whose values on one side are zeros.  And products of parts
//    below 2^-149 are nothing beside the rounding of a sum from 2^-100 on.
//    A lane keeps the largest value it has split.  A block in which all sums are 2^-60 or more and all values 2^32 or less is done.  Another one
//    looks at its sums beside the largest values of their row and column (of the window and the filters).  A sum that is still too small may be one
//    of larger terms that cancelled, as the slices of a product and a few of the terms can tell, or of small values alone, whatever stands
//    beside them: where that is left open the block looks its operands over for values other than zero below 2^-110.
// The check costs half an instruction a value; one for every value's own exponent cost 1.5, and 1000^3 20.7 us for 17.4.  What follows a doubt, 1000^3 and the
// convolution below, 16.5 and 30 us: a row of zeros 18.3 and 29.6, all values 1e-20 18.9 and 30.0, a row of 1e10 18 and 29, an infinity 34.8 and 59.6, all values
// 1e-40 33 and 62 (23 and 41 us in the general pipeline, whatever the values); 2048^3 with every 16th point of an operand of whole numbers other than zero looks its
// operands over, 158 us for 103.
constexpr const char* kDeviceSplitParts = R"HIP(
namespace __tc {
typedef __attribute__((address_space(3))) char ldschar;
typedef __attribute__((address_space(3))) int ldsint;
typedef __attribute__((address_space(3))) float ldsfloat;
typedef __attribute__((address_space(3))) floatx4 ldsfloatx4;
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) bf16x8 ldsbf16x8;
struct SplitParts { bf16x8 part[3]; };
// The largest magnitude of one operand that a lane has split.
struct SplitRange {
  float most = 0.0f;
  // (one instruction; fmaxf would quiet NaNs first)
  __device__ __forceinline__ void see(float a, float b) { asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(most) : "v"(a), "v"(b)); }
  __device__ __forceinline__ bool isDoubtful() const { return most > 0x1p32f; }
};
// (by the bits: fast math takes every float for finite)
__device__ __forceinline__ unsigned magnitudeBits(float x) { return 2 * __builtin_bit_cast(unsigned, x); }
__device__ __forceinline__ constexpr unsigned magnitudeBitsOfPower(int exponent) { return 2u * ((unsigned)(127 + exponent) << 23); }
// a sum that is zero, below 2^-60 or not finite
__device__ __forceinline__ bool isDoubtfulSum(float x) {
  return magnitudeBits(x) - magnitudeBitsOfPower(-60) >= magnitudeBitsOfPower(128) - magnitudeBitsOfPower(-60);
}
// one that is not finite, or below 2^-100 but not zero
__device__ __forceinline__ bool isUnfitSum(float x) {
  return magnitudeBits(x) - magnitudeBitsOfPower(-100) >= magnitudeBitsOfPower(128) - magnitudeBitsOfPower(-100) && magnitudeBits(x) != 0;
}
// what small values could have been lost in, beside the largest values on its two sides: a sum, or the largest one of its parts
__device__ __forceinline__ bool isUnsureSum(float x, float mostA, float mostB) {
  const float most = __builtin_fmaxf(mostA, mostB);
  return __builtin_bit_cast(int, mostA) != 0 && __builtin_bit_cast(int, mostB) != 0 && __builtin_fabsf(x) < 0x1p-92f * most;
}
// a value below 2^-110 but not zero
__device__ __forceinline__ bool isUnfitValue(float x) { return magnitudeBits(x) - 1 < magnitudeBitsOfPower(-110) - 1; }
__device__ __forceinline__ void raiseTo(ldsfloat* most, float x) { // (floats from zero on are in the order of their bits)
  __hip_atomic_fetch_max((ldsint*)most, __builtin_bit_cast(int, x), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// Whether any thread of the block says so.  The flag is zero at the barrier before.  (__syncthreads_or has 256 bytes of LDS of its own.)
__device__ __forceinline__ bool isAnyOfBlock(bool is, ldsint* flag) {
  if (is) *flag = 1;
  __syncthreads();
  return *flag != 0;
}
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
// The six products of the parts of 16 rows and 16 columns, 32 terms each, in the order of `q`; the last one is high * high.
constexpr int kSplitProducts = 6;
__device__ __forceinline__ constexpr int splitPartA(int q) { return q == 0 ? 2 : q == 1 || q == 3 ? 1 : 0; }
__device__ __forceinline__ constexpr int splitPartB(int q) { return q == 2 ? 2 : q == 1 || q == 4 ? 1 : 0; }
}
)HIP";

// A convolution in kernels the mapper gives to it (mapper.cc, takeSplitConvolution), stride 1, no padding:
//
//   O(n, g, f, h, w) = sum over c, kh, kw of I(n, g, c, h + kh, w + kw) * W1(g, f, c, kh, kw)  [+ B(g, f)]
//
// A block computes 16 * PT consecutive pixels of one image's plane for 16 * FB filters of a group.  It goes through the
// channels CC at a time: the window of the input rows below those pixels and the filters' weights are read from memory in
// registers while the chunk before is multiplied, split once each, and laid down in LDS with eight channels of a pixel, or of
// a weight's place in the window, in 16 bytes, three such planes.  A step of the matrix instruction multiplies
// four of those: a lane group reads its eight channels of a pixel at its own place of the window, whatever place that
// is.  WF x WP wavefronts divide the filters and the pixels; a lane ends up with four consecutive pixels of a filter.
// Rows of pixels and of weights are an odd number of 16-byte units apart, which leaves the conflicts between the lane groups of a read.
//
// What bounds it, at 16 x 64 x 57 x 57, 64 filters 3 x 3 (24 x 2 tiles, chunks of 16, 1 x 8 wavefronts, one block a compute
// unit): 27 to 30 us (on the float instruction 41 to 44, whose matrix cores alone take 23), by counters 60 600 cycles: 23 000 of matrix
// instructions (38 %; a tenth of them for steps that do not exist: 18 places of eight channels in five steps), 23 000 of LDS instructions and 11 400
// of bank conflicts, 16 700 of vector instructions, in turn at the barriers of a chunk, one block being all that fits.  Two smaller blocks a compute unit instead 33 to 37 us, a chunk of 8
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
  static constexpr int kFlag = 3 * (kPartI + kPartW); // 16 bytes behind the parts
  static constexpr int FT = FB / WF, PW = PT / WP; // tiles of a wavefront

  // Where a block and a thread are.
  struct Place {
    int tid, lane, wave, f0, group, n, p0, row0;
    const float *image, *weights;
    __device__ __forceinline__ Place(const float* pI, const float* pW, int t) : tid(t), lane(t & 63), wave(__builtin_amdgcn_readfirstlane(t >> 6)) {
      int block = blockIdx.x;
      const int band = block % kBands;
      block /= kBands;
      f0 = block % kFilterBlocks * kFiltersOfBlock;
      block /= kFilterBlocks;
      group = block % G, n = block / G;
      p0 = band * kPixelsOfBlock, row0 = tmin(p0 / OW, H - kRows);
      image = pI + (n * G + group) * (C * H * W);
      weights = pW + group * (F * C * kPlaces);
    }
  };

  // The sums of a lane, of the parts of the floats or of the floats themselves (two planes of four channels instead of three).
  template <bool InParts> static __device__ __forceinline__ void multiply(const Place& at, ldschar* lds, floatx4 (&large)[PW][FT], SplitRange& rangeI, SplitRange& rangeW) {
    const int tid = at.tid, lane = at.lane, wave = at.wave, f0 = at.f0, p0 = at.p0, row0 = at.row0;
    const float *const image = at.image, *const weights = at.weights;
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
    auto lay = [&](float (&v)[8], int firstChannel, ldschar* to, int part, SplitRange& range) __attribute__((always_inline)) {
      if constexpr (C % CC != 0) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = firstChannel + e < C ? v[e] : 0.0f;
      }
      if constexpr (InParts) {
        const SplitParts s = splitFloats(v, range);
#pragma unroll
        for (int q = 0; q < 3; ++q) *(ldsbf16x8*)(to + q * part) = s.part[q];
      } else {
#pragma unroll
        for (int q = 0; q < 2; ++q) *(ldsfloatx4*)(to + q * part) = floatx4{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
      }
    };
    load(0);
    if (InParts && tid < 4) ((ldsint*)(lds + kFlag))[tid] = 0;
    if constexpr (InParts && kSlots % 4 != 0) { // the weights of slots that do not exist; the input is read at some other place there
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
    floatx4 small[PW][FT];
#pragma unroll
    for (int t = 0; t < PW; ++t)
#pragma unroll
      for (int f = 0; f < FT; ++f) large[t][f] = small[t][f] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
    for (int c = 0; c < kChunks; ++c) {
#pragma unroll
      for (int i = 0; i < kTurnsI; ++i) lay(rawI[i], c * CC + 8 * (tmin(i * kThreads + tid, kItemsI - 1) / kPixels), li + toI[i], kPartI, rangeI);
#pragma unroll
      for (int i = 0; i < kTurnsW; ++i) lay(rawW[i], c * CC + 8 * (tmin(i * kThreads + tid, kItemsW - 1) % kSlots / kPlaces), lw + toW[i], kPartW, rangeW);
      __syncthreads();
      load(tmin(c + 1, kChunks - 1) * CC);
#pragma unroll
      for (int j = 0; j < kSteps; ++j) {
        if constexpr (InParts) {
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
        } else {
          floatx4 vw[FT][2], vi[PW][2];
          const bool isSlot = 4 * j + g < kSlots; // (the weights are zero where there is none, the input need not be finite)
#pragma unroll
          for (int q = 0; q < 2; ++q) {
#pragma unroll
            for (int f = 0; f < FT; ++f) vw[f][q] = *(const ldsfloatx4*)(lw + atW + f * 16 * kPitchW + 64 * j + q * kPartW);
#pragma unroll
            for (int t = 0; t < PW; ++t) {
              vi[t][q] = *(const ldsfloatx4*)(li + atI[t] + slotI[j] + q * kPartI);
              if (4 * j + 3 >= kSlots) vi[t][q] = isSlot ? vi[t][q] : floatx4{0.0f, 0.0f, 0.0f, 0.0f};
            }
          }
#pragma unroll
          for (int e = 0; e < 8; ++e)
#pragma unroll
            for (int t = 0; t < PW; ++t)
#pragma unroll
              for (int f = 0; f < FT; ++f) large[t][f] = __builtin_amdgcn_mfma_f32_16x16x4f32(vi[t][e / 4][e % 4], vw[f][e / 4][e % 4], large[t][f], 0, 0, 0);
        }
      }
      __syncthreads();
    }
    if constexpr (InParts) {
#pragma unroll
      for (int t = 0; t < PW; ++t)
#pragma unroll
        for (int f = 0; f < FT; ++f) large[t][f] += small[t][f];
    }
  }

  static __device__ __forceinline__ void run(float* pO, const float* pI, const float* pW, const float* pB, ldschar* lds) {
    int t = threadIdx.x + 64 * threadIdx.y;
    const Place at(pI, pW, t);
    floatx4 large[PW][FT];
    SplitRange rangeI, rangeW;
    multiply<true>(at, lds, large, rangeI, rangeW);
    const int tid = at.tid, f0 = at.f0, group = at.group, n = at.n, p0 = at.p0, r = at.lane & 15, g = at.lane >> 4, wf = at.wave % WF, wp = at.wave / WF;
    bool doubtful = rangeI.isDoubtful() || rangeW.isDoubtful();
#pragma unroll
    for (int t = 0; t < PW; ++t)
#pragma unroll
      for (int f = 0; f < FT; ++f)
#pragma unroll
        for (int e = 0; e < 4; ++e) doubtful |= isDoubtfulSum(large[t][f][e]);
    ldsint* const flags = (ldsint*)(lds + kFlag);
    bool again = false;
    if (isAnyOfBlock(doubtful, flags)) {
      ldsfloat* const most = (ldsfloat*)lds; // of the window, of the filters
      if (tid < 2) most[tid] = 0.0f;
      __syncthreads();
      float mostI = rangeI.most, mostW = rangeW.most;
#pragma unroll
      for (int d = 32; d > 0; d /= 2) { // (64 lanes at one word are 64 turns)
        mostI = __builtin_fmaxf(mostI, __shfl_xor(mostI, d));
        mostW = __builtin_fmaxf(mostW, __shfl_xor(mostW, d));
      }
      if (at.lane == 0) {
        raiseTo(most, mostI);
        raiseTo(most + 1, mostW);
      }
      __syncthreads();
      bool unsure = false;
#pragma unroll
      for (int t = 0; t < PW; ++t)
#pragma unroll
        for (int f = 0; f < FT; ++f)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            again |= isUnfitSum(large[t][f][e]);
            unsure |= isUnsureSum(large[t][f][e], most[0], most[1]);
          }
      if (unsure) flags[1] = 1;
      again = isAnyOfBlock(again, flags + 2);
      doubtful = !again && flags[1] != 0;
    } else {
      doubtful = false;
    }
    if (doubtful) {
      // (in loops of their own: with the staging's offsets kept for them the kernel took up to 60 registers more)
      constexpr int kFlight = 16, kTurnsOfWindow = (C * kPixels + kFlight * kThreads - 1) / (kFlight * kThreads);
      const __amdgpu_buffer_rsrc_t rsI = __builtin_amdgcn_make_buffer_rsrc((void*)(at.image + at.row0 * W), 0, (C * H * W - at.row0 * W) * 4, 0x00020000);
      int pixel = tid % kPixels;
      unsigned from = tid / kPixels * (H * W) + pixel;
#pragma unroll 1
      for (int i = 0; i < kTurnsOfWindow; ++i) {
#pragma unroll
        for (int j = 0; j < kFlight; ++j) { // (behind the last channel it reads zeros)
          again |= isUnfitValue(__builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsI, from * 4, 0, 0)));
          pixel += kThreads % kPixels;
          from += kThreads / kPixels * (H * W) + kThreads % kPixels;
          if (pixel >= kPixels) pixel -= kPixels, from += H * W - kPixels;
        }
      }
      const int valuesW = tmin(kFiltersOfBlock, F - f0) * (C * kPlaces);
      const __amdgpu_buffer_rsrc_t rsW = __builtin_amdgcn_make_buffer_rsrc((void*)(at.weights + f0 * (C * kPlaces)), 0, valuesW * 4, 0x00020000);
#pragma unroll 1
      for (int i = tid; i < valuesW; i += kFlight * kThreads) {
#pragma unroll
        for (int j = 0; j < kFlight; ++j) again |= isUnfitValue(__builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsW, (i + j * kThreads) * 4, 0, 0)));
      }
      again = isAnyOfBlock(again, flags + 3);
    }
    if (again) {
      asm("" : "+v"(t)); // (or the offsets of this pass are those of the first one, kept)
      multiply<false>(Place(pI, pW, t), lds, large, rangeI, rangeW);
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

// A product of matrices in kernels the mapper gives to it (mapper.cc, takeSlicedProduct):
//
//   O(m, n) = sum over k of A * B [+ bias(n)], A stored (m, k) or (k, m), B stored (n, k) or (k, n)
//
// GA x GB x S wavefronts a block; one computes TA x TB tiles of 16 x 16 outputs over every S-th step of 32 reduction points.
// There is no LDS and no barrier in its loop: the lanes load what the instruction wants of them straight from memory,
// a step ahead, and split it in registers.  With the reduction innermost a lane group reads 64 bytes of its rows; with it
// outermost a lane reads TA (TB) neighbouring positions of a point, which become the same row (column) of as many tiles, so
// that a tile holds every TA-th position.  As the wavefronts of a block divide the reduction, each element of its rows and
// columns is loaded and split once a block, and a sum is S short chains.  The partial tiles meet in LDS, are added and
// stored in 256-byte runs.
//
// What bounds it at 1000^3 (64 x 64 outputs a block, 8 slices, one block a compute unit; 16.5 to 17 us, 23.4 in the general pipeline, whose matrix
// cores alone take 13.3): by counters 35 100 cycles, 12 300 of matrix instructions (35 %) and 17 900 of vector instructions, which one wavefront's
// instructions cannot overlap beyond two vector instructions a multiplication, the first loads (2 us), the sums' way through LDS and the launch.
// Operands laid in LDS as parts and shared by the wavefronts of a block: 22.4 us there, 92 at 2048^3 (here 89, given tiles
// 126.7): the same work behind barriers.  Parts through v_dot2_f32_bf16 save a third of the vector instructions, but it occupies the
// matrix cores.  Steps two ahead in registers, parts of the next step made under the multiplications of this one: 18.2 to 25.
constexpr const char* kDeviceSlicedProduct = R"HIP(
namespace __tc {
template <bool KInner, int P, int K, int TP> struct SlicedOperand {
  static constexpr int kOffsets = KInner ? TP : 8;
  const float* p;
  int group;             // of 16 lanes
  int offset[kOffsets];  // bytes from the step's first point: of this lane's rows, or of its points
  float value[TP][8];
  // the reduction points of a lane group, the same in both operands
  static __device__ __forceinline__ constexpr int point(int g, int j) { return 4 * g + (j & 3) + (j >> 2) * 16; }
  static __device__ __forceinline__ int position(int tile, int r) { return KInner ? 16 * tile + r : TP * r + tile; }
  __device__ __forceinline__ void init(const float* base, int first, int lane) {
    p = base;
    group = lane >> 4;
    const int r = lane & 15;
#pragma unroll
    for (int i = 0; i < kOffsets; ++i) {
      offset[i] = (KInner ? tmin(first + 16 * i + r, P - 1) * K + point(group, 0) : point(group, i) * P + tmin(first + TP * r, P - 1)) * 4;
    }
  }
  // (the descriptor begins at the step and ends with the operand: what lies behind, and steps past the last, read zeros)
  __device__ __forceinline__ void load(int k0) {
    typedef float floatx2 __attribute__((ext_vector_type(2)));
    const int skip = KInner ? k0 : k0 * P;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)(p + (k0 < K ? skip : 0)), 0, k0 < K ? (P * K - skip) * 4 : 0, 0x00020000);
    if constexpr (KInner) {
#pragma unroll
      for (int y = 0; y < TP; ++y)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const floatx4 v = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(rs, offset[y] + 64 * h, 0, 0));
#pragma unroll
          for (int e = 0; e < 4; ++e) value[y][4 * h + e] = v[e];
        }
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if constexpr (TP == 4) {
          const floatx4 v = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(rs, offset[j], 0, 0));
#pragma unroll
          for (int y = 0; y < 4; ++y) value[y][j] = v[y];
        } else if constexpr (TP == 2) {
          const floatx2 v = __builtin_bit_cast(floatx2, __builtin_amdgcn_raw_buffer_load_b64(rs, offset[j], 0, 0));
#pragma unroll
          for (int y = 0; y < 2; ++y) value[y][j] = v[y];
        } else {
          value[0][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, offset[j], 0, 0));
        }
      }
    }
  }
  // zeros behind the end of a row, where the next one begins
  __device__ __forceinline__ void cut(int k0) {
    if constexpr (KInner && K % 32 != 0) {
      if (k0 + 32 > K) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const bool is = k0 + point(group, j) < K;
#pragma unroll
          for (int y = 0; y < TP; ++y) value[y][j] = is ? value[y][j] : 0.0f;
        }
      }
    }
  }
  __device__ __forceinline__ bool isUnfit() const {
    bool is = false;
#pragma unroll
    for (int y = 0; y < TP; ++y)
#pragma unroll
      for (int j = 0; j < 8; ++j) is |= isUnfitValue(value[y][j]);
    return is;
  }
};

// Outputs whose sums are in doubt: how many, and the first ones.
constexpr int kMostNoted = 256, kSampledTerms = 16;
__device__ __forceinline__ void note(ldsint* noted, int output) {
  const int at = __hip_atomic_fetch_add(noted, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  if (at < kMostNoted) noted[1 + at] = output;
}
template <bool Bias, bool AKInner, bool BKInner, int M, int N, int K, int TA, int TB, int GA, int GB, int S> struct SlicedProduct {
  static_assert((AKInner || TA == 1 || TA == 2 || TA == 4) && (TB == 1 || TB == 2 || TB == 4), "positions a lane loads at once");
  static constexpr int kRowsOfBlock = 16 * TA * GA, kColumnsOfBlock = 16 * TB * GB;
  static constexpr int kRows = (M + kRowsOfBlock - 1) / kRowsOfBlock, kColumns = (N + kColumnsOfBlock - 1) / kColumnsOfBlock, kBlocks = kRows * kColumns;
  static constexpr int kPitch = 16 * TB + 4, kTile = 16 * TA * kPitch, kLds = 4 * GA * GB * S * kTile; // (floats of a row and a tile of partial sums, bytes of all)
  static_assert(kLds >= 4 * (128 + kRowsOfBlock + kColumnsOfBlock + 1 + kMostNoted), "what doubts are looked into with");
  static constexpr int kTurns = ((K + 31) / 32 + S - 1) / S;
  static constexpr int kVectors = 4 * TB, kUnits = 16 * TA * kVectors / 64, kShare = (kUnits + S - 1) / S; // 16-byte vectors of a row, 64 of them, of a slice
  // The sums of a wavefront's steps: of the parts of the floats, or of the floats themselves.
  template <bool InParts> static __device__ __forceinline__ void multiply(SlicedOperand<AKInner, M, K, TA>& a, SlicedOperand<BKInner, N, K, TB>& b, int slice,
                                                                          floatx4 (&sum)[TB][TA], SplitRange (&rangeA)[TA], SplitRange (&rangeB)[TB]) {
    // (small products have sums of their own where the registers hold them)
    constexpr int kSums = InParts && TA * TB < 16 ? 2 : 1;
    floatx4 sums[kSums][TB][TA];
#pragma unroll
    for (int d = 0; d < kSums; ++d)
#pragma unroll
      for (int x = 0; x < TB; ++x)
#pragma unroll
        for (int y = 0; y < TA; ++y) sums[d][x][y] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    a.load(32 * slice);
    b.load(32 * slice);
#pragma unroll 1
    for (int t = 0; t < kTurns; ++t) {
      const int k0 = 32 * (slice + t * S);
      if constexpr (InParts) {
        SplitParts pa[TA], pb[TB];
        a.cut(k0);
#pragma unroll
        for (int y = 0; y < TA; ++y) pa[y] = splitFloats(a.value[y], rangeA[y]);
        // (or the scheduler puts the loads in front of the last uses of what they overwrite, and waits for them at the end of the turn)
        __builtin_amdgcn_sched_barrier(0);
        a.load(k0 + 32 * S);
        b.cut(k0);
#pragma unroll
        for (int x = 0; x < TB; ++x) pb[x] = splitFloats(b.value[x], rangeB[x]);
        b.load(k0 + 32 * S);
#pragma unroll
        for (int x = 0; x < TB; ++x)
#pragma unroll
          for (int q = 0; q < kSplitProducts; ++q)
#pragma unroll
            for (int y = 0; y < TA; ++y) {
              floatx4& sum = sums[q == kSplitProducts - 1 ? 0 : kSums - 1][x][y];
              sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pb[x].part[splitPartB(q)], pa[y].part[splitPartA(q)], sum, 0, 0, 0);
            }
      } else {
        a.cut(k0);
        b.cut(k0);
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
          for (int x = 0; x < TB; ++x)
#pragma unroll
            for (int y = 0; y < TA; ++y) sums[0][x][y] = __builtin_amdgcn_mfma_f32_16x16x4f32(b.value[x][j], a.value[y][j], sums[0][x][y], 0, 0, 0);
        a.load(k0 + 32 * S);
        b.load(k0 + 32 * S);
      }
    }
#pragma unroll
    for (int x = 0; x < TB; ++x)
#pragma unroll
      for (int y = 0; y < TA; ++y) {
        sum[x][y] = sums[0][x][y];
        if constexpr (kSums == 2) sum[x][y] += sums[1][x][y];
      }
  }
  // Where the i-th vector of a lane's share is in a tile.
  static __device__ __forceinline__ int place(int slice, int i, int lane) {
    const int unit = tmin(slice * kShare + i, kUnits - 1) * 64 + lane;
    return unit / kVectors * kPitch + unit % kVectors * 4;
  }
  // Adds the slices of a rectangle of tiles; a lane gets its share of them, vectors of four neighbouring columns.
  static __device__ __forceinline__ void meet(const floatx4 (&mine)[TB][TA], const SlicedOperand<AKInner, M, K, TA>& a, int wave, int slice, int lane, ldschar* lds, floatx4 (&sum)[kShare]) {
    const int r = lane & 15, g = lane >> 4;
    // A lane holds columns 4 g ... 4 g + 3 of its tiles, in whatever order the tiles hold the positions: four neighbouring ones in LDS.
    ldsfloat* const tile = (ldsfloat*)lds + wave * kTile;
#pragma unroll
    for (int y = 0; y < TA; ++y) {
      ldsfloat* row = tile + a.position(y, r) * kPitch;
#pragma unroll
      for (int x = 0; x < TB; ++x) {
        if constexpr (BKInner) {
          *(ldsfloatx4*)(row + 16 * x + 4 * g) = mine[x][y];
        } else {
          floatx4 v;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = mine[(4 * x + e) % TB][y][(4 * x + e) / TB];
          *(ldsfloatx4*)(row + 4 * TB * g + 4 * x) = v;
        }
      }
    }
    __syncthreads();
    const ldsfloat* from = (const ldsfloat*)lds + (wave - slice) * kTile;
#pragma unroll
    for (int i = 0; i < kShare; ++i) {
      const ldsfloat* at = from + place(slice, i, lane);
      sum[i] = *(const ldsfloatx4*)at;
#pragma unroll
      for (int s = 1; s < S; ++s) sum[i] += *(const ldsfloatx4*)(at + s * kTile);
    }
  }
  static __device__ __forceinline__ void run(float* pO, const float* pA, const float* pB, const float* pBias, ldschar* lds) {
    const int lane = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(threadIdx.y);
    const int r = lane & 15, g = lane >> 4, slice = wave % S, ga = wave / S % GA, gb = wave / S / GA;
    // Blocks go round-robin to the 8 XCDs: each takes a run of them in stripes of four block columns, which share rows in its L2.
    const int id = blockIdx.x + gridDim.x * blockIdx.y, xcd = id & 7, run = xcd * (kBlocks / 8) + tmin(xcd, kBlocks % 8) + (id >> 3);
    const int stripe = run / (4 * kRows), width = tmin(4, kColumns - 4 * stripe), in = run - stripe * 4 * kRows;
    const int m0 = in / width * kRowsOfBlock + 16 * TA * ga, n0 = (4 * stripe + in % width) * kColumnsOfBlock + 16 * TB * gb;
    SlicedOperand<AKInner, M, K, TA> a;
    SlicedOperand<BKInner, N, K, TB> b;
    a.init(pA, m0, lane);
    b.init(pB, n0, lane);
    floatx4 mine[TB][TA], sum[kShare];
    SplitRange rangeA[TA], rangeB[TB];
    multiply<true>(a, b, slice, mine, rangeA, rangeB);
    ldsint* const flags = (ldsint*)lds + 16 * TB; // (behind the first row of the first tile, where no sum is)
    if (wave == 0 && lane < 4) flags[lane] = 0;
    meet(mine, a, wave, slice, lane, lds, sum);
    bool doubtful = false, again = false;
#pragma unroll
    for (int y = 0; y < TA; ++y) doubtful |= rangeA[y].isDoubtful();
#pragma unroll
    for (int x = 0; x < TB; ++x) doubtful |= rangeB[x].isDoubtful();
#pragma unroll
    for (int i = 0; i < kShare; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) doubtful |= isDoubtfulSum(sum[i][e]);
    if (isAnyOfBlock(doubtful, flags)) {
      // A sum that cancels has larger ones of its slices in it.
      floatx4 largest[kShare];
#pragma unroll
      for (int i = 0; i < kShare; ++i) {
        const ldsfloat* at = (const ldsfloat*)lds + (wave - slice) * kTile + place(slice, i, lane);
        largest[i] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
        for (int s = 0; s < S; ++s)
#pragma unroll
          for (int e = 0; e < 4; ++e) largest[i][e] = __builtin_fmaxf(largest[i][e], __builtin_fabsf(at[s * kTile + e]));
      }
      __syncthreads();
      ldsfloat* const most = (ldsfloat*)lds + 128; // of the block's rows, of its columns (where partial sums were)
      for (int i = lane + 64 * wave; i <= kRowsOfBlock + kColumnsOfBlock; i += 64 * GA * GB * S) most[i] = 0.0f; // (and the count behind them)
      __syncthreads();
#pragma unroll
      for (int y = 0; y < TA; ++y) raiseTo(most + 16 * TA * ga + a.position(y, r), rangeA[y].most);
#pragma unroll
      for (int x = 0; x < TB; ++x) raiseTo(most + kRowsOfBlock + 16 * TB * gb + b.position(x, r), rangeB[x].most);
      __syncthreads();
      ldsint* const noted = (ldsint*)(most + kRowsOfBlock + kColumnsOfBlock);
#pragma unroll
      for (int i = 0; i < kShare; ++i) {
        const int unit = tmin(slice * kShare + i, kUnits - 1) * 64 + lane;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          again |= isUnfitSum(sum[i][e]);
          const int row = 16 * TA * ga + unit / kVectors, column = 16 * TB * gb + unit % kVectors * 4 + e;
          if (isUnsureSum(largest[i][e], most[row], most[kRowsOfBlock + column])) note(noted, row * kColumnsOfBlock + column);
        }
      }
      again = isAnyOfBlock(again, flags + 1);
      doubtful = !again && *noted != 0;
      if (doubtful && *noted <= kMostNoted) { // or larger terms
        bool isSure = true;
        for (int i = lane + 64 * wave; i < *noted; i += 64 * GA * GB * S) {
          const int output = noted[1 + i], row = output / kColumnsOfBlock, column = output % kColumnsOfBlock;
          const int m = tmin(m0 - 16 * TA * ga + row, M - 1), n = tmin(n0 - 16 * TB * gb + column, N - 1);
          bool is = false;
#pragma unroll
          for (int j = 0; j < kSampledTerms; ++j) {
            const int k = (i + j * (K / kSampledTerms | 1)) % K;
            is |= !isUnsureSum(pA[AKInner ? m * K + k : k * M + m] * pB[BKInner ? n * K + k : k * N + n], most[row], most[kRowsOfBlock + column]);
          }
          isSure &= is;
        }
        doubtful = isAnyOfBlock(!isSure, flags + 2);
      }
    } else {
      doubtful = false;
    }
    if (doubtful) {
#pragma unroll 1
      for (int t = 0; t < kTurns; ++t) {
        const int k0 = 32 * (slice + t * S);
        a.load(k0);
        b.load(k0);
        again |= a.isUnfit() || b.isUnfit(); // (what lies behind the end of a row is of the next one: at worst a block too many computes again)
      }
      again = isAnyOfBlock(again, flags + 3);
    }
    if (again) {
      multiply<false>(a, b, slice, mine, rangeA, rangeB);
      meet(mine, a, wave, slice, lane, lds, sum);
    }
    typedef unsigned uintx4 __attribute__((ext_vector_type(4)));
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)pO, 0, M * N * 4, 0x00020000);
#pragma unroll
    for (int i = 0; i < kShare; ++i) {
      if (kUnits % kShare != 0 && slice * kShare + i >= kUnits) continue;
      if (kShare * S > kUnits && slice * kShare + i >= kUnits) continue;
      const int unit = (slice * kShare + i) * 64 + lane, m = m0 + unit / kVectors, n = n0 + unit % kVectors * 4;
      if (M % kRowsOfBlock != 0 && m >= M) continue;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (Bias) sum[i][e] += pBias[tmin(n + e, N - 1)];
      }
      if (N % kColumnsOfBlock == 0 || n + 4 <= N) {
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(uintx4, sum[i]), rs, (m * N + n) * 4, 0, 16);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (n + e < N) __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, (float)sum[i][e]), rs, (m * N + n + e) * 4, 0, 16);
        }
      }
    }
  }
};
}
)HIP";

} // namespace hip
} // namespace tc
