// Implicit-GEMM convolution in tiles of 64 MB pixels x 32 NB channels (fp16):
// a tile height and width close to what the layer has, where tiles of 128 x 128
// and 256 x 192 are filled badly or come in an awkward number.
//
// GEMM view, packed weights, row table, tap masks and the LDS layout of a tile
// as in igemm.hip.  All eight waves fetch and multiply, 4 (M) x 2 (N), each a
// 16 MB x 16 NB piece of the tile in MFMA blocks of 16 x 16:
//  * a k-step is 128 bytes of K, its input rows and weights go straight into
//    one of NS stages of LDS; one barrier to a k-step.  Small tiles keep a whole
//    k-step's operands in registers ahead of it (AHEAD), larger ones half;
//  * K runs over taps and channels without a break: a lane's 16-byte chunk has
//    its own tap, looked up in a table in LDS, so channels that fill no whole
//    k-step cost nothing.
// Workgroups are dealt to an XCD in blocks of 4 M tiles, whose input rows and
// weights its L2 then fetches once for all of them.
//
// Measured, us, the tiles of 128 and 256 pixels of the other kernels and these in
// turn: 4096 x 4096 x 4096 118.2 -> 105.3 (256 x 256: 1.31 PFLOP/s), 1026 x 1080 x
// 4604 23.7 -> 18.1 (192 x 128), N = 47, 44 x 44, 3 x 3 stride 2, 192 -> 136 24.1 ->
// 18.1 (128 x 160), N = 68, 19 x 19, 3 x 3, 160 -> 160 21.8 -> 15.6 (resident patch).
// What bounds it: a k-step of a 128 x 128 tile takes 0.27 us on a full chip with
// neither loads nor LDS reads in it (512 cycles of MFMAs at the clock the chip's
// power leaves), 0.37 with the reads, 0.42 with the loads, 0.51 with both; 1.14,
// 1.28, 1.37 and 1.50 in one of 256 x 256, whose matrix pipe is busy 67 % of the
// cycles at 1.81 GHz.
#include "igemm_common.hpp"

#include <algorithm>

namespace mxk {
namespace {

/// A word of every 64-byte line of a convolution's arguments, asked for together:
/// the compiler fetches an argument where it is first used, and each line's first
/// fetch is a trip to memory (the scalar cache starts a launch cold).
__device__ __forceinline__ void fetchArgs(const IgemmArgs &a) {
  asm volatile("" ::"s"(a.d.groups), "s"(a.d.loH), "s"(a.d.outStepH),
               "s"(a.divOutW.mul), "s"(a.divKW.mul), "s"(a.divKH.mul),
               "s"(a.mTiles), "s"(a.wBytes), "s"(a.divWideBlock.mul));
}

/// The convolution of a fused launch that workgroup `block` belongs to: all the
/// counts compared at once, not one trip each.
__device__ __forceinline__ uint32_t fusedMember(const IgemmFusedArgs &m,
                                                uint32_t block) {
  uint32_t i = 0;
#pragma unroll
  for (uint32_t k = 1; k != kIgemmMaxFused; ++k)
    i += uint32_t(k < m.count) & uint32_t(block >= m.firstBlock[k]);
  return i;
}

/// What a workgroup of convolution i of a fused launch needs besides, fetched with
/// the first line of its arguments.
struct FusedPointers {
  const char *in, *w;
  const void *bias;
  void *out;
  uint32_t first, end;
};
__device__ __forceinline__ FusedPointers fusedPointers(const IgemmFusedArgs &m,
                                                       uint32_t i) {
  const FusedPointers p = {m.in[i],         m.w[i],
                           m.bias[i],       m.out[i],
                           m.firstBlock[i], m.firstBlock[i + 1]};
  fetchArgs(m.a[i]);
  asm volatile("" ::"s"(p.in), "s"(p.w), "s"(p.bias), "s"(p.out), "s"(p.first),
               "s"(p.end));
  return p;
}

constexpr int kFlexGroup = 4; // M tiles of a block of workgroups
constexpr int kFlexTaps = 32; // (kMaskTaps)

template <int MB, int NB, int NS> struct FlexShape {
  static constexpr int H = 64 * MB, W = 32 * NB;
  static constexpr int kStage = (H + W) * kRowBytes;
  static constexpr bool kOdd = W % 64 != 0;
  // behind the stages: where loads that nobody wants go, the row table and
  // the taps' places
  static constexpr int kDead = NS * kStage;
  static constexpr int kRows = kDead + (kOdd ? kLoadBytes : 0);
  static constexpr int kTaps = kRows + H * int(sizeof(uint2));
  static constexpr int kLoop = kTaps + 4 * (kFlexTaps + 1);
  template <class OutT> static constexpr int outRow() {
    return W * int(sizeof(OutT)) + 16;
  }
  // the tile's bias as fp32, behind both what the loop and what the end needs,
  // and where each of its rows goes
  template <class OutT> static constexpr int biasByte() {
    constexpr int end = H * outRow<OutT>();
    return ((kLoop > end ? kLoop : end) + 15) / 16 * 16;
  }
  template <class OutT> static constexpr int rowOutByte() {
    return biasByte<OutT>() + W * int(sizeof(float));
  }
  template <class OutT> static constexpr int ldsBytes() {
    return rowOutByte<OutT>() + H * int(sizeof(uint32_t));
  }
};

__device__ __forceinline__ uint16_t loadHalf(__amdgpu_buffer_rsrc_t from,
                                             uint32_t byte) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_raw_buffer_load_b16(from, byte, 0, 0);
#else
  return 0;
#endif
}

/// AHEAD: operands are read a whole k-step ahead.  SPLIT: one part of K, whose
/// fp32 sums go to a workspace [part][pixel][channel], without a bias.
template <int MB, int NB, int NS, bool AHEAD, bool SPLIT, class OutT>
__device__ __forceinline__ void
flexTile(const IgemmArgs &a, const char *__restrict__ in,
         const char *__restrict__ w, const OutT *__restrict__ bias,
         OutT *__restrict__ out, uint32_t block, uint32_t blocks) {
  using Shape = FlexShape<MB, NB, NS>;
  constexpr int H = Shape::H, W = Shape::W, kStage = Shape::kStage;
  constexpr int ALOADS = MB, BLOADS = (W + 63) / 64; // per wave and k-step
  extern __shared__ __align__(16) char lds[];
  uint2 *rowTable = reinterpret_cast<uint2 *>(lds + Shape::kRows);
  uint32_t *tapTable = reinterpret_cast<uint32_t *>(lds + Shape::kTaps);
  float *biasLds = reinterpret_cast<float *>(lds + Shape::template biasByte<OutT>());
  fetchArgs(a);
  uint32_t *rowOut =
      reinterpret_cast<uint32_t *>(lds + Shape::template rowOutByte<OutT>());
  const IgemmDesc &d = a.d;
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int wm = wave >> 1, wn = wave & 1;

  // workgroup -> (part of K, group of convolution, block of M tiles, N tile, M
  // tile)
  const uint32_t tile = xcdSwizzle(block, blocks);
  const uint32_t partGroup = a.divMTiles(a.divNTiles(tile));
  const uint32_t part = SPLIT ? a.divGroups(partGroup) : 0;
  const uint32_t g = partGroup - part * d.groups;
  const uint32_t within = tile - partGroup * (a.mTiles * a.nTiles);
  const uint32_t mBlock = a.divWideBlock(within);
  const uint32_t inBlock = within - mBlock * (kFlexGroup * a.nTiles);
  const uint32_t mLeft = a.mTiles - mBlock * kFlexGroup;
  uint32_t nTile, mTile;
  if (mLeft >= kFlexGroup) {
    nTile = inBlock / kFlexGroup, mTile = inBlock % kFlexGroup;
  } else {
    nTile = inBlock / mLeft, mTile = inBlock - nTile * mLeft;
  }
  mTile += mBlock * kFlexGroup;

  const uint32_t firstImage = a.divOutD(a.divOutH(a.divOutW(mTile * H)));
  const uint32_t ciBytes = d.inChansPerGroup * 2;
  const uint32_t pixelBytes = d.groups * ciBytes;
  const uint32_t taps = d.kD * d.kH * d.kW;
  // (the buffer starts `shift` bytes before the tensor: igemm.hip)
  const uint32_t shift = ((uint32_t(d.padD > 0 ? d.padD : 0) * d.inH +
                           uint32_t(d.padH > 0 ? d.padH : 0)) *
                              d.inW +
                          uint32_t(d.padW > 0 ? d.padW : 0)) *
                         pixelBytes;
  const uint64_t skipped = uint64_t(firstImage) * a.imageBytes;
  const uint64_t left = a.inBytes - skipped + shift;
  const __amdgpu_buffer_rsrc_t inBuf =
      bufferOf(in + skipped - shift,
               uint32_t(left < kOutOfRange - 1 ? left : kOutOfRange - 1));
  const __amdgpu_buffer_rsrc_t wBuf = bufferOf(w, a.wBytes);

  // The bias: asked for first, into LDS in front of the loop.  (The parts' sum
  // adds it where K is split.)
  // (without a bias its buffer is empty and reads as zeros)
  const uint32_t biasChan = nTile * W + t;
  const uint16_t biasOwn = loadHalf(
      bufferOf(bias, bias && !SPLIT ? d.groups * d.outChansPerGroup * 2 : 0),
      t < W && biasChan < d.outChansPerGroup
          ? (g * d.outChansPerGroup + biasChan) * 2
          : kOutOfRange);

  // Load r of this wave fills the 8-row block r * 8 + wave of a tile, lane l
  // row position l / 8 and chunk position l % 8 of it.
  const int rowInBlock = (lane >> 3) ^ (wave & 1);
  const uint32_t chunk = (lane & 7) ^ rowInBlock;
  const uint32_t bOff = (g * a.coPadded + nTile * W + wave * 8 + rowInBlock) *
                            a.kPadded * 2 +
                        chunk * 16;
  const uint32_t bStep = 64 * a.kPadded * 2; // 64 rows on
  const uint32_t kFirst = part * a.kSteps * kRowBytes;
  uint32_t kByte = kFirst;
  auto loadBOne = [&](char *__restrict__ into, int r) {
    char *dst = into + (H + wave * 8 + r * 64) * kRowBytes;
    uint32_t outside = kByte < a.kPadded * 2 ? 0u : kOutOfRange;
    if (Shape::kOdd && r == BLOADS - 1 && wave >= 4) {
      // (rows beyond the tile: every wave issues as many loads)
      outside = kOutOfRange;
      dst = lds + Shape::kDead;
    }
    loadToLds(wBuf, (LdsPtr)dst, bOff | outside, r * bStep + kByte);
    if (r == BLOADS - 1)
      kByte += kRowBytes;
  };

  // (the first stage's weights are on their way while the tables are made)
#pragma unroll
  for (int r = 0; r != BLOADS; ++r)
    loadBOne(lds, r);

  // The row table: per output pixel the byte offset of the input element
  // under tap (0, 0) - and the pixel's place in the output - by one thread, the
  // complement of the taps that read inside by another; and every tap's place
  // in the input.  (Places of mapped outputs worked out when they are stored,
  // three divisions to a vector: N = 42, 35 x 35, 3 x 3 stride 2, 136 -> 80
  // backwards 10.8 us, 10.2 so; 25 x 57 x 57, 72 -> 200 20.2 and 19.5.)
  const uint32_t half = uint32_t(t) / (kThreads / 2);
  const uint32_t row = uint32_t(t) % (kThreads / 2);
  if (row < H) {
    const uint32_t m = mTile * H + row;
    const bool rowValid = m < a.M;
    const uint32_t mm = rowValid ? m : 0;
    const uint32_t q = a.divOutW(mm), ow = mm - q * d.outW;
    const uint32_t q2 = a.divOutH(q), oh = q - q2 * d.outH;
    const uint32_t image = a.divOutD(q2), od = q2 - image * d.outD;
    const int idBase = int(od * d.strideD) - d.padD;
    const int ihBase = int(oh * d.strideH) - d.padH;
    const int iwBase = int(ow * d.strideW) - d.padW;
    if (half == 0) {
      const uint32_t b = image - firstImage;
      rowTable[row].x =
          shift +
          (((b * d.inD + uint32_t(idBase)) * d.inH + uint32_t(ihBase)) *
               d.inW +
           uint32_t(iwBase)) *
              pixelBytes +
          g * ciBytes;
      uint32_t pixel = m;
      if (a.outMapped)
        pixel = ((image * d.outFullD + od * d.outStepD + d.outOffD) *
                     d.outFullH +
                 oh * d.outStepH + d.outOffH) *
                    d.outFullW +
                ow * d.outStepW + d.outOffW;
      rowOut[row] = rowValid ? pixel : ~0u;
    } else {
      rowTable[row].y =
          rowValid ? ~tapMaskOf(a, idBase, ihBase, iwBase) : ~0u;
    }
  }
  if (uint32_t(kThreads - 1 - t) <= taps) {
    const uint32_t tap = kThreads - 1 - t;
    const uint32_t kRow = a.divKW(tap), kw = tap - kRow * d.kW;
    const uint32_t kd = a.divKH(kRow), kh = kRow - kd * d.kH;
    tapTable[tap] =
        tap < taps
            ? ((kd * d.dilD * d.inH + kh * d.dilH) * d.inW + kw * d.dilW) *
                  pixelBytes
            : kOutOfRange;
  }
  __syncthreads();
  uint32_t rowOff[ALOADS], noTap[ALOADS];
#pragma unroll
  for (int r = 0; r != ALOADS; ++r) {
    const uint2 e = rowTable[(r * 8 + wave) * 8 + rowInBlock];
    rowOff[r] = e.x;
    noTap[r] = e.y;
  }

  // Where in K the input data loaded next is, this lane's own chunk of it: tap
  // and byte within the tap's channels; `place`: the two in the input, with
  // the top bit for a tap beyond the kernel.
  uint32_t tap = a.divCiBytes(kFirst + chunk * 16);
  uint32_t ciOff = kFirst + chunk * 16 - tap * ciBytes;
  const uint32_t stepTaps = a.divCiBytes(kRowBytes);
  const uint32_t stepBytes = kRowBytes - stepTaps * ciBytes;
  uint32_t toTop, place;
  auto look = [&] {
    const uint32_t known = tap < taps ? tap : taps;
    toTop = 31 - known;
    place = tapTable[known];
  };
  look();
  auto advance = [&] {
    ciOff += stepBytes;
    const uint32_t next = ciOff >= ciBytes ? 1u : 0u;
    ciOff -= next ? ciBytes : 0u;
    tap += stepTaps + next;
    look();
  };
  auto loadAOne = [&](char *__restrict__ into, int r) {
    const uint32_t outside = (noTap[r] << (toTop & 31)) | place;
    loadToLds(inBuf, (LdsPtr)(into + (wave * 8 + r * 64) * kRowBytes),
              ((rowOff[r] + place + ciOff) & 0x7fffffffu) |
                  (outside & 0x80000000u),
              0);
  };
  constexpr int PRODUCTS = MB * NB, OPERANDS = MB + NB;
  constexpr int LOADS = ALOADS + BLOADS;
  // A k-step's loads go out evenly spaced under the products of a whole k-step -
  // of its second half with two stages: a wave whose load has to wait for its
  // turn on the way to LDS multiplies nothing meanwhile (N = 25, 57 x 57, 3 x 3
  // stride 2, 72 -> 200 12.9 us with all of them behind the barrier, 12.5).
  // A k-step has SLOTS slots, and `loadSlot` issues what belongs to one.
  constexpr int SLOTS = NS > 2 || AHEAD ? 2 * PRODUCTS : PRODUCTS;
  auto loadSlot = [&](char *__restrict__ into, auto slot, auto most) {
    constexpr int K = decltype(slot)::value;
    constexpr int MOST = decltype(most)::value;
    constexpr int FROM = (K * LOADS + SLOTS - 1) / SLOTS;
    constexpr int UP = ((K + 1) * LOADS + SLOTS - 1) / SLOTS;
    constexpr int TO = UP < MOST ? UP : MOST;
    staticFor<FROM, TO>([&](auto load) {
      constexpr int L = decltype(load)::value;
      if constexpr (L < ALOADS) {
        loadAOne(into, L);
        if constexpr (L == ALOADS - 1)
          advance();
      } else {
        loadBOne(into, L - ALOADS);
      }
    });
  };
  using All = std::integral_constant<int, LOADS>;
  // The stages before the loop: all of them, or all but what the loop's first
  // half k-step sends.
  constexpr bool ACROSS = NS > 2 && !AHEAD; // over the end of a k-step
  constexpr int LAST = ACROSS ? PRODUCTS : SLOTS;
  constexpr int AHEAD_OF_LAST = (LAST * LOADS + SLOTS - 1) / SLOTS;
  staticFor<0, NS>([&](auto stage) {
    constexpr int N = decltype(stage)::value;
    // (the first stage's weights went out above)
    using Most = std::integral_constant<int, N == 0 ? ALOADS : LOADS>;
    staticFor<0, N == NS - 1 ? LAST : SLOTS>(
        [&](auto slot) { loadSlot(lds + N * kStage, slot, Most{}); });
  });
  if (t < W)
    biasLds[t] = __half2float(__ushort_as_half(biasOwn));

  // Operands: lane l has row l % 16 of a block, and in half h of a k-step
  // 16-byte chunk 2 (l / 16) + h - every second one, because the 16 lanes that
  // LDS serves at a time (0-3, 12-15, 20-27 and so on) are then on all its banks
  // (in a row's order, chunk 4 h + l / 16, half the reads' cycles were conflicts:
  // 1024 x 4096 x 2048 in 128 x 128 tiles 36.6 us, 32.8 so).
  const uint32_t operand =
      ((lane & 15) ^ ((lane >> 3) & 1)) * kRowBytes +
      (((lane >> 4) * 2 ^ (lane & 7)) << 4);
  const uint32_t aAt = wm * 16 * MB * kRowBytes + operand;
  const uint32_t bAt = (H + wn * 16 * NB) * kRowBytes + operand;
  floatx4 acc[MB][NB];
#pragma unroll
  for (int i = 0; i != MB; ++i)
#pragma unroll
    for (int j = 0; j != NB; ++j)
      acc[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
  using Half0 = std::integral_constant<int, 0>;
  using Half1 = std::integral_constant<int, 1>;
  auto pin = [] { __builtin_amdgcn_sched_barrier(0); };
  /// Operands of half a k-step.
  struct Operands {
    half8 a[MB], b[NB];
  };
  auto readOne = [&](Operands &o, const char *__restrict__ stage, auto half,
                     int k) {
    const uint32_t flip = decltype(half)::value * 16;
    if (k < MB)
      o.a[k] = *reinterpret_cast<const half8 *>(stage + (aAt ^ flip) +
                                                k * 16 * kRowBytes);
    else
      o.b[k - MB] = *reinterpret_cast<const half8 *>(
          stage + (bAt ^ flip) + (k - MB) * 16 * kRowBytes);
  };
  auto multiplyOne = [&](const Operands &o, int k) {
    acc[k / NB][k % NB] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
        o.b[k % NB], o.a[k / NB], acc[k / NB][k % NB], 0, 0, 0);
  };
  auto nextStage = [](uint32_t s) {
    return s + kStage == NS * kStage ? 0 : s + kStage;
  };
  MXK_WAIT_LGKMCNT0();
  MXK_WAIT_VMCNT((NS - 2) * LOADS + AHEAD_OF_LAST);
  stepBarrier();
  uint32_t at = 0;
  if constexpr (AHEAD) {
    // A k-step's operands are read a whole k-step ahead: one barrier at its
    // start, behind which the stage read last is free and the one to be read
    // has landed, and nothing in it waits for LDS.
    struct Step {
      Operands half[2];
    };
    Step even, odd;
    auto step = [&](const Step &cur, Step &next, char *__restrict__ freed,
                    const char *__restrict__ from) {
      MXK_WAIT_LGKMCNT0();
      MXK_WAIT_VMCNT((NS - 2) * LOADS);
      stepBarrier();
      pin();
      staticFor<0, 2 * PRODUCTS>([&](auto product) {
        constexpr int K = decltype(product)::value;
        multiplyOne(cur.half[K / PRODUCTS], K % PRODUCTS);
        pin();
        if constexpr (K < OPERANDS) {
          readOne(next.half[0], from, Half0{}, K);
          readOne(next.half[1], from, Half1{}, K);
        }
        loadSlot(freed, product, All{});
        pin();
      });
    };
#pragma unroll
    for (int k = 0; k != OPERANDS; ++k) {
      readOne(even.half[0], lds, Half0{}, k);
      readOne(even.half[1], lds, Half1{}, k);
    }
    uint32_t kt = 0;
    for (; kt + 2 <= a.kSteps; kt += 2) {
      const uint32_t s1 = nextStage(at), s2 = nextStage(s1);
      step(even, odd, lds + at, lds + s1);
      step(odd, even, lds + s1, lds + s2);
      at = s2;
    }
    if (kt < a.kSteps)
      step(even, odd, lds + at, lds + nextStage(at));
  } else {
    // (registers for half a k-step ahead only)  One k-step: `cur` is
    // multiplied, its first half's operands at hand; `next` has been asked for
    // NS - 1 k-steps ago, and what comes after those on the way goes into
    // `cur` behind the barrier.
    static_assert(OPERANDS <= PRODUCTS, "a place for every operand read");
    Operands first, second;
    auto step = [&](char *__restrict__ before, char *__restrict__ cur,
                    const char *__restrict__ next) {
      pin();
      staticFor<0, PRODUCTS>([&](auto product) {
        constexpr int K = decltype(product)::value;
        multiplyOne(first, K);
        pin();
        if constexpr (K < OPERANDS)
          readOne(second, cur, Half1{}, K);
        if constexpr (ACROSS)
          loadSlot(before, std::integral_constant<int, PRODUCTS + K>{},
                     All{});
        pin();
      });
      MXK_WAIT_LGKMCNT0(); // this wave has read all it needs of `cur`
      MXK_WAIT_VMCNT((NS - 2) * LOADS); // its part of `next` has landed
      stepBarrier();
      pin();
      staticFor<0, PRODUCTS>([&](auto product) {
        constexpr int K = decltype(product)::value;
        multiplyOne(second, K);
        pin();
        if constexpr (K < OPERANDS)
          readOne(first, next, Half0{}, K);
        loadSlot(cur, product, All{});
        pin();
      });
    };
#pragma unroll
    for (int k = 0; k != OPERANDS; ++k)
      readOne(first, lds, Half0{}, k);
    uint32_t before = (NS - 1) * kStage;
    for (uint32_t kt = 0; kt < a.kSteps; ++kt) {
      const uint32_t next = nextStage(at);
      step(lds + before, lds + at, lds + next);
      before = at, at = next;
    }
  }
  MXK_WAIT_VMCNT(0);
  MXK_WAIT_LGKMCNT0();

  const uint32_t outChans = d.groups * d.outChansPerGroup;
  const __amdgpu_buffer_rsrc_t outBuf = bufferOf(out, a.outThrough);
  if constexpr (SPLIT) {
    // A lane has four consecutive channels of a pixel: 16 bytes each, 64 of a
    // pixel side by side, straight from the registers.
    float *own = reinterpret_cast<float *>(out) +
                 size_t(part) * a.M * outChans + g * d.outChansPerGroup;
    const __amdgpu_buffer_rsrc_t partBuf =
        bufferOf(own, a.M * outChans * uint32_t(sizeof(float)));
#pragma unroll
    for (int i = 0; i != MB; ++i) {
      const uint32_t m = mTile * H + (wm * MB + i) * 16 + (lane & 15);
#pragma unroll
      for (int j = 0; j != NB; ++j) {
        const uint32_t n = nTile * W + (wn * NB + j) * 16 + (lane >> 4) * 4;
        if (m < a.M && n < d.outChansPerGroup)
          storeThrough(partBuf, (m * outChans + n) * uint32_t(sizeof(float)),
                       __builtin_bit_cast(ThroughWords4, acc[i][j]));
      }
    }
    return;
  }

  // The tile as [H rows][W outputs] (+ 16 bytes of padding per row) into LDS -
  // a lane has four consecutive channels of a pixel - then whole 16-byte
  // vectors out.
  constexpr int kOutRow = Shape::template outRow<OutT>();
  constexpr int kVecElems = 16 / int(sizeof(OutT));
  constexpr int kVecsPerRow = W / kVecElems;
  __syncthreads();
  {
    floatx4 bv[NB];
    const uint32_t n0 = wn * 16 * NB + (lane >> 4) * 4;
#pragma unroll
    for (int j = 0; j != NB; ++j)
      bv[j] = *reinterpret_cast<const floatx4 *>(biasLds + n0 + j * 16);
#pragma unroll
    for (int i = 0; i != MB; ++i) {
      const uint32_t row = (wm * MB + i) * 16 + (lane & 15);
#pragma unroll
      for (int j = 0; j != NB; ++j) {
        float v[4];
#pragma unroll
        for (int e = 0; e != 4; ++e)
          v[e] = acc[i][j][e] + bv[j][e];
        storeOut4(reinterpret_cast<OutT *>(lds + row * kOutRow) + n0 + j * 16,
                  v);
      }
    }
  }
  __syncthreads();
  auto copyOut = [&](auto through) {
    for (int idx = t; idx < H * kVecsPerRow; idx += kThreads) {
      const uint32_t mLocal = idx / kVecsPerRow, vec = idx % kVecsPerRow;
      const uint32_t pixel = rowOut[mLocal];
      const uint32_t n = nTile * W + vec * kVecElems;
      if (pixel == ~0u || n >= d.outChansPerGroup)
        continue;
      const char *src = lds + mLocal * kOutRow + vec * 16;
      OutT *dst = out + size_t(pixel) * outChans + g * d.outChansPerGroup + n;
      if constexpr (decltype(through)::value) {
        storeThrough(outBuf,
                     (pixel * outChans + g * d.outChansPerGroup + n) *
                         uint32_t(sizeof(OutT)),
                     *reinterpret_cast<const uintx4 *>(src));
      } else if (n + kVecElems <= d.outChansPerGroup) {
        const uintx4 whole = *reinterpret_cast<const uintx4 *>(src);
        *reinterpret_cast<AnyWords *>(dst) = whole;
      } else {
        const OutT *e = reinterpret_cast<const OutT *>(src);
        for (int k = 0; k != kVecElems && n + k < d.outChansPerGroup; ++k)
          dst[k] = e[k];
      }
    }
  };
  if (a.outThrough)
    copyOut(std::true_type{});
  else
    copyOut(std::false_type{});
}

/// Whether the registers of a wave hold two k-steps' operands.
constexpr bool flexAhead(int mb, int nb, int perCU) {
    return 16 * (mb + nb) + 4 * mb * nb <= (perCU == 1 ? 128 : 88);
}

/// PER_CU: workgroups that share a CU.
template <int MB, int NB, int NS, int PER_CU, bool SPLIT, class OutT>
__global__ __launch_bounds__(kThreads, 2 * PER_CU) void igemmFlexKernel(
    IgemmArgs a, const char *__restrict__ in, const char *__restrict__ w,
    const OutT *__restrict__ bias, OutT *__restrict__ out) {
  flexTile<MB, NB, NS, flexAhead(MB, NB, PER_CU), SPLIT, OutT>(
      a, in, w, bias, out, blockIdx.x, gridDim.x);
}

/// Several convolutions in one launch, as igemmFusedKernel.
template <int MB, int NB, int NS, int PER_CU, class OutT>
__global__ __launch_bounds__(kThreads, 2 * PER_CU) void igemmFlexFusedKernel(
    IgemmFusedArgs m) {
  const uint32_t i = fusedMember(m, blockIdx.x);
  const FusedPointers p = fusedPointers(m, i);
  flexTile<MB, NB, NS, flexAhead(MB, NB, PER_CU), false, OutT>(
      m.a[i], p.in, p.w, static_cast<const OutT *>(p.bias),
      static_cast<OutT *>(p.out), blockIdx.x - p.first, p.end - p.first);
}

/// Stages of a tile's kernel that has its CU to itself, or shares it (0: the
/// tile is too large for that).
constexpr int flexStages(int mb, int nb, bool shared) {
  const int rows = 64 * mb + 32 * nb;
  if (shared)
    return mb * nb <= 10 && rows <= 288 ? 2 : 0;
  return 155 * 1024 / (rows * kRowBytes) < 6 ? 155 * 1024 / (rows * kRowBytes)
                                             : 6;
}

struct FlexOne {
  const IgemmArgs &a;
  const void *in, *w, *bias;
  void *out;
  hipStream_t stream;
  template <int MB, int NB, int NS, int PER_CU> hipError_t go() const {
    return a.d.splitK > 1 ? run<MB, NB, NS, PER_CU, true>()
                          : run<MB, NB, NS, PER_CU, false>();
  }
  template <int MB, int NB, int NS, int PER_CU, bool SPLIT>
  hipError_t run() const {
    using OutT = __half;
    const uint64_t blocks =
        uint64_t(a.mTiles) * a.nTiles * a.d.groups * a.d.splitK;
    if (blocks == 0)
      return hipSuccess;
    if (blocks > 0x7fffffffull)
      return hipErrorInvalidConfiguration;
    constexpr int kLds = FlexShape<MB, NB, NS>::template ldsBytes<OutT>();
    static_assert(kLds * PER_CU <= 160 * 1024, "a CU's LDS");
    const auto kernel = &igemmFlexKernel<MB, NB, NS, PER_CU, SPLIT, OutT>;
    static const hipError_t attr = raiseLdsLimit(kernel, kLds);
    if (attr != hipSuccess)
      return attr;
    hipLaunchKernelGGL(kernel, dim3(uint32_t(blocks)), dim3(kThreads), kLds,
                       stream, a, static_cast<const char *>(in),
                       static_cast<const char *>(w),
                       static_cast<const OutT *>(bias),
                       static_cast<OutT *>(out));
    return hipGetLastError();
  }
};

struct FlexFused {
  const IgemmFusedArgs &m;
  hipStream_t stream;
  template <int MB, int NB, int NS, int PER_CU> hipError_t go() const {
    const uint32_t blocks = m.firstBlock[m.count];
    if (blocks == 0)
      return hipSuccess;
    constexpr int kLds = FlexShape<MB, NB, NS>::template ldsBytes<__half>();
    const auto kernel = &igemmFlexFusedKernel<MB, NB, NS, PER_CU, __half>;
    static const hipError_t attr = raiseLdsLimit(kernel, kLds);
    if (attr != hipSuccess)
      return attr;
    hipLaunchKernelGGL(kernel, dim3(blocks), dim3(kThreads), kLds, stream, m);
    return hipGetLastError();
  }
};

template <int MB, int NB, class Launch>
hipError_t launchTile(bool shared, const Launch &launch) {
  if constexpr (flexStages(MB, NB, true) != 0) {
    if (shared)
      return launch.template go<MB, NB, flexStages(MB, NB, true), 2>();
  }
  return launch.template go<MB, NB, flexStages(MB, NB, false), 1>();
}

template <int MB, class Launch>
hipError_t launchWidth(const IgemmDesc &d, const Launch &launch) {
  const bool shared = d.flex == 2;
  switch (d.blockN) {
  case 64:
    if constexpr (MB != 4) // (no layer's best)
      return launchTile<MB, 2>(shared, launch);
    return hipErrorInvalidValue;
  case 96:
    return launchTile<MB, 3>(shared, launch);
  case 128:
    return launchTile<MB, 4>(shared, launch);
  case 160:
    return launchTile<MB, 5>(shared, launch);
  case 192:
    return launchTile<MB, 6>(shared, launch);
  case 224:
    return launchTile<MB, 7>(shared, launch);
  case 256:
    return launchTile<MB, 8>(shared, launch);
  }
  return hipErrorInvalidValue;
}

template <class Launch>
hipError_t launchHeight(const IgemmDesc &d, const Launch &launch) {
  switch (d.blockM) {
  case 128:
    return launchWidth<2>(d, launch);
  case 192:
    return launchWidth<3>(d, launch);
  case 256:
    return launchWidth<4>(d, launch);
  }
  return hipErrorInvalidValue;
}

/// Bytes of the weights packed for d's tile width, which a buffer has to reach.
uint64_t flexWeightBytes(const IgemmDesc &d) {
  const uint64_t co =
      (uint64_t(d.outChansPerGroup) + d.blockN - 1) / d.blockN * d.blockN;
  const uint64_t k = (uint64_t(d.kD) * d.kH * d.kW * d.inChansPerGroup + 63) /
                     64 * 64;
  return d.groups * co * k * 2;
}

} // namespace

bool igemmFlexTile(uint32_t blockM, uint32_t blockN, uint32_t flex) {
  return (flex == 1 || flex == 2) &&
         (blockM == 128 || blockM == 192 || blockM == 256) &&
         blockN % 32 == 0 && blockN >= 64 && blockN <= 256 &&
         !(blockM == 256 && blockN == 64) &&
         flexStages(int(blockM / 64), int(blockN / 32), flex == 2) != 0;
}

bool igemmFlexTakes(const IgemmDesc &d, int inType, int outType) {
  return inType == kHalf && outType == kHalf &&
         igemmFlexTile(d.blockM, d.blockN, d.flex) &&
         flexWeightBytes(d) < kOutOfRange &&
         // (whole vectors of fp32 sums, a part of them within a buffer's reach)
         (d.splitK == 1 ||
          (d.outChansPerGroup % 4 == 0 && !d.outFullH && !d.outFullW &&
           uint64_t(d.batch) * d.outD * d.outH * d.outW * d.groups *
                   d.outChansPerGroup * 4 <
               kOutOfRange)) &&
         !d.patch && !d.small && !d.outTransposed &&
         // (places in the output are 32-bit numbers of pixels)
         uint64_t(d.batch) * std::max(d.outFullD, d.outD) *
                 std::max(d.outFullH, d.outH) * std::max(d.outFullW, d.outW) <
             0xffffffffull &&
         igemmTapAddressing(d) == kMaskTaps && igemmAddressable(d, inType);
}

hipError_t launchIgemmFlex(const IgemmArgs &a, const void *in, const void *w,
                           const void *bias, void *out, hipStream_t stream) {
  return launchHeight(a.d, FlexOne{a, in, w, bias, out, stream});
}

hipError_t launchIgemmFlexFused(const IgemmFusedArgs &m, hipStream_t stream) {
  return launchHeight(m.a[0].d, FlexFused{m, stream});
}

} // namespace mxk
