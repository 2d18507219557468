// Implicit-GEMM convolution for problems that fill the chip: tiles of 256
// pixels x 192 or 256 channels, fp16 and fp8.
//
// GEMM view, packed weights, row table and tap masks as in igemm.hip.  What a
// large problem costs is the matrix pipe, and what keeps it waiting is the
// operand traffic: a 128 x 128 tile reads 64 KB of LDS and fetches 32 KB per
// 4.2 MFLOP k-step, about as long as its MFMAs take.  A 256 x 256 tile halves
// both per flop.  So here:
//  * all eight waves multiply, two to a SIMD covering each other's waits: 4 (M)
//    x 2 (N), each a 64 x BN / 2 piece of the tile; all eight fetch, too -
//    4 + BN / 64 loads of 1 KB per wave and k-step, straight into LDS;
//  * two LDS stages of a k-step each.  A stage's loads go out as soon as the
//    last wave has read it, behind the k-step's one barrier, and have a whole
//    k-step (2 048 cycles of MFMAs in a 256 x 256 tile) to land;
//  * LDS reads of sub-step s + 1 are issued under the MFMAs of sub-step s, over
//    the barrier too: it stands before a k-step's last sub-step, whose MFMAs
//    cover the next one's first reads.
// Workgroups are dealt to an XCD in blocks of 4 M tiles, whose input rows and
// weights its L2 then fetches once for all of them.
//
// Measured, fp16, us, tiles of 128 x 128 (two to a CU) and these in turn: 4096 x
// 4096 x 4096 133.0 -> 118.6 (1.16 PFLOP/s), 8192 x 8192 x 8192 1263 -> 866
// (1.27), N = 64, 56 x 56, 3 x 3 stride 2, 256 -> 512 137 -> 124, and N = 71,
// 35 x 35, 3 x 3, 624 -> 136 in tiles of 192 channels 258 -> 213.  What bounds
// it: in 4096 x 4096 x 4096 the matrix pipe is busy 64 % of the chip's cycles,
// at a clock of 1.71 GHz where the chip goes to 2.4 - its power limit, under
// which a loop of nothing but MFMAs holds 1.97.  Tiles of 256 x 128 gained
// nothing over 128 x 128 ones with two workgroups to a CU.
#include "igemm_common.hpp"

namespace mxk {
namespace {

constexpr int kWideM = 256;
constexpr int kWideGroup = 4; // M tiles of a block of workgroups

template <int TN> constexpr int wideStageBytes() {
  return (kWideM + 64 * TN) * kRowBytes;
}
template <int TN, class OutT> constexpr int wideLdsBytes() {
  constexpr int loop = 2 * wideStageBytes<TN>() + kWideM * int(sizeof(uint2));
  constexpr int epilogue =
      128 * (64 * TN * int(sizeof(OutT)) + 16) + 64 * TN * int(sizeof(float));
  return loop > epilogue ? loop : epilogue;
}

/// UNI: every k-step lies inside one kernel tap.  TN: 32-channel blocks of a
/// wave, BN = 64 TN.
template <int EB, int FA, int FB, int TN, bool UNI, class OutT>
__device__ __forceinline__ void
wideTile(const IgemmArgs &a, const char *__restrict__ in,
         const char *__restrict__ w, const OutT *__restrict__ bias,
         OutT *__restrict__ out, float scale, uint32_t block,
         uint32_t blocks) {
  constexpr int BN = 64 * TN;
  constexpr int kStage = wideStageBytes<TN>();
  constexpr int ALOADS = kWideM / 64, BLOADS = TN; // per wave and k-step
  extern __shared__ __align__(16) char lds[];
  uint2 *rowTable = reinterpret_cast<uint2 *>(lds + 2 * kStage);
  const IgemmDesc &d = a.d;
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int wm = wave >> 1, wn = wave & 1;

  // workgroup -> (group of convolution, block of M tiles, N tile, M tile)
  const uint32_t tile = xcdSwizzle(block, blocks);
  const uint32_t perGroup = a.mTiles * a.nTiles;
  const uint32_t g = a.divMTiles(a.divNTiles(tile));
  const uint32_t within = tile - g * perGroup;
  const uint32_t mBlock = a.divWideBlock(within);
  const uint32_t inBlock = within - mBlock * (kWideGroup * a.nTiles);
  const uint32_t mLeft = a.mTiles - mBlock * kWideGroup;
  uint32_t nTile, mTile;
  if (mLeft >= kWideGroup) {
    nTile = inBlock / kWideGroup, mTile = inBlock % kWideGroup;
  } else {
    nTile = inBlock / mLeft, mTile = inBlock - nTile * mLeft;
  }
  mTile += mBlock * kWideGroup;

  const uint32_t firstImage =
      a.divOutD(a.divOutH(a.divOutW(mTile * kWideM)));
  const uint32_t ciBytes = d.inChansPerGroup * EB;
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

  // Load r of this wave fills the 8-row block r * 8 + wave of a tile, lane l
  // row position l / 8 and chunk position l % 8 of it.
  const int rowInBlock = (lane >> 3) ^ (wave & 1);
  const int chunk = (lane & 7) ^ rowInBlock;
  const uint32_t bOff = (g * a.coPadded + nTile * BN + wave * 8 + rowInBlock) *
                            a.kPadded * EB +
                        chunk * 16;
  const uint32_t bStep = 64 * a.kPadded * EB; // 64 rows on
  uint32_t kByte = 0;
  auto loadBOne = [&](char *__restrict__ into, int r) {
    loadToLds(wBuf, (LdsPtr)(into + (kWideM + wave * 8 + r * 64) * kRowBytes),
              bOff | (kByte < a.kPadded * EB ? 0u : kOutOfRange),
              r * bStep + kByte);
    if (r == BLOADS - 1)
      kByte += kRowBytes;
  };
  auto loadB = [&](char *__restrict__ into) {
#pragma unroll
    for (int r = 0; r != BLOADS; ++r)
      loadBOne(into, r);
  };
  loadB(lds);

  // The row table: per output pixel the byte offset of the input element
  // under tap (0, 0), and the complement of the taps that read inside.
  if (t < kWideM) {
    const uint32_t m = mTile * kWideM + t;
    const bool rowValid = m < a.M;
    const uint32_t mm = rowValid ? m : 0;
    const uint32_t q = a.divOutW(mm), ow = mm - q * d.outW;
    const uint32_t q2 = a.divOutH(q), oh = q - q2 * d.outH;
    const uint32_t image = a.divOutD(q2), od = q2 - image * d.outD;
    const uint32_t b = image - firstImage;
    const int idBase = int(od * d.strideD) - d.padD;
    const int ihBase = int(oh * d.strideH) - d.padH;
    const int iwBase = int(ow * d.strideW) - d.padW;
    const uint32_t offset =
        shift +
        (((b * d.inD + uint32_t(idBase)) * d.inH + uint32_t(ihBase)) * d.inW +
         uint32_t(iwBase)) *
            pixelBytes +
        g * ciBytes;
    rowTable[t] =
        uint2{offset, rowValid ? ~tapMaskOf(a, idBase, ihBase, iwBase) : ~0u};
  }
  __syncthreads();
  uint32_t rowOff[ALOADS], noTap[ALOADS];
#pragma unroll
  for (int r = 0; r != ALOADS; ++r) {
    const uint2 e = rowTable[(r * 8 + wave) * 8 + rowInBlock];
    rowOff[r] = e.x + chunk * 16;
    noTap[r] = e.y;
  }

  // Position inside K of the input data loaded next: wave-uniform where a
  // k-step lies inside one tap, this lane's own chunk's elsewhere.
  uint32_t aByte = UNI ? 0 : chunk * 16;
  uint32_t tap = a.divCiBytes(aByte), ciOff = aByte - tap * ciBytes;
  uint32_t kRow = a.divKW(tap), kw = tap - kRow * d.kW;
  uint32_t kd = a.divKH(kRow), kh = kRow - kd * d.kH;
  // the tap's place in the input, its bit of noTap (or a tap beyond the
  // kernel) on the way to bit 31
  uint32_t tapOff, toTop, never;
  auto place = [&] {
    tapOff = ((kd * d.dilD * d.inH + kh * d.dilH) * d.inW + kw * d.dilW) *
             pixelBytes;
    toTop = tap < taps ? 31 - tap : 0;
    never = tap < taps ? 0u : kOutOfRange;
  };
  place();
  auto loadAOne = [&](char *__restrict__ into, int r) {
    const uint32_t outside = ((noTap[r] << toTop) & 0x80000000u) | never;
    LdsPtr dst = (LdsPtr)(into + (wave * 8 + r * 64) * kRowBytes);
    if constexpr (UNI)
      loadToLds(inBuf, dst, (rowOff[r] & 0x7fffffffu) | outside,
                tapOff + ciOff);
    else
      loadToLds(inBuf, dst,
                ((rowOff[r] - chunk * 16 + tapOff + ciOff) & 0x7fffffffu) |
                    outside,
                0);
  };
  auto advance = [&] {
    if constexpr (UNI) {
      ciOff += kRowBytes;
      // (selects, not branches: they run in the middle of the MFMAs)
      const uint32_t next = ciOff >= ciBytes ? 1u : 0u;
      ciOff -= next ? ciBytes : 0u;
      tap += next, kw += next;
      const uint32_t wrapW = kw == d.kW ? 1u : 0u;
      kw = wrapW ? 0u : kw;
      kh += wrapW;
      const uint32_t wrapH = kh == d.kH ? 1u : 0u;
      kh = wrapH ? 0u : kh;
      kd += wrapH;
    } else {
      aByte += kRowBytes;
      tap = a.divCiBytes(aByte);
      ciOff = aByte - tap * ciBytes;
      kRow = a.divKW(tap), kw = tap - kRow * d.kW;
      kd = a.divKH(kRow), kh = kRow - kd * d.kH;
    }
    place();
  };
  auto loadA = [&](char *__restrict__ into) {
#pragma unroll
    for (int r = 0; r != ALOADS; ++r)
      loadAOne(into, r);
    advance();
  };
  loadA(lds);
  loadA(lds + kStage);
  loadB(lds + kStage);

  using M = Mma<EB>;
  constexpr int SS = M::kSubSteps;
  typename M::template Frags<TN> f;
  floatx16 acc[2][TN];
#pragma unroll
  for (int i = 0; i != 2; ++i)
#pragma unroll
    for (int j = 0; j != TN; ++j)
#pragma unroll
      for (int v = 0; v != 16; ++v)
        acc[i][j][v] = 0.0f;
  const int rowOffset = fragmentRowOffset(lane);
  auto operandsOf = [&](const char *stage) {
    const char *tileA = stage + wm * 64 * kRowBytes + rowOffset;
    return FragmentAddress{
        {tileA, tileA + 32 * kRowBytes},
        {lane & 7, lane & 7},
        0,
        stage + (kWideM + wn * (BN / 2)) * kRowBytes + rowOffset,
        lane & 7};
  };
  auto fetch = [&](const char *__restrict__ stage, auto sub) {
    M::template load<decltype(sub)::value, TN>(operandsOf(stage), lane, f);
  };
  auto pin = [] { __builtin_amdgcn_sched_barrier(0); };

  // One k-step: `cur` is multiplied, its first P sub-steps' operands at hand;
  // `next` has been asked for a k-step ago.  Sub-step S asks for the operands
  // of S + P; what goes out under which product is pinned: an operand read
  // under each of the first, behind the barrier a load of the k-step after
  // next (fp8: two).
  constexpr int P = SS / 2, PRODUCTS = 2 * TN, OPERANDS = 2 + TN;
  constexpr int PER = (ALOADS + BLOADS + P * PRODUCTS - 1) / (P * PRODUCTS);
  auto step = [&](char *__restrict__ cur, char *__restrict__ next) {
    const FragmentAddress curAt = operandsOf(cur), nextAt = operandsOf(next);
    staticFor<0, SS>([&](auto sub) {
      constexpr int S = decltype(sub)::value;
      if constexpr (S == SS - P) {
        MXK_WAIT_LGKMCNT0(); // this wave has read all it needs of `cur`
        MXK_WAIT_VMCNT(0);   // its part of `next` has landed
        stepBarrier();
      }
      pin();
      staticFor<0, PRODUCTS>([&](auto product) {
        constexpr int K = decltype(product)::value;
        M::template mulOne<S, K, TN, FA, FB>(f, acc);
        pin();
        if constexpr (K < OPERANDS) {
          if constexpr (S + P < SS)
            M::template loadOne<S + P, K, TN>(curAt, lane, f);
          else
            M::template loadOne<S + P - SS, K, TN>(nextAt, lane, f);
        }
        constexpr int FIRST = ((S - (SS - P)) * PRODUCTS + K) * PER;
        staticFor<0, PER>([&](auto more) {
          constexpr int L = FIRST + decltype(more)::value;
          if constexpr (L >= 0 && L < ALOADS) {
            loadAOne(cur, L);
            if constexpr (L == ALOADS - 1)
              advance();
          } else if constexpr (L >= ALOADS && L < ALOADS + BLOADS) {
            loadBOne(cur, L - ALOADS);
          }
        });
        pin();
      });
    });
  };
  static_assert(OPERANDS <= PRODUCTS, "a place for every operand read");
  MXK_WAIT_VMCNT(ALOADS + BLOADS);
  stepBarrier();
  staticFor<0, P>([&](auto sub) { fetch(lds, sub); });
  // (steps beyond the last load and multiply zeros: an odd count is rounded
  // up, so that the stages are known at compile time)
  for (uint32_t kt = 0; kt < a.kSteps; kt += 2) {
    step(lds, lds + kStage);
    step(lds + kStage, lds);
  }
  MXK_WAIT_VMCNT(0);
  MXK_WAIT_LGKMCNT0();

  // Epilogue, 128 rows of the tile at a time: accumulators (lane = pixel,
  // registers = runs of four channels) to LDS, then whole 16-byte vectors out.
  constexpr int kOutRow = BN * int(sizeof(OutT)) + 16;
  constexpr int kVecElems = 16 / int(sizeof(OutT));
  constexpr int kVecsPerRow = BN / kVecElems;
  const uint32_t outChans = d.groups * d.outChansPerGroup;
  // (the tile's bias as fp32, behind the rows)
  float *biasLds = reinterpret_cast<float *>(lds + 128 * kOutRow);
  __syncthreads();
  if (t < BN) {
    const uint32_t n = nTile * BN + t;
    biasLds[t] = bias && n < d.outChansPerGroup
                     ? Load<OutT>::at(bias, g * d.outChansPerGroup + n, 0)
                     : 0.0f;
  }
#pragma unroll 1
  for (int pass = 0; pass != 2; ++pass) {
    __syncthreads();
    if (wm >> 1 == pass) {
      const uint32_t mRow = lane & 31, nOff4 = (lane >> 5) * 4;
#pragma unroll
      for (int j = 0; j != TN; ++j)
#pragma unroll
        for (int q = 0; q != 4; ++q) {
          const uint32_t nLocal = wn * (BN / 2) + j * 32 + 8 * q + nOff4;
          const floatx4 bv =
              *reinterpret_cast<const floatx4 *>(biasLds + nLocal);
#pragma unroll
          for (int i = 0; i != 2; ++i) {
            const uint32_t mLocal = (wm & 1) * 64 + i * 32 + mRow;
            float v[4];
#pragma unroll
            for (int e = 0; e != 4; ++e)
              v[e] = acc[i][j][q * 4 + e] * scale + bv[e];
            storeOut4(reinterpret_cast<OutT *>(lds + mLocal * kOutRow) + nLocal,
                      v);
          }
        }
    }
    __syncthreads();
    const __amdgpu_buffer_rsrc_t outBuf = bufferOf(out, a.outThrough);
    auto copyOut = [&](auto through) {
      for (int idx = t; idx < 128 * kVecsPerRow; idx += kThreads) {
        const uint32_t mLocal = idx / kVecsPerRow, vec = idx % kVecsPerRow;
        const uint32_t m = mTile * kWideM + pass * 128 + mLocal;
        const uint32_t n = nTile * BN + vec * kVecElems;
        if (m >= a.M || n >= d.outChansPerGroup)
          continue;
        const char *src = lds + mLocal * kOutRow + vec * 16;
        const size_t pixel = outPixel(a, m);
        OutT *dst = out + pixel * outChans + g * d.outChansPerGroup + n;
        if constexpr (decltype(through)::value) {
          storeThrough(outBuf,
                       (uint32_t(pixel) * outChans + g * d.outChansPerGroup +
                        n) * uint32_t(sizeof(OutT)),
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
}

template <int EB, int FA, int FB, int TN, bool UNI, class OutT>
__global__ __launch_bounds__(kThreads, 2) void igemmWideKernel(
    IgemmArgs a, const char *__restrict__ in, const char *__restrict__ w,
    const OutT *__restrict__ bias, OutT *__restrict__ out, float scale) {
  wideTile<EB, FA, FB, TN, UNI, OutT>(a, in, w, bias, out, scale, blockIdx.x,
                                      gridDim.x);
}

template <int EB, int FA, int FB, int TN, bool UNI, class OutT>
hipError_t launchKernel(const IgemmArgs &a, uint32_t blocks, const void *in,
                        const void *w, const void *bias, void *out, float scale,
                        hipStream_t stream) {
  constexpr int kLds = wideLdsBytes<TN, OutT>();
  auto kernel = &igemmWideKernel<EB, FA, FB, TN, UNI, OutT>;
  static const hipError_t attr = hipFuncSetAttribute(
      reinterpret_cast<const void *>(kernel),
      hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
  if (attr != hipSuccess)
    return attr;
  hipLaunchKernelGGL(kernel, dim3(blocks), dim3(kThreads), kLds, stream, a,
                     static_cast<const char *>(in),
                     static_cast<const char *>(w),
                     static_cast<const OutT *>(bias),
                     static_cast<OutT *>(out), scale);
  return hipGetLastError();
}

} // namespace

bool igemmWideTakes(const IgemmDesc &d, int inType, int outType) {
  return (outType == kHalf || outType == kFloat) &&
         (inType == kHalf || inType == kQuarter) &&
         d.blockM == uint32_t(kWideM) &&
         (d.blockN == 192 || d.blockN == 256) &&
         d.splitK == 1 && !d.noTaps && !d.outTransposed &&
         igemmTapAddressing(d) == kMaskTaps && igemmAddressable(d, inType);
}

hipError_t launchIgemmWide(const IgemmArgs &a, int inType, int outType,
                           const void *in, const void *w, const void *bias,
                           void *out, const QuarterInfo &q,
                           hipStream_t stream) {
  if (!igemmWideTakes(a.d, inType, outType))
    return hipErrorInvalidValue;
  const uint64_t blocks = uint64_t(a.mTiles) * a.nTiles * a.d.groups;
  if (blocks == 0)
    return hipSuccess;
  if (blocks > 0x7fffffffull)
    return hipErrorInvalidConfiguration;
  const float scale = inType == kQuarter ? q.scale : 1.0f;
  auto go = [&](auto eb, auto fa, auto fb, auto tn) {
    constexpr int EB = decltype(eb)::value, FA = decltype(fa)::value;
    constexpr int FB = decltype(fb)::value, TN = decltype(tn)::value;
    const bool uni = a.d.inChansPerGroup * EB % kRowBytes == 0;
    const uint32_t n = uint32_t(blocks);
    if (outType == kHalf)
      return uni ? launchKernel<EB, FA, FB, TN, true, __half>(
                       a, n, in, w, bias, out, scale, stream)
                 : launchKernel<EB, FA, FB, TN, false, __half>(
                       a, n, in, w, bias, out, scale, stream);
    return uni ? launchKernel<EB, FA, FB, TN, true, float>(
                     a, n, in, w, bias, out, scale, stream)
               : launchKernel<EB, FA, FB, TN, false, float>(
                     a, n, in, w, bias, out, scale, stream);
  };
  auto width = [&](auto eb, auto fa, auto fb) {
    return a.d.blockN == 192
               ? go(eb, fa, fb, std::integral_constant<int, 3>{})
               : go(eb, fa, fb, std::integral_constant<int, 4>{});
  };
  using Zero = std::integral_constant<int, 0>;
  using One = std::integral_constant<int, 1>;
  if (inType == kHalf)
    return width(std::integral_constant<int, 2>{}, Zero{}, Zero{});
  const bool fa = q.inFormat != kE4M3, fb = q.weightFormat != kE4M3;
  if (!fa && !fb)
    return width(One{}, Zero{}, Zero{});
  if (!fa)
    return width(One{}, Zero{}, One{});
  if (!fb)
    return width(One{}, One{}, Zero{});
  return width(One{}, One{}, One{});
}

} // namespace mxk
