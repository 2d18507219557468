// Implicit-GEMM convolution for problems too small to fill the chip with
// 128-pixel tiles: one image, a deep layer of a small batch, a matrix with few
// rows.
//
// GEMM view as in igemm.hip: M = output pixels, N = output channels, K =
// kernel taps x input channels.  What such a problem costs is latency - the
// launch, one trip to memory for the arguments, one for the operands, one for
// the results - so everything here is laid out for one trip of each kind:
//  * small tiles (16 x 16 to 64 x 32 outputs), so that there are workgroups
//    for the whole chip;
//  * K is split over the 2 to 16 waves of a workgroup, whose sums meet in LDS
//    in a fixed order: no partial tiles in memory, no second kernel;
//  * no start-up table and no producer waves: every wave works out its own
//    operands' addresses and has the loads of two groups of k-steps in flight.
// A k-step is 64 bytes of K: one 16 x 16 MFMA block of fp16 (K = 32), two of
// fp8 or four of fp32.
//
// Operands.  The weights are packed in MFMA operand order, [G][16-channel
// block][k-step][64 lanes][16 bytes], and go to registers with loads of 1 KB
// of consecutive memory.  The pixels go through LDS, in a part of it that is
// the wave's own (no barrier): four lanes bring a pixel's 64 bytes, written as
// [16 pixels][64 bytes] with chunk c of pixel r at position c ^ (r / 4), so
// that the 16 lanes of an operand read cover all 64 banks.  (Read straight
// into registers, neighbouring lanes would ask for 16 different lines.)
// The results are stored through the L2, which has nothing to write back when
// the kernel ends (246 problems of up to 5 MB 1.2 % faster on average).
// Padding, truncation, dilation and a zero-stuffed input are address
// arithmetic: a chunk that meets none of the input gets an offset beyond the
// buffer, for which zeros arrive.
#include "igemm_common.hpp"

namespace mxk {
namespace {

constexpr uint32_t kSmallStepBytes = 64;
constexpr uint32_t kSmallMostWaves = 16;

struct SmallArgs {
  const char *in, *w;
  const void *bias;
  void *out;
  uint64_t inBytes;
  uint32_t M, nTiles, steps, chunks, stepsPerWave, waves;
  uint32_t outChans, co, ciBytes, pixelBytes, rowBytes, imageBytes, wBytes;
  uint32_t loH, spanH, loW, spanW;
  int16_t padH, padW;
  uint16_t strideH, strideW, dilH, dilW;
  uint16_t inDilH, inDilW;
  uint16_t kW, outW, outH;
  // 1: the result as [channel][pixel]; 2: into a larger field
  uint16_t outMode;
  uint32_t outFullH, outFullW, outOffH, outOffW;
  uint32_t outThrough; // bytes of the output, 0 where it is out of a buffer's reach
  float scale;
  uint32_t formats; // fp8: bit 0 input, bit 1 weights in E5M2
  FastDiv divNTiles, divMTiles, divOutW, divOutH, divChunks, divKW;
  FastDiv divInDilH, divInDilW;
};

/// A single tap that always reads inside the input (a 1 x 1 kernel without
/// padding), whose chunks are consecutive; any window; a window over a
/// zero-stuffed input.
enum : int { kSmallOneTap = 0, kSmallWindow = 1, kSmallDilated = 2 };

template <int EB>
__device__ __forceinline__ floatx4 smallMma(uintx4 wv, uintx4 av, floatx4 acc,
                                            uint32_t formats) {
#if defined(__HIP_DEVICE_COMPILE__)
  if constexpr (EB == 2) {
    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(
        __builtin_bit_cast(half8, wv), __builtin_bit_cast(half8, av), acc, 0,
        0, 0);
  } else if constexpr (EB == 4) {
    const floatx4 wf = __builtin_bit_cast(floatx4, wv);
    const floatx4 af = __builtin_bit_cast(floatx4, av);
#pragma unroll
    for (int e = 0; e != 4; ++e)
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[e], af[e], acc, 0, 0, 0);
  } else {
    // which 32 of a step's 64 channels an instruction multiplies does not
    // matter: both operands split the lane's 16 bytes alike
    typedef long longx2 __attribute__((ext_vector_type(2)));
    const longx2 wl = __builtin_bit_cast(longx2, wv);
    const longx2 al = __builtin_bit_cast(longx2, av);
#pragma unroll
    for (int e = 0; e != 2; ++e) {
      if (formats == 0)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(wl[e], al[e], acc, 0,
                                                         0, 0);
      else if (formats == 1)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_fp8_bf8(wl[e], al[e], acc, 0,
                                                         0, 0);
      else if (formats == 2)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf8_fp8(wl[e], al[e], acc, 0,
                                                         0, 0);
      else
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf8_bf8(wl[e], al[e], acc, 0,
                                                         0, 0);
    }
  }
#endif
  return acc;
}

/// Tile of 16 TM pixels x 16 TN channels, U k-steps per group of loads.  TAPS: how a chunk's place in the input is found.
template <int EB, int TM, int TN, int U, int TAPS, class OutT>
__device__ __forceinline__ void igemmSmallTile(const SmallArgs &a,
                                               uint32_t block) {
  // one or two groups of U * TM KB per wave
  extern __shared__ __align__(16) char lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

  // (Named here, the arguments come in the one fetch at the kernel's start; the
  // compiler would fetch some where they are first used, each a round trip.)
  asm volatile("" ::"s"(a.out), "s"(a.inBytes), "s"(a.rowBytes), "s"(a.loH),
               "s"(a.spanW), "s"(a.scale), "s"(a.formats));
  const uint32_t overN = a.divNTiles(block);
  const uint32_t nTile = block - overN * a.nTiles;
  const uint32_t g = a.divMTiles(overN);
  const uint32_t mTiles = (a.M + 16 * TM - 1) / (16 * TM);
  const uint32_t m0 = (overN - g * mTiles) * 16 * TM;

  const uint32_t sBegin = wave * a.stepsPerWave;
  const uint32_t sEnd =
      sBegin + a.stepsPerWave < a.steps ? sBegin + a.stepsPerWave : a.steps;
  const __amdgpu_buffer_rsrc_t wBuf = bufferOf(a.w, a.wBytes);
  struct Weights {
    uintx4 v[U][TN];
  };
  const uint32_t wStart = (g * a.nTiles + nTile) * TN * a.steps * 1024;
  auto loadWeights = [&](uint32_t s0, Weights &wv) {
#pragma unroll
    for (int u = 0; u != U; ++u) {
      const uint32_t s = s0 + u;
      // (beyond the wave's last step: from beyond the buffer, zeros)
      const uint32_t at = lane * 16u | (s < sEnd ? 0u : kOutOfRange);
#pragma unroll
      for (int j = 0; j != TN; ++j)
        wv.v[u][j] = __builtin_amdgcn_raw_buffer_load_b128(
            wBuf, at, wStart + (j * a.steps + (s < sEnd ? s : 0)) * 1024, 0);
    }
  };
  // The part of the result this lane writes in the end - four channels of a
  // pixel of the blocks wave, wave + waves, ..., which are of one column (an
  // even number of waves, up to two columns) - and its bias: asked for now,
  // with the first weights.
  static_assert(TN <= 2, "waves step over whole rows of blocks");
  const uint32_t outN = (nTile * TN + wave % TN) * 16 + 4 * (lane >> 4);
  Weights even, odd;
  loadWeights(sBegin, even);
  // (no bias: an empty buffer, which reads as zeros; kept as loaded - a
  // conversion here would wait for it)
  const __amdgpu_buffer_rsrc_t biasBuf = bufferOf(
      a.bias, a.bias ? a.outChans * uint32_t(sizeof(OutT)) : 0u);
  uint32_t biasRaw[4];
#pragma unroll
  for (int e = 0; e != 4; ++e) {
    const uint32_t at = (g * a.co + outN + e) * uint32_t(sizeof(OutT));
    if constexpr (sizeof(OutT) == 2)
      biasRaw[e] = __builtin_amdgcn_raw_buffer_load_b16(biasBuf, at, 0, 0);
    else
      biasRaw[e] = __builtin_amdgcn_raw_buffer_load_b32(biasBuf, at, 0, 0);
  }

  // This lane's pixel of every 16-pixel block, and its chunk of a k-step.
  const uint32_t row = lane >> 2;
  const uint32_t chunk = (lane & 3) ^ (row >> 2);
  const uint32_t firstImage = a.divOutH(a.divOutW(m0));
  const uint64_t skipped = uint64_t(firstImage) * a.imageBytes;
  const uint64_t left = a.inBytes - skipped;
  const __amdgpu_buffer_rsrc_t inBuf = bufferOf(
      a.in + skipped,
      uint32_t(left < kOutOfRange - 1 ? left : kOutOfRange - 1));
  uint32_t rowOff[TM];
  int originH[TM], originW[TM];
#pragma unroll
  for (int i = 0; i != TM; ++i) {
    const uint32_t m = m0 + i * 16 + row;
    const bool valid = m < a.M;
    const uint32_t mm = valid ? m : m0;
    const uint32_t q = a.divOutW(mm), ow = mm - q * a.outW;
    const uint32_t b = a.divOutH(q), oh = q - b * a.outH;
    originH[i] = int(oh * a.strideH) - a.padH;
    originW[i] = int(ow * a.strideW) - a.padW;
    rowOff[i] = (b - firstImage) * a.imageBytes + g * a.ciBytes;
    if constexpr (TAPS == kSmallOneTap)
      rowOff[i] = valid ? rowOff[i] + uint32_t(originH[i]) * a.rowBytes +
                              uint32_t(originW[i]) * a.pixelBytes
                        : kOutOfRange;
    else if (!valid)
      originH[i] = -0x40000000; // no tap of it is ever inside
  }

  auto loadPixels = [&](uint32_t s0, char *__restrict__ into) {
#pragma unroll
    for (int u = 0; u != U; ++u) {
      const uint32_t s = s0 + u;
      const uint32_t c = s * 4 + chunk;
      const uint32_t inK = uint32_t(s < sEnd) & uint32_t(c < a.chunks);
      if constexpr (TAPS == kSmallOneTap) {
#pragma unroll
        for (int i = 0; i != TM; ++i)
          loadToLds(inBuf, (LdsPtr)(into + (u * TM + i) * 1024),
                    inK ? rowOff[i] + c * 16 : kOutOfRange, 0);
      } else {
        const uint32_t tap = a.divChunks(c);
        const uint32_t within = (c - tap * (a.ciBytes >> 4)) * 16;
        const uint32_t kh = a.divKW(tap), kw = tap - kh * a.kW;
#pragma unroll
        for (int i = 0; i != TM; ++i) {
          int ih = originH[i] + int(kh * a.dilH);
          int iw = originW[i] + int(kw * a.dilW);
          uint32_t ok = inK;
          if constexpr (TAPS == kSmallDilated) {
            // (a negative position becomes one that is no input's)
            const int dh = int(a.divInDilH(uint32_t(ih) & 0x7fffffffu));
            const int dw = int(a.divInDilW(uint32_t(iw) & 0x7fffffffu));
            ok &= uint32_t(dh * a.inDilH == ih) &
                  uint32_t(dw * a.inDilW == iw);
            ih = dh, iw = dw;
          }
          ok &= uint32_t(uint32_t(ih) - a.loH < a.spanH) &
                uint32_t(uint32_t(iw) - a.loW < a.spanW);
          loadToLds(inBuf, (LdsPtr)(into + (u * TM + i) * 1024),
                    ok ? rowOff[i] + uint32_t(ih) * a.rowBytes +
                             uint32_t(iw) * a.pixelBytes + within
                       : kOutOfRange,
                    0);
        }
      }
    }
  };
  floatx4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i != TM; ++i)
#pragma unroll
    for (int j = 0; j != TN; ++j)
      acc[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
  // operand read: pixel lane % 16, chunk lane / 16
  const uint32_t readAt =
      (lane & 15) * 64 + (((lane >> 4) ^ ((lane & 15) >> 2)) * 16);
  auto multiply = [&](const Weights &wv, const char *__restrict__ from) {
#pragma unroll
    for (int u = 0; u != U; ++u)
#pragma unroll
      for (int i = 0; i != TM; ++i) {
        const uintx4 av = *reinterpret_cast<const uintx4 *>(
            from + (u * TM + i) * 1024 + readAt);
#pragma unroll
        for (int j = 0; j != TN; ++j)
          acc[i][j] = smallMma<EB>(wv.v[u][j], av, acc[i][j], a.formats);
      }
  };
  // (`__restrict__` on the part being loaded and the part being read: without
  // it every read would wait for the loads just issued)
  auto stage = [&](uint32_t next, Weights &nextW, const Weights &curW,
                   char *__restrict__ into, const char *__restrict__ from) {
    loadWeights(next, nextW);
    loadPixels(next, into);
    MXK_WAIT_VMCNT(U * (TM + TN));
    multiply(curW, from);
    MXK_WAIT_LGKMCNT0(); // `from` may be loaded into again
  };
  if (sBegin < sEnd) {
    char *own =
        lds + wave * ((a.stepsPerWave > U ? 2 : 1) * U * TM * 1024);
    char *other = own + U * TM * 1024;
    loadPixels(sBegin, own);
    uint32_t s = sBegin;
    for (;;) {
      if (s + U >= sEnd) {
        MXK_WAIT_VMCNT(0);
        multiply(even, own);
        break;
      }
      stage(s + U, odd, even, other, own);
      s += U;
      if (s + U >= sEnd) {
        MXK_WAIT_VMCNT(0);
        multiply(odd, other);
        break;
      }
      stage(s + U, even, odd, own, other);
      s += U;
    }
  }

  // The waves' sums meet in LDS: [wave][block][lane].  With the weights as
  // the row operand a lane holds channels 4 (lane / 16) ... + 3 of pixel
  // lane % 16.
  __syncthreads();
  floatx4 *sums = reinterpret_cast<floatx4 *>(lds);
#pragma unroll
  for (int i = 0; i != TM; ++i)
#pragma unroll
    for (int j = 0; j != TN; ++j)
      sums[(wave * TM * TN + i * TN + j) * 64 + lane] = acc[i][j];
  __syncthreads();
  OutT *out = static_cast<OutT *>(a.out);
  for (uint32_t blk = wave; blk < TM * TN; blk += a.waves) {
    // four reads in flight at a time (an even number of waves)
    floatx4 sum = {0.0f, 0.0f, 0.0f, 0.0f};
    for (uint32_t wv = 0; wv < a.waves; wv += 4) {
      floatx4 part[4];
#pragma unroll
      for (uint32_t k = 0; k != 4; ++k) {
        const uint32_t from = wv + k < a.waves ? wv + k : wv;
        part[k] = sums[(from * TM * TN + blk) * 64 + lane];
      }
      const bool more = wv + 2 < a.waves;
#pragma unroll
      for (int e = 0; e != 4; ++e)
        sum[e] += (part[0][e] + part[1][e]) +
                  (more ? part[2][e] + part[3][e] : 0.0f);
    }
    const uint32_t m = m0 + (blk / TN) * 16 + (lane & 15);
    const uint32_t n = outN;
    if (m >= a.M || n >= a.co)
      continue;
    float v[4];
#pragma unroll
    for (int e = 0; e != 4; ++e)
      v[e] = sum[e] * a.scale +
             (sizeof(OutT) == 2
                  ? __half2float(__ushort_as_half(uint16_t(biasRaw[e])))
                  : __uint_as_float(biasRaw[e]));
    if (a.outMode == 1) {
      for (int e = 0; e != 4 && n + e < a.co; ++e)
        storeOut(out, size_t(g * a.co + n + e) * a.M + m, v[e]);
      continue;
    }
    size_t pixel = m;
    if (a.outMode == 2) {
      const uint32_t q = a.divOutW(m), ow = m - q * a.outW;
      const uint32_t b = a.divOutH(q), oh = q - b * a.outH;
      pixel = (size_t(b) * a.outFullH + oh + a.outOffH) * a.outFullW + ow +
              a.outOffW;
    }
    if (a.co % 4 == 0 && a.outThrough) {
      storeOut4Through(bufferOf(out, a.outThrough),
                       uint32_t(pixel) * a.outChans + g * a.co + n, out, v);
    } else {
      OutT *at = out + pixel * a.outChans + g * a.co + n;
      for (int e = 0; e != 4 && n + e < a.co; ++e)
        storeOut(at, e, v[e]);
    }
  }
}

template <int EB, int TM, int TN, int U, int TAPS, class OutT>
__global__ __launch_bounds__(kSmallMostWaves * 64) void igemmSmallKernel(SmallArgs a) {
  igemmSmallTile<EB, TM, TN, U, TAPS, OutT>(a, blockIdx.x);
}

/// Several convolutions in one launch: the grid is the concatenation of their
/// tiles.
struct SmallFusedArgs {
  uint32_t count;
  uint32_t firstBlock[kIgemmMaxFused + 1];
  SmallArgs a[kIgemmMaxFused];
};
template <int EB, int TM, int TN, int U, int TAPS, class OutT>
__global__ __launch_bounds__(kSmallMostWaves * 64) void
igemmSmallFusedKernel(SmallFusedArgs m) {
  uint32_t i = 0;
  while (i + 1 < m.count && blockIdx.x >= m.firstBlock[i + 1])
    ++i;
  igemmSmallTile<EB, TM, TN, U, TAPS, OutT>(
      m.a[i], blockIdx.x - m.firstBlock[i]);
}

/// The tiles, by IgemmDesc::small: pixels and channels in blocks of 16, k-steps
/// per group of loads (two groups of 16 waves fit 128 KB of LDS).
struct SmallTile {
  uint32_t tm, tn, u;
};
constexpr SmallTile kSmallTiles[kIgemmSmallTiles + 1] = {
    {0, 0, 1}, {1, 1, 4}, {1, 2, 4}, {2, 2, 2}, {4, 2, 1}};

int tapsOf(const IgemmDesc &d) {
  if (d.inDilH != 1 || d.inDilW != 1)
    return kSmallDilated;
  return d.kH == 1 && d.kW == 1 && d.padH == 0 && d.padW == 0 && d.loH == 0 &&
                 d.loW == 0 && d.hiH == d.inH && d.hiW == d.inW &&
                 (d.outH == 0 || (d.outH - 1) * d.strideH < d.inH) &&
                 (d.outW == 0 || (d.outW - 1) * d.strideW < d.inW)
             ? kSmallOneTap
             : kSmallWindow;
}

uint32_t elemBytesOf(int type) {
  return type == kFloat ? 4 : type == kHalf ? 2 : 1;
}

uint32_t smallSteps(const IgemmDesc &d, uint32_t eb) {
  return (d.kH * d.kW * d.inChansPerGroup * eb + kSmallStepBytes - 1) /
         kSmallStepBytes;
}

/// One convolution, or several in one grid.
struct SmallLaunch {
  const SmallArgs *one;
  const SmallFusedArgs *fused;
  uint32_t blocks, waves, groups; // groups of loads a wave has room for
  int taps;
  int outType;
  hipStream_t stream;
};

template <int EB, int TM, int TN, int U, int TAPS, class OutT>
hipError_t launchKernel(const SmallLaunch &l) {
  auto raise = [](const void *kernel) {
    return hipFuncSetAttribute(
        kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 128 * 1024);
  };
  // the groups of loads, later the waves' sums
  const uint32_t ldsBytes =
      l.waves * 1024 *
      (l.groups * U * TM > TM * TN ? l.groups * U * TM : TM * TN);
  const dim3 grid{l.blocks}, block{l.waves * 64};
  if (l.one) {
    auto kernel = &igemmSmallKernel<EB, TM, TN, U, TAPS, OutT>;
    static const hipError_t attr =
        raise(reinterpret_cast<const void *>(kernel));
    if (attr != hipSuccess)
      return attr;
    hipLaunchKernelGGL(kernel, grid, block, ldsBytes, l.stream, *l.one);
  } else {
    auto kernel = &igemmSmallFusedKernel<EB, TM, TN, U, TAPS, OutT>;
    static const hipError_t attr =
        raise(reinterpret_cast<const void *>(kernel));
    if (attr != hipSuccess)
      return attr;
    hipLaunchKernelGGL(kernel, grid, block, ldsBytes, l.stream, *l.fused);
  }
  return hipGetLastError();
}

template <int EB, int TM, int TN, int U>
hipError_t launchTile(const SmallLaunch &l) {
  auto taps = [&](auto out) {
    using OutT = decltype(out);
    switch (l.taps) {
    case kSmallOneTap:
      return launchKernel<EB, TM, TN, U, kSmallOneTap, OutT>(l);
    case kSmallWindow:
      return launchKernel<EB, TM, TN, U, kSmallWindow, OutT>(l);
    }
    return launchKernel<EB, TM, TN, U, kSmallDilated, OutT>(l);
  };
  return l.outType == kHalf ? taps(__half{}) : taps(0.0f);
}

template <int EB> hipError_t launchType(uint32_t tile, const SmallLaunch &l) {
  switch (tile) {
  case 1:
    return launchTile<EB, 1, 1, kSmallTiles[1].u>(l);
  case 2:
    return launchTile<EB, 1, 2, kSmallTiles[2].u>(l);
  case 3:
    return launchTile<EB, 2, 2, kSmallTiles[3].u>(l);
  case 4:
    return launchTile<EB, 4, 2, kSmallTiles[4].u>(l);
  }
  return hipErrorInvalidValue;
}

hipError_t launchSmall(int inType, uint32_t tile, const SmallLaunch &l) {
  if (inType == kHalf)
    return launchType<2>(tile, l);
  return inType == kFloat ? launchType<4>(tile, l) : launchType<1>(tile, l);
}

} // namespace

uint32_t igemmSmallTilePixels(uint32_t tile) {
  return tile <= kIgemmSmallTiles ? kSmallTiles[tile].tm * 16 : 0;
}
uint32_t igemmSmallTileChans(uint32_t tile) {
  return tile <= kIgemmSmallTiles ? kSmallTiles[tile].tn * 16 : 0;
}

uint64_t igemmSmallTileCount(const IgemmDesc &d) {
  const SmallTile t = kSmallTiles[d.small];
  const uint64_t m = uint64_t(d.batch) * d.outH * d.outW;
  return (m + t.tm * 16 - 1) / (t.tm * 16) *
         ((d.outChansPerGroup + t.tn * 16 - 1) / (t.tn * 16)) * d.groups;
}

uint32_t igemmSmallWaves(const IgemmDesc &d, int inType) {
  // As many waves as K has groups of k-steps - a wave with one group waits for
  // memory once - and an even number of them; up to 16 where the workgroups
  // have a CU to themselves, 8 where they share one (4 x 28 x 28, 3 x 3, 128 ->
  // 128 in 392 tiles: 5.7 us with 8, 8.5 with 16).
  const SmallTile t = kSmallTiles[d.small];
  const uint32_t groups = (smallSteps(d, elemBytesOf(inType)) + t.u - 1) / t.u;
  const uint32_t waves = (groups + 1) / 2 * 2;
  const uint32_t most = igemmSmallTileCount(d) <= 256 ? kSmallMostWaves : 8;
  return waves > most ? most : waves < 2 ? 2 : waves;
}

uint64_t igemmSmallPackedElems(const IgemmDesc &d, int inType) {
  const uint32_t eb = elemBytesOf(inType);
  const uint64_t perTile = igemmSmallTileChans(d.small);
  const uint64_t co = (d.outChansPerGroup + perTile - 1) / perTile * perTile;
  return d.groups * co * smallSteps(d, eb) * (kSmallStepBytes / eb);
}

bool igemmSmallTakes(const IgemmDesc &d, int inType, int outType) {
  if (d.small == 0 || d.small > kIgemmSmallTiles ||
      (inType != kHalf && inType != kFloat && inType != kQuarter) ||
      (outType != kHalf && outType != kFloat))
    return false;
  const uint32_t eb = elemBytesOf(inType);
  const uint64_t M = uint64_t(d.batch) * d.outH * d.outW;
  auto fits16 = [](uint64_t v) { return v < 32768; };
  return d.inD == 1 && d.outD == 1 && d.kD == 1 && d.padD == 0 &&
         d.loD == 0 && d.hiD == 1 && d.outFullD <= 1 && d.outOffD == 0 &&
         d.noTaps == 0 &&
         d.outStepH == 1 && d.outStepW == 1 && d.inDilH != 0 &&
         d.inDilW != 0 && d.inChansPerGroup != 0 &&
         d.inChansPerGroup % (16 / eb) == 0 && M != 0 && M < (1u << 30) &&
         fits16(d.outH) && fits16(d.outW) && fits16(d.strideH) &&
         fits16(d.strideW) && fits16(d.dilH) && fits16(d.dilW) &&
         fits16(d.inDilH) && fits16(d.inDilW) && fits16(d.kW) &&
         fits16(uint64_t(d.padH < 0 ? -d.padH : d.padH)) &&
         fits16(uint64_t(d.padW < 0 ? -d.padW : d.padW)) &&
         uint64_t(d.kH) * d.kW * d.inChansPerGroup * eb < (1u << 30) &&
         igemmSmallPackedElems(d, inType) * eb < (1ull << 31) &&
         igemmAddressable(d, inType);
}

PackJob igemmSmallPackJob(const IgemmDesc &d, int inType) {
  const uint32_t eb = elemBytesOf(inType);
  PackJob j;
  j.steps = smallSteps(d, eb);
  j.blocks = uint32_t(igemmSmallPackedElems(d, inType) * eb / 1024 / j.steps /
                      d.groups);
  j.ciPadded = d.inChansPerGroup;
  j.taps = d.kH * d.kW;
  return j;
}

namespace {
hipError_t prepareSmall(const IgemmDesc &d, int inType, int outType,
                        const void *in, const void *weightsPacked,
                        const void *bias, void *out, const QuarterInfo &q,
                        SmallArgs &a, uint32_t &blocks) {
  if (!igemmSmallTakes(d, inType, outType))
    return hipErrorInvalidValue;
  const uint32_t eb = elemBytesOf(inType);
  const SmallTile tile = kSmallTiles[d.small];
  a = SmallArgs{};
  a.in = static_cast<const char *>(in);
  a.w = static_cast<const char *>(weightsPacked);
  a.bias = bias, a.out = out;
  a.M = d.batch * d.outH * d.outW;
  const uint32_t mTiles = (a.M + tile.tm * 16 - 1) / (tile.tm * 16);
  a.nTiles = (d.outChansPerGroup + tile.tn * 16 - 1) / (tile.tn * 16);
  a.steps = smallSteps(d, eb);
  a.chunks = d.kH * d.kW * d.inChansPerGroup * eb / 16;
  a.waves = igemmSmallWaves(d, inType);
  a.stepsPerWave = (a.steps + a.waves - 1) / a.waves;
  a.co = d.outChansPerGroup, a.outChans = d.groups * a.co;
  a.ciBytes = d.inChansPerGroup * eb;
  a.pixelBytes = d.groups * a.ciBytes;
  a.rowBytes = d.inW * a.pixelBytes;
  a.imageBytes = d.inH * a.rowBytes;
  a.inBytes = uint64_t(d.batch) * a.imageBytes;
  a.wBytes = uint32_t(igemmSmallPackedElems(d, inType) * eb);
  a.loH = d.loH, a.spanH = d.hiH - d.loH;
  a.loW = d.loW, a.spanW = d.hiW - d.loW;
  a.padH = int16_t(d.padH), a.padW = int16_t(d.padW);
  a.strideH = uint16_t(d.strideH), a.strideW = uint16_t(d.strideW);
  a.dilH = uint16_t(d.dilH), a.dilW = uint16_t(d.dilW);
  a.inDilH = uint16_t(d.inDilH), a.inDilW = uint16_t(d.inDilW);
  a.kW = uint16_t(d.kW);
  a.outW = uint16_t(d.outW), a.outH = uint16_t(d.outH);
  a.outMode = d.outTransposed ? 1 : d.outFullH || d.outFullW ? 2 : 0;
  a.outFullH = d.outFullH, a.outFullW = d.outFullW;
  a.outOffH = d.outOffH, a.outOffW = d.outOffW;
  a.outThrough = reachableBytes(
      uint64_t(d.batch) *
      (a.outMode == 2 ? uint64_t(d.outFullH) * d.outFullW
                      : uint64_t(d.outH) * d.outW) *
      a.outChans * (outType == kFloat ? 4 : 2));
  a.scale = inType == kQuarter ? q.scale : 1.0f;
  a.formats = inType != kQuarter
                  ? 0
                  : (q.inFormat != kE4M3 ? 1u : 0u) |
                        (q.weightFormat != kE4M3 ? 2u : 0u);
  a.divNTiles = makeFastDiv(a.nTiles), a.divMTiles = makeFastDiv(mTiles);
  a.divOutW = makeFastDiv(d.outW), a.divOutH = makeFastDiv(d.outH);
  a.divChunks = makeFastDiv(a.ciBytes / 16), a.divKW = makeFastDiv(d.kW);
  a.divInDilH = makeFastDiv(d.inDilH), a.divInDilW = makeFastDiv(d.inDilW);
  const uint64_t all = uint64_t(mTiles) * a.nTiles * d.groups;
  if (all > 0x7fffffffull)
    return hipErrorInvalidConfiguration;
  blocks = uint32_t(all);
  return hipSuccess;
}
} // namespace

hipError_t launchIgemmSmall(const IgemmDesc &d, int inType, int outType,
                            const void *in, const void *weightsPacked,
                            const void *bias, void *out, const QuarterInfo &q,
                            hipStream_t stream) {
  SmallArgs a;
  uint32_t blocks = 0;
  const hipError_t e = prepareSmall(d, inType, outType, in, weightsPacked,
                                    bias, out, q, a, blocks);
  if (e != hipSuccess)
    return e;
  return launchSmall(inType, d.small,
                     {&a, nullptr, blocks, a.waves,
                      a.stepsPerWave > kSmallTiles[d.small].u ? 2u : 1u,
                      tapsOf(d), outType, stream});
}

bool igemmSmallFusable(const IgemmFusedItem &x, const IgemmFusedItem &y) {
  return x.d->small != 0 && x.d->small == y.d->small &&
         x.inType == y.inType && x.outType == y.outType &&
         igemmSmallWaves(*x.d, x.inType) == igemmSmallWaves(*y.d, y.inType) &&
         tapsOf(*x.d) == tapsOf(*y.d);
}

hipError_t launchIgemmSmallFused(const IgemmFusedItem *items, size_t count,
                                 hipStream_t stream) {
  if (count == 0)
    return hipSuccess;
  if (count > kIgemmMaxFused)
    return hipErrorInvalidValue;
  SmallFusedArgs m{};
  m.count = uint32_t(count);
  uint64_t blocks = 0;
  uint32_t groups = 1;
  for (size_t i = 0; i != count; ++i) {
    const IgemmFusedItem &x = items[i];
    if (!igemmSmallFusable(items[0], x))
      return hipErrorInvalidValue;
    uint32_t own = 0;
    const hipError_t e =
        prepareSmall(*x.d, x.inType, x.outType, x.in, x.weightsPacked, x.bias,
                     x.out, x.q, m.a[i], own);
    if (e != hipSuccess)
      return e;
    if (m.a[i].stepsPerWave > kSmallTiles[x.d->small].u)
      groups = 2;
    m.firstBlock[i] = uint32_t(blocks);
    blocks += own;
    if (blocks > 0x7fffffffull)
      return hipErrorInvalidConfiguration;
  }
  m.firstBlock[count] = uint32_t(blocks);
  return launchSmall(items[0].inType, items[0].d->small,
                     {nullptr, &m, uint32_t(blocks), m.a[0].waves, groups,
                      tapsOf(*items[0].d), items[0].outType, stream});
}

} // namespace mxk
