// Layout conversions between the external tensor layouts of the convolution
// API ([B][G*C][field...] activations, [G][Co][Ci][kernel...] weights) and the
// device layouts the kernels use, plus the stand-alone bias add.
#include "device_types.hpp"
#include "kernels.hpp"

namespace mxk {
namespace {

/// Where element i of a permuted tensor comes from: the strides in the source
/// of the destination's dimensions (backwards through it where negative, as
/// wrapped numbers) from `srcBase` on.
struct PermuteArgs {
  uint64_t dstDims[4];
  uint64_t srcStride[4];
  uint64_t total, srcBase;
};
/// ... of fewer than 2^31 elements: 31-bit indices taken apart with
/// multiply-high divisions instead of eight 64-bit ones per element, and
/// arguments that a launch copies in a microsecond less.
struct PermuteSmallArgs {
  uint32_t total, srcBase;
  uint32_t dstDims[3]; // the inner three
  uint32_t srcStride[4];
  FastDiv div[3];
};

/// Any permutation, one element per thread.
template <class T>
__global__ __launch_bounds__(256) void permuteKernel(PermuteArgs a,
                                                     const T *__restrict__ src,
                                                     T *__restrict__ dst) {
  const uint64_t tid = uint64_t(blockIdx.x) * 256 + threadIdx.x;
  if (tid >= a.total)
    return;
  uint64_t srcIndex = a.srcBase, rest = tid;
  for (int j = 3; j >= 0; --j) {
    srcIndex += (rest % a.dstDims[j]) * a.srcStride[j];
    rest /= a.dstDims[j];
  }
  dst[tid] = src[srcIndex];
}
template <class T>
__global__ __launch_bounds__(256) void
permuteSmallKernel(PermuteSmallArgs a, const T *__restrict__ src,
                   T *__restrict__ dst) {
  const uint32_t tid = blockIdx.x * 256 + threadIdx.x;
  if (tid >= a.total)
    return;
  uint32_t srcIndex = a.srcBase, rest = tid;
#pragma unroll
  for (int j = 2; j >= 0; --j) {
    const uint32_t q = a.div[j](rest);
    srcIndex += (rest - q * a.dstDims[j]) * a.srcStride[j + 1];
    rest = q;
  }
  dst[tid] = src[srcIndex + rest * a.srcStride[0]];
}

/// [batch][rows][cols] -> [batch][cols][rows] in tiles of 64 x 64 turned round
/// in LDS: 16-byte loads along the columns, 16-byte stores along the rows.
/// Bound by HBM.  The LDS pitch of an odd number of words keeps both the
/// element writes down a column and the word reads along it off each other's
/// banks.
constexpr uint32_t kTurnTile = 64;
template <class T>
__global__ __launch_bounds__(256) void transposeKernel(
    const T *__restrict__ src, T *__restrict__ dst, uint64_t batch,
    uint32_t rows, uint32_t cols, uint32_t colTiles) {
  constexpr uint32_t kVec = 16 / sizeof(T);
  constexpr uint32_t kLanes = kTurnTile / kVec;  // threads per tile row
  constexpr uint32_t kRows = 256 / kLanes;       // tile rows per pass
  constexpr uint32_t kPitch = kTurnTile + 4 / sizeof(T);
  constexpr uint32_t kPasses = (kTurnTile + kRows - 1) / kRows;
  __shared__ __align__(16) T tile[kTurnTile * kPitch];
  const uint32_t rowTile = blockIdx.x / colTiles;
  const uint32_t r0 = rowTile * kTurnTile;
  const uint32_t c0 = (blockIdx.x - rowTile * colTiles) * kTurnTile;
  const uint32_t lane = (threadIdx.x % kLanes) * kVec;
  const uint32_t line = threadIdx.x / kLanes;
  for (uint64_t b = blockIdx.y; b < batch; b += gridDim.y) {
    const T *from = src + b * rows * cols;
    T *to = dst + b * rows * cols;
    Piece<T> v[kPasses];
#pragma unroll
    for (uint32_t i = 0; i != kPasses; ++i) {
      const uint32_t r = r0 + i * kRows + line, c = c0 + lane;
      const T *at = from + uint64_t(r) * cols + c;
      if (r < rows && c + kVec <= cols) {
        v[i] = loadPiece(at);
      } else {
#pragma unroll
        for (uint32_t e = 0; e != kVec; ++e)
          v[i].e[e] = r < rows && c + e < cols ? at[e] : T(0);
      }
    }
#pragma unroll
    for (uint32_t i = 0; i != kPasses; ++i)
#pragma unroll
      for (uint32_t e = 0; e != kVec; ++e)
        tile[(lane + e) * kPitch + i * kRows + line] = v[i].e[e];
    __syncthreads();
#pragma unroll
    for (uint32_t i = 0; i != kPasses; ++i) {
      const uint32_t c = c0 + i * kRows + line, r = r0 + lane;
      const uint32_t *words = reinterpret_cast<const uint32_t *>(
          tile + (i * kRows + line) * kPitch + lane);
      Piece<T> out;
#pragma unroll
      for (int w = 0; w != 4; ++w)
        out.w[w] = words[w];
      T *at = to + uint64_t(c) * rows + r;
      if (c < cols && r + kVec <= rows) {
        storePiece(at, out);
      } else if (c < cols) {
#pragma unroll
        for (uint32_t e = 0; e != kVec; ++e)
          if (r + e < rows)
            at[e] = out.e[e];
      }
    }
    __syncthreads();
  }
}

/// The same where one side is only N elements - an image's channels: TO_LAST
/// [batch][N][pixels] -> [batch][pixels][N], else the other way round.  A
/// workgroup takes a vector of pixels per thread; a thread turns N vectors round in
/// registers, and LDS makes both sides' accesses consecutive 16-byte pieces.
/// Bound by HBM (N = 32 images of 3 x 224 x 224 halves: 18.5 -> 5.6 us).
template <class T, int N, bool TO_LAST, uint32_t THREADS>
__global__ __launch_bounds__(THREADS) void interleaveKernel(
    const T *__restrict__ src, T *__restrict__ dst, uint64_t pixels,
    uint32_t blocksPerImage) {
  constexpr uint32_t kVec = 16 / sizeof(T), kPixels = THREADS * kVec;
  __shared__ uint4 packed[THREADS * N];
  const uint32_t image = blockIdx.x / blocksPerImage;
  const uint64_t p0 =
      uint64_t(blockIdx.x - image * blocksPerImage) * kPixels;
  const uint64_t base = uint64_t(image) * N * pixels;
  // this image's planes, and its interleaved elements from p0 on
  const T *planes = (TO_LAST ? src : dst) + base;
  const uint64_t p = p0 + threadIdx.x * kVec;
  union Block {
    Piece<T> plane[N];
    uint4 raw[N];
    T e[N * kVec];
  } in, out;
  const bool whole = p + kVec <= pixels;
  const uint64_t left = (pixels - p0) * N; // interleaved elements from p0
  if constexpr (TO_LAST) {
#pragma unroll
    for (int n = 0; n != N; ++n) {
      const T *at = planes + n * pixels + p;
      if (whole) {
        in.plane[n] = loadPiece(at);
      } else {
#pragma unroll
        for (uint32_t e = 0; e != kVec; ++e)
          in.plane[n].e[e] = p + e < pixels ? at[e] : T(0);
      }
    }
#pragma unroll
    for (uint32_t i = 0; i != N * kVec; ++i)
      out.e[i] = in.e[(i % N) * kVec + i / N];
#pragma unroll
    for (int n = 0; n != N; ++n)
      packed[threadIdx.x * N + n] = out.raw[n];
    __syncthreads();
    T *to = dst + base + p0 * N;
#pragma unroll
    for (int n = 0; n != N; ++n) {
      const uint32_t i = (n * THREADS + threadIdx.x) * kVec;
      union {
        uint4 raw;
        Piece<T> p;
      } v;
      v.raw = packed[n * THREADS + threadIdx.x];
      if (i + kVec <= left) {
        storePiece(to + i, v.p);
      } else {
#pragma unroll
        for (uint32_t e = 0; e != kVec; ++e)
          if (i + e < left)
            to[i + e] = v.p.e[e];
      }
    }
  } else {
    const T *from = src + base + p0 * N;
#pragma unroll
    for (int n = 0; n != N; ++n) {
      const uint32_t i = (n * THREADS + threadIdx.x) * kVec;
      union {
        uint4 raw;
        Piece<T> p;
      } v;
      if (i + kVec <= left) {
        v.p = loadPiece(from + i);
      } else {
#pragma unroll
        for (uint32_t e = 0; e != kVec; ++e)
          v.p.e[e] = i + e < left ? from[i + e] : T(0);
      }
      packed[n * THREADS + threadIdx.x] = v.raw;
    }
    __syncthreads();
#pragma unroll
    for (int n = 0; n != N; ++n)
      in.raw[n] = packed[threadIdx.x * N + n];
#pragma unroll
    for (uint32_t i = 0; i != N * kVec; ++i)
      out.e[(i % N) * kVec + i / N] = in.e[i];
    T *to = dst + base + p;
#pragma unroll
    for (int n = 0; n != N; ++n) {
      if (whole) {
        storePiece(to + n * pixels, out.plane[n]);
      } else {
#pragma unroll
        for (uint32_t e = 0; e != kVec; ++e)
          if (p + e < pixels)
            to[n * pixels + e] = out.plane[n].e[e];
      }
    }
  }
}

/// One 16-byte vector of the padded tensor per thread, read as one where the
/// source's channels fill it.  Bound by HBM: N = 13, 15 x 15, 327 channels
/// 4.4 us element by element, 3.6 so.
template <class T>
__global__ __launch_bounds__(256) void padChansKernel(
    const T *__restrict__ src, T *__restrict__ dst, uint64_t vectors,
    uint32_t ci, uint32_t ciPadded) {
  constexpr uint32_t kVec = 16 / sizeof(T);
  const uint64_t tid = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (tid >= vectors)
    return;
  const uint32_t perGroup = ciPadded / kVec;
  const uint64_t pg = tid / perGroup; // pixel * groups + group
  const uint32_t c0 = uint32_t(tid - pg * perGroup) * kVec;
  union {
    T e[kVec];
    uint4 u;
  } v;
  const T *at = src + pg * ci + c0;
  if (c0 + kVec <= ci) {
    const Piece<T> p = loadPiece(at);
    v.u = uint4{p.w[0], p.w[1], p.w[2], p.w[3]};
  } else {
#pragma unroll
    for (uint32_t i = 0; i != kVec; ++i)
      v.e[i] = c0 + i < ci ? at[i] : T(0);
  }
  reinterpret_cast<uint4 *>(dst)[tid] = v.u;
}

template <class T>
__global__ __launch_bounds__(256) void addBiasKernel(T *acts,
                                                     const T *__restrict__ bias,
                                                     uint64_t total,
                                                     uint64_t channels) {
  const uint64_t tid = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (tid >= total)
    return;
  const float v = Load<T>::at(acts, tid, 0) + Load<T>::at(bias, tid % channels, 0);
  storeOut(acts, tid, v);
}

template <typename T>
__global__ __launch_bounds__(256) void scaledAddKernel(T *a,
                                                       float scaleA,
                                                       const T *__restrict__ b,
                                                       float scaleB,
                                                       uint64_t total) {
  const uint64_t tid = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (tid >= total)
    return;
  storeOut(a, tid,
           scaleA * Load<T>::at(a, tid, 0) + scaleB * Load<T>::at(b, tid, 0));
}

constexpr uint32_t kSwapChans = 64, kSwapRows = 128;

struct SwapArgs {
  uint32_t batch, pixels, groups, chans; // source [batch][pixels][groups][chans]
  uint32_t pixelsPerTile, batchPerTile;  // their product is kSwapRows
  uint64_t strideG, strideC, strideP;    // destination strides; batch has 1
  uint32_t vectorStores; // 1: 16-byte stores of consecutive batch entries
};

/// dst[g * strideG + c * strideC + p * strideP + b] = src[b][p][g][c]: the
/// batch axis becomes the innermost one.  A workgroup moves a tile of 128
/// (pixel, batch) rows by 64 channels through LDS: loads run along the
/// channels, stores along the batch (and on along the pixels where the
/// destination keeps them adjacent).
template <class T, bool VEC>
__device__ __forceinline__ void
swapBatchChansTile(const SwapArgs &a, const T *__restrict__ src,
                   T *__restrict__ dst, uint32_t blockX, uint32_t blockY,
                   uint32_t blockZ) {
  __shared__ uint32_t tile[kSwapRows][kSwapChans + 1];
  const uint32_t cBlocks = (a.chans + kSwapChans - 1) / kSwapChans;
  const uint32_t c0 = (blockX % cBlocks) * kSwapChans;
  const uint32_t g = blockX / cBlocks;
  const uint32_t p0 = blockY * a.pixelsPerTile;
  const uint32_t b0 = blockZ * a.batchPerTile;
  const uint32_t lane = threadIdx.x % 64, wave = threadIdx.x / 64;
  // row = pLocal * batchPerTile + bLocal
  auto source = [&](uint32_t row, uint32_t c) {
    const uint32_t p = p0 + row / a.batchPerTile;
    const uint32_t b = b0 + row % a.batchPerTile;
    return p < a.pixels && b < a.batch && c < a.chans
               ? src + ((uint64_t(b) * a.pixels + p) * a.groups + g) * a.chans +
                     c
               : nullptr;
  };
  if constexpr (VEC) {
    // 16-byte loads: kVec channels per thread, all loads of a thread issued
    // before the first is used.  The channel count is a multiple of kVec.
    constexpr uint32_t kVec = 16 / sizeof(T);
    constexpr uint32_t kLanesPerRow = kSwapChans / kVec;
    constexpr uint32_t kRowsPerPass = 256 / kLanesPerRow;
    constexpr uint32_t kPasses = kSwapRows / kRowsPerPass;
    const uint32_t cLocal = (threadIdx.x % kLanesPerRow) * kVec;
    const uint32_t rowInPass = threadIdx.x / kLanesPerRow;
    uint4 v[kPasses];
#pragma unroll
    for (uint32_t i = 0; i != kPasses; ++i) {
      const T *from = source(i * kRowsPerPass + rowInPass, c0 + cLocal);
      v[i] = from ? *reinterpret_cast<const uint4 *>(from) : uint4{0, 0, 0, 0};
    }
#pragma unroll
    for (uint32_t i = 0; i != kPasses; ++i) {
      const T *e = reinterpret_cast<const T *>(&v[i]);
#pragma unroll
      for (uint32_t k = 0; k != kVec; ++k)
        tile[i * kRowsPerPass + rowInPass][cLocal + k] = e[k];
    }
  } else {
    constexpr uint32_t kPasses = kSwapRows / 4;
    T v[kPasses];
#pragma unroll
    for (uint32_t i = 0; i != kPasses; ++i) {
      const T *from = source(i * 4 + wave, c0 + lane);
      v[i] = from ? *from : T(0);
    }
#pragma unroll
    for (uint32_t i = 0; i != kPasses; ++i)
      tile[i * 4 + wave][lane] = v[i];
  }
  __syncthreads();
  if (a.vectorStores) {
    // A thread gathers 16 bytes of consecutive batch entries of one channel
    // (consecutive rows of the tile); consecutive lanes take consecutive
    // such pieces, then the next channel.  The batch size and every stride
    // are multiples of the vector length.
    constexpr uint32_t kVec = 16 / sizeof(T);
    constexpr uint32_t kPieces = kSwapRows / kVec;
#pragma unroll 2
    for (uint32_t i = threadIdx.x; i < kSwapChans * kPieces; i += 256) {
      const uint32_t cLocal = i / kPieces, row = (i % kPieces) * kVec;
      const uint32_t p = p0 + row / a.batchPerTile;
      const uint32_t b = b0 + row % a.batchPerTile;
      const uint32_t c = c0 + cLocal;
      if (p < a.pixels && b < a.batch && c < a.chans) {
        union {
          uint4 raw;
          T e[kVec];
        } v;
#pragma unroll
        for (uint32_t k = 0; k != kVec; ++k)
          v.e[k] = T(tile[row + k][cLocal]);
        *reinterpret_cast<uint4 *>(dst + g * a.strideG + c * a.strideC +
                                   p * a.strideP + b) = v.raw;
      }
    }
    return;
  }
  // 64 lanes = 64 consecutive rows of the tile: consecutive batch entries,
  // then the next pixel.
#pragma unroll 4
  for (uint32_t i = wave; i < kSwapChans * 2; i += 4) {
    const uint32_t cLocal = i / 2, row = (i % 2) * 64 + lane;
    const uint32_t p = p0 + row / a.batchPerTile;
    const uint32_t b = b0 + row % a.batchPerTile;
    const uint32_t c = c0 + cLocal;
    if (p < a.pixels && b < a.batch && c < a.chans)
      dst[g * a.strideG + c * a.strideC + p * a.strideP + b] =
          T(tile[row][cLocal]);
  }
}

template <class T, bool VEC>
__global__ __launch_bounds__(256) void swapBatchChansKernel(
    SwapArgs a, const T *__restrict__ src, T *__restrict__ dst) {
  swapBatchChansTile<T, VEC>(a, src, dst, blockIdx.x, blockIdx.y, blockIdx.z);
}

/// Two such rearrangements in one launch (the two operands of a weight update
/// pass): the grid's z extent is the sum of theirs, x and y cover the larger;
/// workgroups outside their tensor's own grid have nothing to do.
struct SwapPairArgs {
  SwapArgs a[2];
  uint32_t gridX[2], gridY[2], gridZ0; // z blocks of the first
};
template <class T>
__global__ __launch_bounds__(256) void swapBatchChansPairKernel(
    SwapPairArgs m, const T *__restrict__ src0, T *__restrict__ dst0,
    const T *__restrict__ src1, T *__restrict__ dst1) {
  const uint32_t which = blockIdx.z < m.gridZ0 ? 0 : 1;
  if (blockIdx.x >= m.gridX[which] || blockIdx.y >= m.gridY[which])
    return;
  if (which == 0)
    swapBatchChansTile<T, true>(m.a[0], src0, dst0, blockIdx.x, blockIdx.y,
                                blockIdx.z);
  else
    swapBatchChansTile<T, true>(m.a[1], src1, dst1, blockIdx.x, blockIdx.y,
                                blockIdx.z - m.gridZ0);
}

template <class T>
__global__ __launch_bounds__(256) void zeroKernel(T *dst, uint64_t total) {
  const uint64_t tid = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (tid < total)
    dst[tid] = T(0);
}

/// partial[split][c] = sum over the rows of `split` of z[row][c], fp32.
/// A workgroup takes up to 64 vectors of VEC neighbouring channels (16 bytes;
/// VEC = 1 where the channels are no whole vectors) and as many rows side by
/// side as its 256 threads hold; a thread keeps eight rows' loads in flight
/// and the row lanes meet in LDS.  Bound by HBM: with one element per load and
/// one load in flight per thread it took 9.2 us for 6.4 MB (25 088 rows of 128
/// halves) and 41 us for 28.9 MB, now 3.8 and 7.9.
constexpr uint32_t kReduceVecs = 64, kReduceUnroll = 8;
template <typename T, int VEC>
__global__ __launch_bounds__(256) void channelSumKernel(
    const T *__restrict__ z, float *__restrict__ partial, uint64_t rows,
    uint64_t channels, uint64_t rowsPerSplit, uint32_t vecsPerBlock) {
  __shared__ float lanes[256 * VEC];
  const uint32_t rowLanes = 256 / vecsPerBlock;
  const uint32_t rowLane = threadIdx.x / vecsPerBlock;
  const uint32_t vec = threadIdx.x - rowLane * vecsPerBlock;
  const uint64_t c = (uint64_t(blockIdx.x) * vecsPerBlock + vec) * VEC;
  const uint64_t first = min(blockIdx.y * rowsPerSplit, rows);
  const uint32_t last = uint32_t(min(rowsPerSplit, rows - first));
  struct alignas(sizeof(T) * VEC) Vec {
    T e[VEC];
  };
  float sum[VEC] = {};
  if (rowLane < rowLanes && c < channels) {
    uint32_t r = rowLane; // within the split
    const T *at = z + (first + r) * channels + c;
    const uint64_t step = uint64_t(rowLanes) * channels;
    // (whole groups first; then what is left of the rows, at once, those beyond
    // the last the last again and not added)
    for (; r + (kReduceUnroll - 1) * rowLanes < last;
         r += kReduceUnroll * rowLanes) {
      Vec v[kReduceUnroll];
#pragma unroll
      for (uint32_t u = 0; u != kReduceUnroll; ++u, at += step)
        v[u] = *reinterpret_cast<const Vec *>(at);
#pragma unroll
      for (uint32_t u = 0; u != kReduceUnroll; ++u)
#pragma unroll
        for (int e = 0; e != VEC; ++e)
          sum[e] += Load<T>::at(v[u].e, e, 0);
    }
    if (r < last) {
      Vec v[kReduceUnroll];
#pragma unroll
      for (uint32_t u = 0; u != kReduceUnroll; ++u) {
        v[u] = *reinterpret_cast<const Vec *>(at);
        at += r + (u + 1) * rowLanes < last ? step : 0;
      }
#pragma unroll
      for (uint32_t u = 0; u != kReduceUnroll; ++u)
        if (r + u * rowLanes < last)
#pragma unroll
          for (int e = 0; e != VEC; ++e)
            sum[e] += Load<T>::at(v[u].e, e, 0);
    }
  }
#pragma unroll
  for (int e = 0; e != VEC; ++e)
    lanes[threadIdx.x * VEC + e] = sum[e];
  __syncthreads();
  // lanes is [row lane][vector][element] as it stands
  const uint32_t own = vecsPerBlock * VEC;
  for (uint32_t i = threadIdx.x; i < own; i += 256) {
    const uint64_t ch = uint64_t(blockIdx.x) * own + i;
    if (ch >= channels)
      break;
    float total = lanes[i];
#pragma unroll 8
    for (uint32_t l = 1; l != rowLanes; ++l)
      total += lanes[l * own + i];
    partial[uint64_t(blockIdx.y) * channels + ch] = total;
  }
}

/// biases[c] += scale * sum over splits of partial[split][c].  16 channels per
/// workgroup, 16 lanes to a channel, each with all of its splits' loads in
/// flight; the lanes' sums are added in order.  (One thread per channel walking
/// the splits one after the other took 46 us for 196 splits of 128 channels -
/// a chain of 196 memory latencies; now 2.2.)
constexpr uint32_t kBiasChans = 16, kBiasLanes = 16, kBiasSplits = 256;
/// WIDE: the sums' offsets are beyond 31 bits.
template <typename T, bool WIDE>
__global__ __launch_bounds__(256) void biasUpdateKernel(
    T *biases, const float *__restrict__ partial, float scale,
    uint64_t channels, uint32_t splits) {
  __shared__ float lanes[kBiasLanes][kBiasChans];
  const uint32_t cLocal = threadIdx.x % kBiasChans;
  const uint32_t lane = threadIdx.x / kBiasChans;
  const uint64_t c = uint64_t(blockIdx.x) * kBiasChans + cLocal;
  const uint64_t cIn = c < channels ? c : channels - 1;
  const float before = Load<T>::at(biases, cIn, 0);
  // (splits beyond the last: zeros from beyond the buffer's end, or the last
  // again and not added.  Under a condition each, the first was waited for on its
  // own: 77 updates 1.04 times as fast so, up to 1.14; 65 1.024 times with 32-bit
  // offsets, one instruction to a load in place of eight.)
  float v[kBiasSplits / kBiasLanes];
  if constexpr (WIDE) {
#pragma unroll
    for (uint32_t i = 0; i != kBiasSplits / kBiasLanes; ++i) {
      const uint32_t s = i * kBiasLanes + lane;
      v[i] = partial[uint64_t(s < splits ? s : splits - 1) * channels + cIn];
    }
#pragma unroll
    for (uint32_t i = 0; i != kBiasSplits / kBiasLanes; ++i)
      v[i] = i * kBiasLanes + lane < splits ? v[i] : 0.f;
  } else {
    const __amdgpu_buffer_rsrc_t buffer = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(partial), short(0),
        int(splits * uint32_t(channels) * 4), 0x00020000);
    const uint32_t step = kBiasLanes * uint32_t(channels) * 4;
    const uint32_t at = (lane * uint32_t(channels) + uint32_t(cIn)) * 4;
#pragma unroll
    for (uint32_t i = 0; i != kBiasSplits / kBiasLanes; ++i)
      v[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                           buffer, at + i * step, 0, 0));
  }
  float sum = 0.f;
#pragma unroll
  for (uint32_t i = 0; i != kBiasSplits / kBiasLanes; ++i)
    sum += v[i];
  lanes[lane][cLocal] = sum;
  __syncthreads();
  if (lane != 0 || c >= channels)
    return;
  float total = lanes[0][cLocal];
#pragma unroll
  for (uint32_t l = 1; l != kBiasLanes; ++l)
    total += lanes[l][cLocal];
  storeOut(biases, c, before + scale * total);
}

/// The same in one launch, for few rows: a workgroup takes 32 channels (64
/// bytes of halves, four lanes to a row; one channel per lane where they are
/// no whole vectors) through all the rows, eight rows' loads in flight per
/// thread; the row lanes' sums meet in LDS.  Of halves that is half a 128-byte
/// line, so the two workgroups of a line are `paired`: dealt to one XCD, whose
/// L2 fetches it once (8192 halves in 2 048 rows 13.3 -> 9.9 us).
/// A single CU reads 64 bytes a cycle at best, which the second launch
/// outweighs up to 2 048 rows - 3 200 of 1 MB in all, 4 096 of a single line,
/// but 1 024 of no whole vectors.  The call, host and all, us, on rows from
/// memory and on rows just read, with this kernel and with two:
///   halves   64 x 4 096   6.8, 4.7   6.4, 6.3     144 x 2 048  5.3, 3.9   6.4, 6.4
///           144 x 3 136   7.3, 4.5   6.4, 6.5   1 024 x 2 048  8.8, 3.9   6.7, 6.5
///         1 024 x 4 096  15.3, 5.0   7.0, 6.5   8 192 x 2 048 10.4, 4.9  10.8, 7.3
///   floats  144 x 2 048   5.5, 4.9   6.5, 6.8   2 048 x 2 048  9.4, 3.9   8.2, 6.4
/// In a layer's training step the rows are somewhere between: 16 images of
/// 14 x 14, 1 x 1, 512 -> 1024 (3 136 rows) 55.1 us with this kernel, 52.4 with
/// two, 64 of 8 x 8, 3 x 3, 256 -> 512 (4 096) 74.8 and 71.2, but 4 of 28 x 28,
/// 1 x 1, 64 -> 144 (3 136) 33.0 and 35.4.
constexpr uint32_t kDirectRows = 2048, kDirectRaggedRows = 1024;
constexpr uint32_t kDirectSmallRows = 3200, kDirectLineRows = 4096;
constexpr uint32_t kDirectChans = 32;
template <typename T, int VEC, typename B>
__global__ __launch_bounds__(1024) void biasDirectKernel(
    const T *__restrict__ z, B *biases, float scale, uint32_t rows,
    uint64_t channels, uint32_t paired) {
  constexpr uint32_t kVecLanes = kDirectChans / VEC;
  constexpr uint32_t kRowLanes = 1024 / kVecLanes, kParts = 32;
  constexpr uint32_t kPerPart = (kRowLanes + kParts - 1) / kParts;
  __shared__ float lanes[kRowLanes][kDirectChans];
  __shared__ float parts[kParts][kDirectChans];
  const uint32_t vec = threadIdx.x % kVecLanes;
  const uint32_t rowLane = threadIdx.x / kVecLanes;
  // (workgroups b and b + 8 of every 16 run on one XCD)
  const uint32_t b = blockIdx.x;
  const uint32_t block =
      b < paired ? (b & ~15u) | ((b & 7u) << 1) | ((b >> 3) & 1u) : b;
  const uint64_t c0 = uint64_t(block) * kDirectChans;
  const uint64_t c = c0 + vec * VEC;
  struct alignas(sizeof(T) * VEC) Vec {
    T e[VEC];
  };
  float sum[VEC] = {};
  if (c < channels) {
    const T *at = z + c;
    for (uint32_t r = rowLane; r < rows; r += kReduceUnroll * kRowLanes) {
      Vec v[kReduceUnroll];
#pragma unroll
      for (uint32_t u = 0; u != kReduceUnroll; ++u) {
        // (rows beyond the last: the last again, not added)
        const uint32_t row = r + u * kRowLanes;
        v[u] = *reinterpret_cast<const Vec *>(
            at + uint64_t(row < rows ? row : rows - 1) * channels);
      }
#pragma unroll
      for (uint32_t u = 0; u != kReduceUnroll; ++u)
        if (r + u * kRowLanes < rows)
#pragma unroll
          for (int e = 0; e != VEC; ++e)
            sum[e] += Load<T>::at(v[u].e, e, 0);
    }
  }
#pragma unroll
  for (int e = 0; e != VEC; ++e)
    lanes[rowLane][vec * VEC + e] = sum[e];
  __syncthreads();
  const uint32_t own = threadIdx.x % kDirectChans;
  const uint32_t part = threadIdx.x / kDirectChans;
  float some = 0.0f;
#pragma unroll
  for (uint32_t l = 0; l != kPerPart; ++l)
    some += lanes[part * kPerPart + l][own];
  parts[part][own] = some;
  __syncthreads();
  if (threadIdx.x < kDirectChans && c0 + own < channels) {
    float total = 0.0f;
#pragma unroll
    for (uint32_t p = 0; p != kParts; ++p)
      total += parts[p][own];
    storeOut(biases, c0 + own,
             Load<B>::at(biases, c0 + own, 0) + scale * total);
  }
}

/// Weight deltas of groups that ran f as one: the f diagonal blocks of every
/// fused group of [G / f][f co][f ci][taps] -> [G][co][ci][taps].  One element
/// of the result per thread.
template <class T>
__global__ __launch_bounds__(256) void
unfuseGroupWeightsKernel(const T *__restrict__ src, T *__restrict__ dst,
                         uint64_t f, uint64_t co, uint64_t ci, uint64_t taps,
                         uint64_t total) {
  const uint64_t i = uint64_t(blockIdx.x) * 256 + threadIdx.x;
  if (i >= total)
    return;
  const uint64_t tap = i % taps;
  uint64_t rest = i / taps;
  const uint64_t k = rest % ci;
  rest /= ci;
  const uint64_t n = rest % co;
  const uint64_t g = rest / co;
  const uint64_t fused = g / f, a = g % f;
  dst[i] = src[((fused * f * co + a * co + n) * (f * ci) + a * ci + k) * taps +
               tap];
}

} // namespace

namespace {
template <class T>
hipError_t permuteAny(const void *src, void *dst, const PermuteArgs &a,
                      hipStream_t stream) {
  const uint64_t blocks = (a.total + 255) / 256;
  if (blocks > 0x7fffffffull)
    return hipErrorInvalidConfiguration;
  const dim3 grid{uint32_t(blocks)}, block{256};
  if (a.total < 0x7fffffffull) {
    PermuteSmallArgs s;
    s.total = uint32_t(a.total), s.srcBase = uint32_t(a.srcBase);
    for (int j = 0; j != 4; ++j) {
      s.srcStride[j] = uint32_t(a.srcStride[j]);
      if (j != 0) {
        s.dstDims[j - 1] = uint32_t(a.dstDims[j]);
        s.div[j - 1] = makeFastDiv(uint32_t(a.dstDims[j]));
      }
    }
    hipLaunchKernelGGL(permuteSmallKernel<T>, grid, block, 0, stream, s,
                       static_cast<const T *>(src), static_cast<T *>(dst));
  } else {
    hipLaunchKernelGGL(permuteKernel<T>, grid, block, 0, stream, a,
                       static_cast<const T *>(src), static_cast<T *>(dst));
  }
  return hipGetLastError();
}

template <class T, int N, bool TO_LAST>
hipError_t interleave(const void *src, void *dst, uint64_t batch,
                      uint64_t pixels, hipStream_t stream) {
  constexpr uint32_t kVec = 16 / sizeof(T);
  auto launch = [&](auto threads) {
    constexpr uint32_t THREADS = decltype(threads)::value;
    const uint64_t perImage =
        (pixels + THREADS * kVec - 1) / (THREADS * kVec);
    const uint64_t blocks = batch * perImage;
    if (blocks > 0x7fffffffull)
      return hipErrorInvalidConfiguration;
    hipLaunchKernelGGL((interleaveKernel<T, N, TO_LAST, THREADS>),
                       dim3{uint32_t(blocks)}, dim3{THREADS}, 0, stream,
                       static_cast<const T *>(src), static_cast<T *>(dst),
                       pixels, uint32_t(perImage));
    return hipGetLastError();
  };
  // Few images: single-wave workgroups, or a handful of CUs do all the work.
  if (batch * pixels < 256ull * 256 * kVec)
    return launch(std::integral_constant<uint32_t, 64>{});
  return launch(std::integral_constant<uint32_t, 256>{});
}

/// [batch][rows][cols] -> [batch][cols][rows]; *taken = false and nothing
/// launched where another kernel is the better one.
template <class T>
hipError_t transposeBatches(const void *src, void *dst, uint64_t batch,
                            uint64_t rows, uint64_t cols, hipStream_t stream,
                            bool *taken) {
  *taken = true;
  // Two to four elements on one side (an image's channels): tiles of 64 would
  // be nearly empty.  Worth it from half a workgroup of pixels on, and from a
  // few vectors for every CU: below, an element per thread is the shorter
  // chain (halves of three channels, 191 x 191 pixels: 2.8 against 3.5 us;
  // three images of 239 x 239: 3.7 against 3.4).
  const uint64_t fewest = 128 * (16 / sizeof(T));
  const bool many = batch * rows * cols >= 256 * 1024;
  if (many && cols >= fewest) {
    if (rows == 2)
      return interleave<T, 2, true>(src, dst, batch, cols, stream);
    if (rows == 3)
      return interleave<T, 3, true>(src, dst, batch, cols, stream);
    if (rows == 4)
      return interleave<T, 4, true>(src, dst, batch, cols, stream);
  }
  if (many && rows >= fewest) {
    if (cols == 2)
      return interleave<T, 2, false>(src, dst, batch, rows, stream);
    if (cols == 3)
      return interleave<T, 3, false>(src, dst, batch, rows, stream);
    if (cols == 4)
      return interleave<T, 4, false>(src, dst, batch, rows, stream);
  }
  // Tiles want at least an eighth of their rows and columns in use.
  const uint64_t rowTiles = (rows + kTurnTile - 1) / kTurnTile;
  const uint64_t colTiles = (cols + kTurnTile - 1) / kTurnTile;
  if (rows < kTurnTile / 8 || cols < kTurnTile / 8 ||
      rows > 0x7fffffffull || cols > 0x7fffffffull ||
      rowTiles * colTiles > 0x7fffffffull) {
    *taken = false;
    return hipSuccess;
  }
  const dim3 grid{uint32_t(rowTiles * colTiles),
                  uint32_t(batch < 65535 ? batch : 65535)};
  hipLaunchKernelGGL(transposeKernel<T>, grid, dim3{256}, 0, stream,
                     static_cast<const T *>(src), static_cast<T *>(dst), batch,
                     uint32_t(rows), uint32_t(cols), uint32_t(colTiles));
  return hipGetLastError();
}
} // namespace

hipError_t launchPermute4(const void *src, void *dst, const uint64_t srcDims[4],
                          const int perm[4], int elemBytes,
                          hipStream_t stream) {
  if (elemBytes != 1 && elemBytes != 2 && elemBytes != 4)
    return hipErrorInvalidValue;
  if (srcDims[0] * srcDims[1] * srcDims[2] * srcDims[3] == 0)
    return hipSuccess;
  // The permutation in its simplest form: extents of 1 left out, source
  // dimensions that stay neighbours in order taken as one.
  uint64_t dims[4]; // source extents
  int order[4];     // destination dimension j walks source dimension order[j]
  int n = 0;
  {
    int runStart[4], runs = 0;
    uint64_t runSize[4];
    int last = -1;
    for (int j = 0; j != 4; ++j) {
      const int d = perm[j];
      if (srcDims[d] == 1)
        continue;
      // the next source dimension with an extent, after `last`
      int next = last + 1;
      while (last >= 0 && next < 4 && srcDims[next] == 1)
        ++next;
      if (last >= 0 && d == next) {
        runSize[runs - 1] *= srcDims[d];
      } else {
        runStart[runs] = d;
        runSize[runs++] = srcDims[d];
      }
      last = d;
    }
    n = runs;
    for (int j = 0; j != n; ++j) {
      order[j] = 0;
      for (int i = 0; i != n; ++i)
        order[j] += runStart[i] < runStart[j];
    }
    for (int j = 0; j != n; ++j)
      dims[order[j]] = runSize[j];
  }
  const bool swapsLastTwo =
      (n == 2 && order[0] == 1) || (n == 3 && order[0] == 0 && order[1] == 2);
  if (swapsLastTwo) {
    const uint64_t batch = n == 3 ? dims[0] : 1;
    const uint64_t rows = dims[n - 2], cols = dims[n - 1];
    bool taken = false;
    hipError_t e = hipSuccess;
    if (elemBytes == 1)
      e = transposeBatches<uint8_t>(src, dst, batch, rows, cols, stream,
                                    &taken);
    else if (elemBytes == 2)
      e = transposeBatches<uint16_t>(src, dst, batch, rows, cols, stream,
                                     &taken);
    else
      e = transposeBatches<uint32_t>(src, dst, batch, rows, cols, stream,
                                     &taken);
    if (taken || e != hipSuccess)
      return e;
  }
  // Innermost runs that stay together and are whole vectors move as such.
  if (n != 0 && order[n - 1] == n - 1 &&
      dims[n - 1] * elemBytes % 16 == 0 &&
      reinterpret_cast<uintptr_t>(src) % 16 == 0 &&
      reinterpret_cast<uintptr_t>(dst) % 16 == 0) {
    dims[n - 1] = dims[n - 1] * elemBytes / 16;
    elemBytes = 16;
  }
  uint64_t stride[4], s = 1;
  for (int i = n - 1; i >= 0; --i) {
    stride[i] = s;
    s *= dims[i];
  }
  PermuteArgs a;
  a.total = s, a.srcBase = 0;
  for (int j = 0; j != 4; ++j) {
    // destination dimensions, right-aligned
    const int d = j - (4 - n);
    a.dstDims[j] = d >= 0 ? dims[order[d]] : 1;
    a.srcStride[j] = d >= 0 ? stride[order[d]] : 0;
  }
  switch (elemBytes) {
  case 1:
    return permuteAny<uint8_t>(src, dst, a, stream);
  case 2:
    return permuteAny<uint16_t>(src, dst, a, stream);
  case 4:
    return permuteAny<uint32_t>(src, dst, a, stream);
  }
  return permuteAny<uint4>(src, dst, a, stream);
}


hipError_t launchPadChans(const void *src, void *dst, uint64_t pixels,
                          uint32_t groups, uint32_t ci, uint32_t ciPadded,
                          int elemBytes, hipStream_t stream) {
  if ((elemBytes != 1 && elemBytes != 2 && elemBytes != 4) || ciPadded < ci ||
      (uint64_t(ciPadded) * elemBytes) % 16 != 0)
    return hipErrorInvalidValue;
  const uint64_t vectors =
      pixels * groups * (uint64_t(ciPadded) * elemBytes / 16);
  if (vectors == 0)
    return hipSuccess;
  const uint64_t blocks = (vectors + 255) / 256;
  if (blocks > 0x7fffffffull)
    return hipErrorInvalidConfiguration;
  const dim3 grid{uint32_t(blocks)}, block{256};
  if (elemBytes == 1)
    hipLaunchKernelGGL(padChansKernel<uint8_t>, grid, block, 0, stream,
                       static_cast<const uint8_t *>(src),
                       static_cast<uint8_t *>(dst), vectors, ci, ciPadded);
  else if (elemBytes == 2)
    hipLaunchKernelGGL(padChansKernel<uint16_t>, grid, block, 0, stream,
                       static_cast<const uint16_t *>(src),
                       static_cast<uint16_t *>(dst), vectors, ci, ciPadded);
  else
    hipLaunchKernelGGL(padChansKernel<uint32_t>, grid, block, 0, stream,
                       static_cast<const uint32_t *>(src),
                       static_cast<uint32_t *>(dst), vectors, ci, ciPadded);
  return hipGetLastError();
}

hipError_t launchWeightsTransposeChansFlipXY(const void *src, void *dst,
                                             uint64_t groups, uint64_t co,
                                             uint64_t ci, uint32_t numDims,
                                             const uint32_t *kernelShape,
                                             int elemBytes,
                                             hipStream_t stream) {
  if (numDims > uint32_t(kMaxDims))
    return hipErrorInvalidValue;
  uint64_t taps = 1;
  for (uint32_t d = 0; d != numDims; ++d)
    taps *= kernelShape[d];
  PermuteArgs a;
  a.total = groups * co * ci * taps;
  if (a.total == 0)
    return hipSuccess;
  if (taps == 1) {
    const uint64_t dims[4] = {1, groups, co, ci};
    const int perm[4] = {0, 1, 3, 2};
    return launchPermute4(src, dst, dims, perm, elemBytes, stream);
  }
  // dst [g][ci][co][k] = src [g][co][ci][taps - 1 - k]: every axis of the
  // window reversed is its row-major index read from the end
  const uint64_t dims[4] = {groups, ci, co, taps};
  const uint64_t stride[4] = {co * ci * taps, taps, ci * taps, ~0ull};
  for (int j = 0; j != 4; ++j)
    a.dstDims[j] = dims[j], a.srcStride[j] = stride[j];
  a.srcBase = taps - 1;
  if (elemBytes == 1)
    return permuteAny<uint8_t>(src, dst, a, stream);
  if (elemBytes == 2)
    return permuteAny<uint16_t>(src, dst, a, stream);
  if (elemBytes == 4)
    return permuteAny<uint32_t>(src, dst, a, stream);
  return hipErrorInvalidValue;
}

hipError_t launchAddBias(int type, void *acts, const void *bias,
                         uint64_t outerElems, uint64_t channels,
                         hipStream_t stream) {
  const uint64_t total = outerElems * channels;
  if (total == 0)
    return hipSuccess;
  const uint64_t blocks = (total + 255) / 256;
  if (blocks > 0x7fffffffull)
    return hipErrorInvalidConfiguration;
  const dim3 grid{uint32_t(blocks)}, block{256};
  if (type == kFloat)
    hipLaunchKernelGGL(addBiasKernel<float>, grid, block, 0, stream,
                       static_cast<float *>(acts),
                       static_cast<const float *>(bias), total, channels);
  else if (type == kHalf)
    hipLaunchKernelGGL(addBiasKernel<__half>, grid, block, 0, stream,
                       static_cast<__half *>(acts),
                       static_cast<const __half *>(bias), total, channels);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

namespace {
struct SwapLaunch {
  SwapArgs a;
  dim3 grid;
  bool vectorLoads;
};

/// Tile shape, grid and vector widths of one rearrangement.
hipError_t prepareSwap(const void *src, const void *dst, uint32_t batch,
                       uint32_t pixels, uint32_t groups, uint32_t chans,
                       uint64_t strideG, uint64_t strideC, uint64_t strideP,
                       int elemBytes, SwapLaunch &l) {
  if (elemBytes != 2 && elemBytes != 4)
    return hipErrorInvalidValue;
  SwapArgs &a = l.a;
  a.batch = batch, a.pixels = pixels, a.groups = groups, a.chans = chans;
  // As much of the batch as a tile takes (a power of two, so that it divides
  // the 128 rows), the rest of the rows for neighbouring pixels.
  a.batchPerTile = 1;
  while (a.batchPerTile < kSwapRows && a.batchPerTile < batch)
    a.batchPerTile *= 2;
  a.pixelsPerTile = kSwapRows / a.batchPerTile;
  a.strideG = strideG, a.strideC = strideC, a.strideP = strideP;
  const uint64_t gx = uint64_t((chans + kSwapChans - 1) / kSwapChans) * groups;
  const uint64_t gy = (pixels + a.pixelsPerTile - 1) / a.pixelsPerTile;
  const uint64_t gz = (batch + a.batchPerTile - 1) / a.batchPerTile;
  if (gx > 0x7fffffffull || gy > 65535 || gz > 65535)
    return hipErrorInvalidConfiguration;
  l.grid = dim3{uint32_t(gx), uint32_t(gy), uint32_t(gz)};
  // 16-byte loads need every row of channels to start on a 16-byte boundary;
  // 16-byte stores, every run of batch entries.
  const uint32_t perVector = uint32_t(16 / elemBytes);
  l.vectorLoads = chans % perVector == 0 &&
                  reinterpret_cast<uintptr_t>(src) % 16 == 0;
  a.vectorStores = batch % perVector == 0 && a.batchPerTile >= perVector &&
                   strideG % perVector == 0 && strideC % perVector == 0 &&
                   strideP % perVector == 0 &&
                   reinterpret_cast<uintptr_t>(dst) % 16 == 0;
  return hipSuccess;
}
} // namespace

hipError_t launchSwapBatchChans(const void *src, void *dst, uint32_t batch,
                                uint32_t pixels, uint32_t groups,
                                uint32_t chans, uint64_t strideG,
                                uint64_t strideC, uint64_t strideP,
                                int elemBytes, hipStream_t stream) {
  if (uint64_t(batch) * pixels * groups * chans == 0)
    return hipSuccess;
  SwapLaunch l;
  const hipError_t e = prepareSwap(src, dst, batch, pixels, groups, chans,
                                   strideG, strideC, strideP, elemBytes, l);
  if (e != hipSuccess)
    return e;
  const SwapArgs &a = l.a;
  const dim3 grid = l.grid, block{256};
  const bool vec = l.vectorLoads;
  if (elemBytes == 2) {
    const auto *from = static_cast<const uint16_t *>(src);
    auto *to = static_cast<uint16_t *>(dst);
    if (vec)
      hipLaunchKernelGGL((swapBatchChansKernel<uint16_t, true>), grid, block, 0,
                         stream, a, from, to);
    else
      hipLaunchKernelGGL((swapBatchChansKernel<uint16_t, false>), grid, block,
                         0, stream, a, from, to);
  } else {
    const auto *from = static_cast<const uint32_t *>(src);
    auto *to = static_cast<uint32_t *>(dst);
    if (vec)
      hipLaunchKernelGGL((swapBatchChansKernel<uint32_t, true>), grid, block, 0,
                         stream, a, from, to);
    else
      hipLaunchKernelGGL((swapBatchChansKernel<uint32_t, false>), grid, block,
                         0, stream, a, from, to);
  }
  return hipGetLastError();
}

hipError_t launchSwapBatchChansPair(const SwapBatchChans &first,
                                    const SwapBatchChans &second,
                                    int elemBytes, hipStream_t stream) {
  auto alone = [&](const SwapBatchChans &x) {
    return launchSwapBatchChans(x.src, x.dst, x.batch, x.pixels, x.groups,
                                x.chans, x.strideG, x.strideC, x.strideP,
                                elemBytes, stream);
  };
  auto empty = [](const SwapBatchChans &x) {
    return uint64_t(x.batch) * x.pixels * x.groups * x.chans == 0;
  };
  SwapLaunch l[2];
  bool together = !empty(first) && !empty(second);
  if (together) {
    const SwapBatchChans *both[2] = {&first, &second};
    for (int i = 0; i != 2 && together; ++i) {
      const SwapBatchChans &x = *both[i];
      together = prepareSwap(x.src, x.dst, x.batch, x.pixels, x.groups,
                             x.chans, x.strideG, x.strideC, x.strideP,
                             elemBytes, l[i]) == hipSuccess &&
                 l[i].vectorLoads;
    }
    together = together && l[0].grid.z + l[1].grid.z <= 65535;
  }
  if (!together) {
    const hipError_t e = alone(first);
    return e != hipSuccess ? e : alone(second);
  }
  SwapPairArgs m;
  for (int i = 0; i != 2; ++i)
    m.a[i] = l[i].a, m.gridX[i] = l[i].grid.x, m.gridY[i] = l[i].grid.y;
  m.gridZ0 = l[0].grid.z;
  const dim3 grid{l[0].grid.x > l[1].grid.x ? l[0].grid.x : l[1].grid.x,
                  l[0].grid.y > l[1].grid.y ? l[0].grid.y : l[1].grid.y,
                  l[0].grid.z + l[1].grid.z};
  if (elemBytes == 2)
    hipLaunchKernelGGL(swapBatchChansPairKernel<uint16_t>, grid, dim3{256}, 0,
                       stream, m, static_cast<const uint16_t *>(first.src),
                       static_cast<uint16_t *>(first.dst),
                       static_cast<const uint16_t *>(second.src),
                       static_cast<uint16_t *>(second.dst));
  else
    hipLaunchKernelGGL(swapBatchChansPairKernel<uint32_t>, grid, dim3{256}, 0,
                       stream, m, static_cast<const uint32_t *>(first.src),
                       static_cast<uint32_t *>(first.dst),
                       static_cast<const uint32_t *>(second.src),
                       static_cast<uint32_t *>(second.dst));
  return hipGetLastError();
}

hipError_t launchZero(void *dst, uint64_t bytes, hipStream_t stream) {
  if (bytes == 0)
    return hipSuccess;
  if (bytes % 4 != 0)
    return hipErrorInvalidValue;
  const uint64_t total = bytes / 4, blocks = (total + 255) / 256;
  if (blocks > 0x7fffffffull)
    return hipErrorInvalidConfiguration;
  hipLaunchKernelGGL(zeroKernel<uint32_t>, dim3(uint32_t(blocks)), dim3(256), 0,
                     stream, static_cast<uint32_t *>(dst), total);
  return hipGetLastError();
}

namespace {
/// One element of the padded output field per thread; those inside the
/// convolution's own outputs are left alone.
template <class T>
__global__ __launch_bounds__(256) void fillOutputPaddingKernel(
    T *__restrict__ out, const T *__restrict__ bias, uint64_t total,
    uint32_t fullD, uint32_t fullH, uint32_t fullW, uint32_t offD,
    uint32_t offH, uint32_t offW, uint32_t insideD, uint32_t insideH,
    uint32_t insideW, uint32_t chans) {
  const uint64_t tid = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (tid >= total)
    return;
  const uint64_t pixel = tid / chans;
  const uint32_t c = uint32_t(tid - pixel * chans);
  const uint32_t w = uint32_t(pixel % fullW);
  const uint32_t h = uint32_t((pixel / fullW) % fullH);
  const uint32_t z = uint32_t((pixel / fullW / fullH) % fullD);
  if (z - offD < insideD && h - offH < insideH && w - offW < insideW)
    return;
  out[tid] = bias ? bias[c] : T(0);
}
} // namespace

namespace {
/// The same with one 16-byte vector per thread and 32-bit arithmetic inside
/// an image (blockIdx.y, .z: the image); channel counts that are whole
/// vectors.
template <class T>
__global__ __launch_bounds__(256) void fillOutputPaddingVectorKernel(
    T *__restrict__ out, const T *__restrict__ bias, uint32_t imageVectors,
    uint32_t fullH, uint32_t fullW, uint32_t offD, uint32_t offH,
    uint32_t offW, uint32_t insideD, uint32_t insideH, uint32_t insideW,
    uint32_t vecsPerPixel) {
  constexpr uint32_t kVec = 16 / sizeof(T);
  const uint32_t idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= imageVectors)
    return;
  const uint32_t pixel = idx / vecsPerPixel, vec = idx - pixel * vecsPerPixel;
  const uint32_t row = pixel / fullW, w = pixel - row * fullW;
  const uint32_t z = row / fullH, h = row - z * fullH;
  if (z - offD < insideD && h - offH < insideH && w - offW < insideW)
    return;
  const uint64_t image = uint64_t(blockIdx.z) * gridDim.y + blockIdx.y;
  uint4 v{0, 0, 0, 0};
  if (bias)
    v = *reinterpret_cast<const uint4 *>(bias + vec * kVec);
  reinterpret_cast<uint4 *>(out)[image * imageVectors + idx] = v;
}
} // namespace

hipError_t launchFillOutputPadding(int type, void *out, const void *bias,
                                   uint64_t images, uint32_t fullD,
                                   uint32_t fullH, uint32_t fullW,
                                   uint32_t offD, uint32_t offH,
                                   uint32_t offW, uint32_t insideD,
                                   uint32_t insideH, uint32_t insideW,
                                   uint32_t chans, hipStream_t stream) {
  const uint64_t total = images * fullD * fullH * fullW * chans;
  if (total == 0)
    return hipSuccess;
  const uint32_t vecElems = type == kHalf ? 8 : 4;
  const uint64_t imageVectors =
      uint64_t(fullD) * fullH * fullW * (chans / vecElems);
  if ((type == kHalf || type == kFloat) && chans % vecElems == 0 &&
      imageVectors < (1ull << 31) &&
      (bias == nullptr || reinterpret_cast<uintptr_t>(bias) % 16 == 0) &&
      reinterpret_cast<uintptr_t>(out) % 16 == 0) {
    // images as grid y (and z beyond 32768 of them)
    const uint32_t gy = uint32_t(images < 32768 ? images : 32768);
    if (images % gy == 0 && images / gy < 65536) {
      const dim3 grid{uint32_t((imageVectors + 255) / 256), gy,
                      uint32_t(images / gy)};
      if (type == kHalf)
        hipLaunchKernelGGL(fillOutputPaddingVectorKernel<__half>, grid,
                           dim3(256), 0, stream, static_cast<__half *>(out),
                           static_cast<const __half *>(bias),
                           uint32_t(imageVectors), fullH, fullW, offD, offH,
                           offW, insideD, insideH, insideW, chans / vecElems);
      else
        hipLaunchKernelGGL(fillOutputPaddingVectorKernel<float>, grid,
                           dim3(256), 0, stream, static_cast<float *>(out),
                           static_cast<const float *>(bias),
                           uint32_t(imageVectors), fullH, fullW, offD, offH,
                           offW, insideD, insideH, insideW, chans / vecElems);
      return hipGetLastError();
    }
  }
  const uint64_t blocks = (total + 255) / 256;
  if (blocks > 0x7fffffffull)
    return hipErrorInvalidConfiguration;
  if (type == kHalf)
    hipLaunchKernelGGL(fillOutputPaddingKernel<__half>, dim3(uint32_t(blocks)),
                       dim3(256), 0, stream, static_cast<__half *>(out),
                       static_cast<const __half *>(bias), total, fullD, fullH,
                       fullW, offD, offH, offW, insideD, insideH, insideW,
                       chans);
  else if (type == kFloat)
    hipLaunchKernelGGL(fillOutputPaddingKernel<float>, dim3(uint32_t(blocks)),
                       dim3(256), 0, stream, static_cast<float *>(out),
                       static_cast<const float *>(bias), total, fullD, fullH,
                       fullW, offD, offH, offW, insideD, insideH, insideW,
                       chans);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

/// Parts the rows are summed in: 64 rows or more each, one workgroup per CU
/// at most (biasUpdateKernel takes kBiasSplits of them).
uint32_t biasUpdateSplits(uint64_t rows) {
  const uint64_t splits = (rows + 63) / 64;
  return uint32_t(splits < 1 ? 1 : splits > kBiasSplits ? kBiasSplits : splits);
}

size_t biasUpdateWorkspaceBytes(uint64_t rows, uint64_t channels) {
  return size_t(biasUpdateSplits(rows)) * channels * sizeof(float);
}

namespace {
template <typename T>
hipError_t launchChannelSum(const T *z, float *partial, uint64_t rows,
                            uint64_t channels, uint32_t splits,
                            hipStream_t stream) {
  constexpr uint32_t kVec = 16 / sizeof(T);
  const bool vectors =
      channels % kVec == 0 && reinterpret_cast<uintptr_t>(z) % 16 == 0;
  const uint64_t vecs = vectors ? channels / kVec : channels;
  const uint64_t chunks = (vecs + kReduceVecs - 1) / kReduceVecs;
  const uint32_t perBlock = uint32_t((vecs + chunks - 1) / chunks);
  const uint64_t rowsPerSplit = (rows + splits - 1) / splits;
  if (chunks > 0x7fffffffull || rowsPerSplit > 0x7fffffffull)
    return hipErrorInvalidConfiguration;
  const dim3 grid{uint32_t(chunks), splits}, block{256};
  if (vectors)
    hipLaunchKernelGGL((channelSumKernel<T, kVec>), grid, block, 0, stream, z,
                       partial, rows, channels, rowsPerSplit, perBlock);
  else
    hipLaunchKernelGGL((channelSumKernel<T, 1>), grid, block, 0, stream, z,
                       partial, rows, channels, rowsPerSplit, perBlock);
  return hipGetLastError();
}
} // namespace

hipError_t launchBiasUpdate(int deltasType, const void *zDeltas, uint64_t rows,
                            uint64_t channels, int biasType, void *biases,
                            float scale, void *workspace, hipStream_t stream) {
  if (channels == 0)
    return hipSuccess;
  const uint64_t blocks = (channels + kBiasChans - 1) / kBiasChans;
  if (blocks > 0x7fffffffull)
    return hipErrorInvalidConfiguration;
  const uint64_t vecElems = deltasType == kFloat ? 4 : 8;
  const bool vectors = channels % vecElems == 0 &&
                       reinterpret_cast<uintptr_t>(zDeltas) % 16 == 0;
  const uint64_t rowBytes = channels * (deltasType == kFloat ? 4 : 2);
  if (rows <= (!vectors                        ? kDirectRaggedRows
               : rowBytes <= 128               ? kDirectLineRows
               : rows * rowBytes <= (1u << 20) ? kDirectSmallRows
                                               : kDirectRows)) {
    auto direct = [&](auto *z, auto *b) {
      using T = std::remove_const_t<std::remove_pointer_t<decltype(z)>>;
      using B = std::remove_pointer_t<decltype(b)>;
      constexpr int kVec = 16 / sizeof(T);
      const uint32_t n =
          uint32_t((channels + kDirectChans - 1) / kDirectChans);
      const uint32_t paired = sizeof(T) == 2 ? n & ~15u : 0;
      if (vectors)
        hipLaunchKernelGGL((biasDirectKernel<T, kVec, B>), dim3{n}, dim3{1024},
                           0, stream, z, b, scale, uint32_t(rows), channels,
                           paired);
      else
        hipLaunchKernelGGL((biasDirectKernel<T, 1, B>), dim3{n}, dim3{1024}, 0,
                           stream, z, b, scale, uint32_t(rows), channels,
                           paired);
      return hipGetLastError();
    };
    auto ofBias = [&](auto *z) {
      return biasType == kFloat  ? direct(z, static_cast<float *>(biases))
             : biasType == kHalf ? direct(z, static_cast<__half *>(biases))
                                 : hipErrorInvalidValue;
    };
    return deltasType == kFloat ? ofBias(static_cast<const float *>(zDeltas))
           : deltasType == kHalf
               ? ofBias(static_cast<const __half *>(zDeltas))
               : hipErrorInvalidValue;
  }
  const uint32_t splits = biasUpdateSplits(rows);
  float *partial = static_cast<float *>(workspace);
  hipError_t e;
  if (deltasType == kFloat)
    e = launchChannelSum(static_cast<const float *>(zDeltas), partial, rows,
                         channels, splits, stream);
  else if (deltasType == kHalf)
    e = launchChannelSum(static_cast<const __half *>(zDeltas), partial, rows,
                         channels, splits, stream);
  else
    return hipErrorInvalidValue;
  if (e != hipSuccess)
    return e;
  const dim3 grid{uint32_t(blocks)}, block{256};
  const bool wide = channels * kBiasSplits * 4 >= (1ull << 31);
  auto update = [&](auto *b) {
    using T = std::remove_pointer_t<decltype(b)>;
    hipLaunchKernelGGL((wide ? &biasUpdateKernel<T, true>
                             : &biasUpdateKernel<T, false>),
                       grid, block, 0, stream, b, partial, scale, channels,
                       splits);
  };
  if (biasType == kFloat)
    update(static_cast<float *>(biases));
  else if (biasType == kHalf)
    update(static_cast<__half *>(biases));
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

hipError_t launchUnfuseGroupWeights(const void *src, void *dst,
                                    uint64_t groups, uint64_t perGroup,
                                    uint64_t co, uint64_t ci, uint64_t taps,
                                    int elemBytes, hipStream_t stream) {
  const uint64_t total = groups * co * ci * taps;
  if (total == 0)
    return hipSuccess;
  const uint64_t blocks = (total + 255) / 256;
  if (blocks > 0x7fffffffull || groups % perGroup != 0)
    return hipErrorInvalidConfiguration;
  const dim3 grid{uint32_t(blocks)}, block{256};
  if (elemBytes == 4)
    hipLaunchKernelGGL(unfuseGroupWeightsKernel<uint32_t>, grid, block, 0,
                       stream, static_cast<const uint32_t *>(src),
                       static_cast<uint32_t *>(dst), perGroup, co, ci, taps,
                       total);
  else if (elemBytes == 2)
    hipLaunchKernelGGL(unfuseGroupWeightsKernel<uint16_t>, grid, block, 0,
                       stream, static_cast<const uint16_t *>(src),
                       static_cast<uint16_t *>(dst), perGroup, co, ci, taps,
                       total);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

hipError_t launchScaledAdd(int type, void *a, float scaleA, const void *b,
                           float scaleB, uint64_t total, hipStream_t stream) {
  if (total == 0)
    return hipSuccess;
  const uint64_t blocks = (total + 255) / 256;
  if (blocks > 0x7fffffffull)
    return hipErrorInvalidConfiguration;
  const dim3 grid{uint32_t(blocks)}, block{256};
  if (type == kFloat)
    hipLaunchKernelGGL(scaledAddKernel<float>, grid, block, 0, stream,
                       static_cast<float *>(a), scaleA,
                       static_cast<const float *>(b), scaleB, total);
  else if (type == kHalf)
    hipLaunchKernelGGL(scaledAddKernel<__half>, grid, block, 0, stream,
                       static_cast<__half *>(a), scaleA,
                       static_cast<const __half *>(b), scaleB, total);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

} // namespace mxk
