// Weight deltas of a dense layer (any stride) on the matrix cores, straight
// from the layer's own tensors:
//   dW[g][co][ci][kh][kw] = sum over b, y, x of
//       deltas[b][y][x][g][co] *
//           acts[b][y strideH + kh - padH][x strideW + kw - padW][g][ci]
// (PopLibs runs this as a convolution of its own with batch and channels
// exchanged, lib/poplin/Convolution.cpp:3437-3483 calculateWeightDeltas, whose
// tensors Poplar rearranges on the exchange; here that would be two transposes
// through HBM per pass.)
//
// As a matrix product per kernel tap: M = output channels, N = input channels,
// K = pixels (b, y, x).  Both operands are stored with K outermost - a pixel's
// channels are consecutive, the next pixel follows - which is the wrong way
// round for an MFMA (a lane holds 8 consecutive k of one row).  gfx950's
// transposing LDS read (ds_read_b64_tr_b16) turns that round on the way to the
// registers: 16 lanes that point at 4 k-rows of 16 consecutive channels get,
// each, one channel's 4 k values.  So the tensors go from HBM to LDS as they
// are, 1 KB per wave-wide load, and no transposed copy is ever made.
//
// Workgroup = (chunk of pixels, tap, 128 x 128 tile of channels), 8 waves.
// The pixels of a chunk pass through LDS in super-steps of 64: two 32-pixel
// halves, each half a tile of deltas [32][128 co] and one of activations
// [32][128 ci] (the tap's shifted view of the input: pixel + tap offset, zeros
// outside - out-of-range buffer offsets).  Waves 0-3 multiply the first half,
// waves 4-7 the second: a 2 x 2 grid of 64 x 64 tiles per half, the two waves
// of a SIMD covering each other's latencies; their sums meet in LDS at the
// end.  The fp32 tile goes to the workspace as the registers hold it (1 KB
// blocks of 16 x 16 channels, a lane's four sums together); a second kernel
// adds the chunks' tiles in a fixed order and writes the deltas in weight
// order.  N = 32, 28 x 28, 3 x 3, 128 -> 128: 14.8 us (18.9 with a chunk's
// workgroups spread over the XCDs, which store rows of a tile as fast but
// fetch every pixel nine times).  Channel counts that are no whole 16-byte vectors come as copies
// with their channels filled up.
//
// LDS tile: 32 rows (pixels) of 256 bytes, no padding (a wave-wide load
// writes 4 rows at once); the 16-byte chunk c of row r sits at chunk position
// c ^ 2 ((r % 4) + 4 ((r / 8) % 2)), which spreads the 16 rows a transposing
// read touches over all banks.
#include "igemm_common.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace mxk {
namespace {

constexpr int kWuThreads = 512;
constexpr int kWuStages = 4;
constexpr uint32_t kWuTable = 2048; // pixels of the table
constexpr int kWuTileBytes = 32 * 256;           // 32 pixels x 128 channels
constexpr int kWuStageBytes = 4 * kWuTileBytes;   // 2 halves x 2 operands
constexpr uint32_t kWuInvalid = 0x40000000u;

typedef short shortx4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) shortx4 *LdsShortx4;

struct WuTapArgs {
  WuTapDesc d;
  uint32_t M;              // pixels: batch * outH * outW
  uint32_t taps, ciTiles, coTiles;
  uint32_t chunks, tilesPerChunk;
  uint32_t actPixelBytes, deltaPixelBytes; // groups * channels * 2
  uint32_t actImageBytes;                  // inH * inW * actPixelBytes
  uint64_t actBytes, deltaBytes;
  FastDiv divOutW, divOutH, divTaps, divCiTiles, divCoTiles, divKW;
  FastDiv divTilesPerChunk;
};

__device__ __forceinline__ half8 transposedOperand(const char *at) {
#if defined(__HIP_DEVICE_COMPILE__)
  // rows r .. r + 3 and r + 4 .. r + 7 of the lane's 16 channels
  const shortx4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (LdsShortx4)(at));
  const shortx4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (LdsShortx4)(at + 4 * 256));
  typedef short shortx8 __attribute__((ext_vector_type(8)));
  const shortx8 both = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
  return __builtin_bit_cast(half8, both);
#else
  return half8{};
#endif
}

/// IDLE: some tile's channels leave half of its columns or rows, and with them
/// two or more waves, without any.
template <bool IDLE>
__global__ __launch_bounds__(kWuThreads) void wuTapKernel(
    const WuTapArgs a, const char *__restrict__ acts,
    const char *__restrict__ deltas, float *__restrict__ partial) {
  extern __shared__ __align__(16) char lds[];
  const WuTapDesc &d = a.d;
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int grp = wave >> 2, wm = (wave >> 1) & 1, wn = wave & 1;

  // workgroup -> (chunk, group, tap, ci tile, co tile), co tile fastest; an
  // XCD gets whole chunks, whose pixels its L2 fetches once for all the taps
  const uint32_t block = xcdSwizzle(blockIdx.x, gridDim.x);
  const uint32_t chunk = a.divTilesPerChunk(block);
  uint32_t id = block - chunk * a.tilesPerChunk;
  uint32_t q = a.divCoTiles(id);
  const uint32_t coTile = id - q * a.coTiles;
  id = q, q = a.divCiTiles(id);
  const uint32_t ciTile = id - q * a.ciTiles;
  id = q, q = a.divTaps(id);
  const uint32_t tap = id - q * a.taps;
  const uint32_t g = q;
  const uint32_t kh = a.divKW(tap), kw = tap - kh * d.kW;
  const uint32_t p0 = chunk * d.chunkPixels;
  const uint32_t p1 = p0 + d.chunkPixels < a.M ? p0 + d.chunkPixels : a.M;
  const uint32_t steps = (p1 - p0 + 63) >> 6;

  // Loads.  Wave w brings rows 4 w .. 4 w + 3 of every tile: lane l row
  // 4 w + l / 16, chunk position l % 16, which holds channel chunk
  // (l % 16) ^ swizzle(row).
  const uint32_t row = wave * 4 + (lane >> 4);
  const uint32_t chanChunk =
      (lane & 15) ^ (2 * ((row & 3) + 4 * ((row >> 3) & 1)));
  const __amdgpu_buffer_rsrc_t actBuf = bufferOf(
      acts, uint32_t(a.actBytes < kWuInvalid ? a.actBytes : kWuInvalid));
  // (the deltas' buffer ends with the chunk)
  const __amdgpu_buffer_rsrc_t deltaBuf =
      bufferOf(deltas, p1 * a.deltaPixelBytes);
  const uint32_t actChan = ciTile * 128 + chanChunk * 8;
  const uint32_t deltaChan = coTile * 128 + chanChunk * 8;
  const uint32_t actLane = actChan < d.ci ? (g * d.ci + actChan) * 2 : kWuInvalid;
  const uint32_t deltaLane =
      deltaChan < d.co ? (g * d.co + deltaChan) * 2 : kWuInvalid;
  // Where a pixel's activations are under this tap, or that there are none: a
  // table in LDS, worked out a thread per pixel, 512 pixels at a time and two such
  // groups ahead of the loads; an entry is read a step before its load.  (A wave
  // issues an instruction every 5 to 8 cycles, whatever the other one of its SIMD
  // does: with 34 of carries per step and lane in place of the look-up it took
  // 122 a step instead of 66, and the pass 21.9 us for N = 32, 28 x 28, 3 x 3,
  // 128 -> 128, now 20.3; 25 x 57 x 57 at stride 2, 72 -> 200, 24.2 -> 21.3.)
  uint32_t *table = reinterpret_cast<uint32_t *>(lds + kWuStages * kWuStageBytes);
  const uint32_t tapY = kh - uint32_t(d.padH), tapX = kw - uint32_t(d.padW);
  auto workOut = [&](uint32_t n) {
    const uint32_t p = p0 + n + t;
    const uint32_t pr = a.divOutW(p), b = a.divOutH(pr);
    const uint32_t x = p - pr * d.outW, y = pr - b * d.outH;
    const uint32_t iy = y * d.strideH + tapY, ix = x * d.strideW + tapX;
    const bool inside = p < p1 && iy - d.loH < d.hiH - d.loH &&
                        ix - d.loW < d.hiW - d.loW;
    table[(n + t) % kWuTable] =
        inside ? b * a.actImageBytes + (iy * d.inW + ix) * a.actPixelBytes
               : kWuInvalid;
  };
  uint32_t deltaAt[2], actAt[2], looked = row;
#pragma unroll
  for (int h = 0; h != 2; ++h)
    deltaAt[h] = (p0 + h * 32 + row) * a.deltaPixelBytes + deltaLane;
  auto look = [&](const uint32_t *__restrict__ entries) {
#pragma unroll
    for (int h = 0; h != 2; ++h)
      actAt[h] = entries[looked + h * 32];
    looked = (looked + 64) % kWuTable;
  };
  auto load = [&](char *__restrict__ into) {
    char *stage = into + wave * 1024;
#pragma unroll
    for (int h = 0; h != 2; ++h) {
      loadToLds(deltaBuf, (LdsPtr)(stage + (2 * h) * kWuTileBytes), deltaAt[h],
                0);
      // (any sum with a kWuInvalid in it lies beyond the buffer and reads
      // as zeros)
      loadToLds(actBuf, (LdsPtr)(stage + (2 * h + 1) * kWuTileBytes),
                actAt[h] + actLane, 0);
      deltaAt[h] += 64 * a.deltaPixelBytes;
    }
  };

  // Reads.  For a block of 16 channels starting at chunk 2 blk of the tile,
  // lane l = (quarter b = l / 16, i = l % 16) points at row 8 b + i / 4 and
  // the 8 bytes of channels 4 (i % 4) .. + 3.
  const uint32_t rb = lane >> 4, ri = lane & 15;
  const uint32_t readRow = 8 * rb + (ri >> 2);
  const uint32_t readSwizzle = 2 * ((ri >> 2) + 4 * (rb & 1));
  uint32_t deltaOff[4], actOff[4];
#pragma unroll
  for (int blk = 0; blk != 4; ++blk) {
    const uint32_t dChunk = 2 * (wm * 4 + blk) + ((ri & 3) >> 1);
    const uint32_t aChunk = 2 * (wn * 4 + blk) + ((ri & 3) >> 1);
    deltaOff[blk] =
        readRow * 256 + ((dChunk ^ readSwizzle) * 16) + 8 * (ri & 1);
    actOff[blk] = kWuTileBytes + readRow * 256 +
                  ((aChunk ^ readSwizzle) * 16) + 8 * (ri & 1);
  }

  floatx4 acc[4][4];
#pragma unroll
  for (int i = 0; i != 4; ++i)
#pragma unroll
    for (int j = 0; j != 4; ++j)
      acc[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
  // Channels of this tile, and whether this wave's quarter has any.
  const uint32_t ciHere = d.ci - ciTile * 128, coHere = d.co - coTile * 128;
  const bool busy = wn * 64u < ciHere && wm * 64u < coHere;

  // Software pipeline.  Iteration `step`: wait for step + 1's tiles, issue
  // the loads of step + kWuStages into the stage that step's operands were
  // read from (in the iteration before), read step + 1's operands, and only
  // then multiply step's, so that the reads run under the MFMAs.  (The loop
  // waits for the transposing reads and the loads' way from the L2; with a
  // chunk's taps spread over the XCDs it waited for their links to memory.)
  // (`__restrict__` on the stage written and the stage read, so that the
  // compiler does not make the reads wait for the loads just issued: a load
  // that writes LDS is a pending LDS write to it.)
  struct Operands {
    half8 da[4], ab[4];
  };
  auto read = [&](Operands &o, const char *__restrict__ tile) {
#pragma unroll
    for (int blk = 0; blk != 4; ++blk)
      o.da[blk] = transposedOperand(tile + deltaOff[blk]);
#pragma unroll
    for (int blk = 0; blk != 4; ++blk)
      o.ab[blk] = transposedOperand(tile + actOff[blk]);
  };
  auto multiply = [&](const Operands &o) {
#pragma unroll
    for (int i = 0; i != 4; ++i)
#pragma unroll
      for (int j = 0; j != 4; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(o.da[i], o.ab[j],
                                                           acc[i][j], 0, 0, 0);
  };
  auto tileOf = [&](uint32_t step) {
    return lds + (step % kWuStages) * kWuStageBytes + grp * 2 * kWuTileBytes;
  };
  // (No branches in the loop: loads are issued for steps beyond the chunk's
  // last too - all out of range, they write zeros - and an odd count of steps
  // is rounded up, the extra one multiplying zeros.  So the loads of exactly
  // two steps, 4 each, are behind the one waited for.)
  auto iteration = [&](const Operands &cur, Operands &next,
                       char *__restrict__ into, const char *__restrict__ from,
                       const uint32_t *__restrict__ entries) {
    MXK_WAIT_VMCNT(8);
    stepBarrier();
    // (everybody's reads of step's stage finished an iteration ago)
    load(into);
    look(entries);
    if (!IDLE || busy) {
      read(next, from);
      multiply(cur);
    }
    MXK_WAIT_LGKMCNT0();
  };
  workOut(0);
  workOut(kWuThreads);
  __syncthreads();
#pragma unroll
  for (int s = 0; s != kWuStages; ++s) {
    look(table);
    load(lds + s * kWuStageBytes);
  }
  look(table);
  Operands even, odd;
  MXK_WAIT_VMCNT(12);
  stepBarrier();
  read(even, tileOf(0));
  MXK_WAIT_LGKMCNT0();
  for (uint32_t step = 0; step < steps; step += 2) {
    // (looked up eleven steps on at the earliest, behind as many barriers)
    if (step % 8 == 0)
      workOut((step + 16) * 64);
    iteration(even, odd, lds + (step % kWuStages) * kWuStageBytes,
              tileOf(step + 1), table);
    iteration(odd, even, lds + ((step + 1) % kWuStages) * kWuStageBytes,
              tileOf(step + 2), table);
  }
  MXK_WAIT_VMCNT(0);

  // The halves' sums meet: the first half's waves finish the blocks of 16
  // output channels 0 and 1 of a wave's four, the second half's 2 and 3, each
  // getting the other's part through LDS and storing 1 KB per block.
  // Written through the L2: the other kernel reads the tiles from every XCD,
  // and what is left dirty has to be written back before it starts (25.8 ->
  // 25.0 us for the pass).  Blocks without a channel are left out.
  __syncthreads();
  uintx4 *exchange = reinterpret_cast<uintx4 *>(lds);
  const int quadrant = wave & 3;
  float *dst = partial + ((((size_t(chunk) * d.groups + g) * a.taps + tap) *
                               a.ciTiles +
                           ciTile) *
                              a.coTiles +
                          coTile) *
                             (128 * 128);
  const __amdgpu_buffer_rsrc_t tileBuf = bufferOf(dst, 128 * 128 * 4);
  using Low = std::integral_constant<int, 0>;
  using High = std::integral_constant<int, 2>;
  auto handOver = [&](auto first) {
#pragma unroll
    for (int i = 0; i != 2; ++i)
#pragma unroll
      for (int j = 0; j != 4; ++j)
        exchange[((grp * 4 + quadrant) * 8 + i * 4 + j) * 64 + lane] =
            __builtin_bit_cast(uintx4, acc[decltype(first)::value + i][j]);
  };
  auto finish = [&](auto first) {
#pragma unroll
    for (int i = 0; i != 2; ++i)
#pragma unroll
      for (int j = 0; j != 4; ++j) {
        constexpr int FIRST = decltype(first)::value;
        const floatx4 other = __builtin_bit_cast(
            floatx4,
            exchange[(((grp ^ 1) * 4 + quadrant) * 8 + i * 4 + j) * 64 + lane]);
        const floatx4 sum = acc[FIRST + i][j] + other;
        if (wn * 64u + j * 16 < ciHere &&
            wm * 64u + (FIRST + i) * 16 < coHere)
          __builtin_amdgcn_raw_buffer_store_b128(
              __builtin_bit_cast(uintx4, sum), tileBuf,
              ((quadrant * 16 + (FIRST + i) * 4 + j) * 64 + lane) * 16, 0,
              kWriteThroughStore);
      }
  };
  if (grp == 0)
    handOver(High{});
  else
    handOver(Low{});
  __syncthreads();
  if (grp == 0)
    finish(Low{});
  else
    finish(High{});
}

/// deltas[g][co][ci][tap] = sum over the chunks in a fixed order.  Workgroup =
/// ciPer blocks of 16 input channels x 4 output channels and all their taps
/// (kWuSumSlots slots at most): 16 lanes read a tile's 256 bytes, slot (block,
/// tap, part) the chunks part, part + parts, ..., four loads in flight; the
/// parts meet in LDS, whence runs of 16 ciPer input channels x taps leave in
/// weight order.
/// Bound by the tiles' bytes and one trip to memory and back: the 16.5 MB of
/// N = 32, 28 x 28, 3 x 3, 128 -> 128 in 4.6 us.  (A lane per output vector
/// wrote 2 bytes here and there: 5.2 us, and where the result is large, 1 x 1
/// 64 -> 256 or 3 x 3 384 -> 264, 8.1 and 8.6 us against 4.8 and 5.6.)
/// Large results of few taps and chunks make thousands of small workgroups,
/// whose turnover then sets the pace: as many blocks to a workgroup as leave
/// 2 048 of them (1 024 -> 2 048 channels, 1 x 1, two chunks, 32 768 workgroups
/// of a wave each, the pass 32.4 -> 21.2 us; 512 -> 2 048, 7 x 7, 23.1 -> 18.8; a
/// limit of 512, 1 024 or 4 096 is within 3 % over 17 layers).
constexpr uint32_t kWuSumSlots = 64, kWuSumParts = 32;
constexpr uint32_t kWuSumWorkgroups = 2048;

struct WuSumArgs {
  uint32_t groups, chunks, taps;
  uint32_t ci, co; // channels of the result
  uint32_t ciTiles, coTiles;
  uint32_t tapsHere;             // of a workgroup
  uint32_t parts;                // slots that share a tap
  uint32_t ciBlocks, coQuads;
  uint32_t ciPer, ciGroups;      // blocks of a workgroup, groups of them
  FastDiv divParts, divCoQuads, divCiGroups, divTaps, divRun;
};

template <class OutT>
__global__ __launch_bounds__(1024) void wuTapSumKernel(
    const float *__restrict__ partial, OutT *__restrict__ out,
    const WuSumArgs a) {
  __shared__ floatx4 sums[kWuSumSlots * 16];
  uint32_t id = blockIdx.x, q = a.divCoQuads(id);
  const uint32_t coQuad = id - q * a.coQuads;
  id = q, q = a.divCiGroups(id);
  const uint32_t ciBlock0 = (id - q * a.ciGroups) * a.ciPer, g = q;
  const uint32_t tap0 = blockIdx.y * a.tapsHere;
  const uint32_t left = a.taps - tap0;
  const uint32_t taps = left < a.tapsHere ? left : a.tapsHere;
  const uint32_t slot = threadIdx.x >> 4;
  const uint32_t sum = a.divParts(slot), part = slot - sum * a.parts;
  const uint32_t blockHere = a.divTaps(sum);
  const uint32_t tapHere = sum - blockHere * a.tapsHere;
  const uint32_t ciBlock = ciBlock0 + blockHere;
  if (blockHere < a.ciPer && ciBlock < a.ciBlocks && tapHere < taps) {
    const size_t tile = 128 * 128 / 4; // (in vectors)
    const size_t stride =
        size_t(a.groups) * a.taps * a.ciTiles * a.coTiles * tile;
    const floatx4 *src =
        reinterpret_cast<const floatx4 *>(partial) +
        (((size_t(g) * a.taps + tap0 + tapHere) * a.ciTiles + ciBlock / 8) *
             a.coTiles +
         coQuad / 32) *
            tile +
        (((coQuad % 32 / 16) * 2 + ciBlock % 8 / 4) * 16 +
         coQuad % 16 / 4 * 4 + ciBlock % 4) *
            64 +
        coQuad % 4 * 16 + (threadIdx.x & 15);
    floatx4 total = {0.0f, 0.0f, 0.0f, 0.0f};
    uint32_t p = part;
    for (; p + 3 * a.parts < a.chunks; p += 4 * a.parts) {
      const floatx4 v0 = src[p * stride];
      const floatx4 v1 = src[(p + a.parts) * stride];
      const floatx4 v2 = src[(p + 2 * a.parts) * stride];
      const floatx4 v3 = src[(p + 3 * a.parts) * stride];
      total += (v0 + v1) + (v2 + v3);
    }
    for (; p < a.chunks; p += a.parts)
      total += src[p * stride];
    sums[threadIdx.x] = total;
  }
  __syncthreads();
  // element e of the workgroup's 4 x 16 ciPer x taps results, taps fastest
  const float *flat = reinterpret_cast<const float *>(sums);
  const uint32_t run = 16 * a.ciPer * a.tapsHere;
  for (uint32_t e = threadIdx.x; e < 4 * run; e += blockDim.x) {
    const uint32_t c = a.divRun(e), inRun = e - c * run;
    const uint32_t i = a.divTaps(inRun), tap = inRun - i * a.tapsHere;
    const uint32_t co = coQuad * 4 + c, ci = ciBlock0 * 16 + i;
    if (tap >= taps || ci >= a.ci || co >= a.co)
      continue;
    float v = 0.0f;
    const uint32_t first = ((i >> 4) * a.tapsHere + tap) * a.parts;
    for (uint32_t p = 0; p != a.parts; ++p)
      v += flat[((first + p) * 16 + (i & 15)) * 4 + c];
    storeOut(out, ((size_t(g) * a.co + co) * a.ci + ci) * a.taps + tap0 + tap,
             v);
  }
}

uint64_t tilesOf(const WuTapDesc &d) {
  return uint64_t(d.groups) * d.kH * d.kW * ((d.ci + 127) / 128) *
         ((d.co + 127) / 128);
}

} // namespace

bool wuTapTakes(const WuTapDesc &d) {
  const uint64_t M = uint64_t(d.batch) * d.outH * d.outW;
  if (M == 0 || d.ci % 8 != 0 || d.co % 8 != 0 || d.ci == 0 || d.co == 0 ||
      d.kH == 0 || d.kW == 0 || d.strideH == 0 || d.strideW == 0)
    return false;
  const uint64_t actBytes =
      uint64_t(d.batch) * d.inH * d.inW * d.groups * d.ci * 2;
  const uint64_t deltaBytes = M * d.groups * d.co * 2;
  if (actBytes >= kWuInvalid || deltaBytes >= kWuInvalid || M >= kWuInvalid)
    return false;
  if (d.chunkPixels == 0 || d.chunkPixels % 64 != 0)
    return false;
  if (d.resultCi > d.ci || d.resultCo > d.co)
    return false;
  const uint64_t chunks = (M + d.chunkPixels - 1) / d.chunkPixels;
  return chunks * tilesOf(d) <= 0x7fffffffull &&
         wuTapWorkspaceBytes(d) <= (1ull << 31);
}

uint32_t wuTapChunkPixels(const WuTapDesc &d, uint32_t computeUnits) {
  // One workgroup to a CU at a time: as many chunks of whole super-steps of 64
  // pixels as the estimate finds the fastest, which are about one workgroup for
  // every CU or some whole rounds of them (N = 32, 14 x 14, 3 x 3, 512 -> 512, 144
  // tiles: one chunk 67 us with the sum, three 58).
  const uint64_t M = uint64_t(d.batch) * d.outH * d.outW;
  const uint64_t tiles = std::max<uint64_t>(1, tilesOf(d));
  uint64_t best = 0;
  double bestUs = 0;
  for (uint64_t n = 1; n <= 8 || n * tiles <= computeUnits; ++n) {
    uint64_t pixels = (M + n - 1) / n;
    pixels = std::max<uint64_t>(256, (pixels + 63) / 64 * 64);
    const uint64_t chunks = (M + pixels - 1) / pixels;
    // (no more than the workspace may hold: wuTapTakes)
    if (best && chunks * tiles * 65536 > (1ull << 31))
      break;
    WuTapDesc t = d;
    t.chunkPixels = uint32_t(std::min<uint64_t>(pixels, 1u << 30));
    const double us = wuTapEstimateUs(t, computeUnits);
    if (!best || us < bestUs)
      best = t.chunkPixels, bestUs = us;
    if (pixels == 256)
      break;
  }
  return uint32_t(best);
}

uint64_t wuTapWorkspaceBytes(const WuTapDesc &d) {
  const uint64_t M = uint64_t(d.batch) * d.outH * d.outW;
  if (d.chunkPixels == 0)
    return 0;
  const uint64_t chunks = (M + d.chunkPixels - 1) / d.chunkPixels;
  return chunks * tilesOf(d) * 128 * 128 * 4;
}

double wuTapEstimateUs(const WuTapDesc &d, uint32_t computeUnits) {
  // Fitted to 3 070 measurements on 379 random layers (4 to 64 images of 7 to 64
  // squared, 24 to 512 channels, 1 x 1 to 5 x 5, up to ten counts of chunks each),
  // within 5 %; the count picked by it is on average 1 % behind the best.
  const uint64_t M = uint64_t(d.batch) * d.outH * d.outW;
  const double steps =
      double((std::min<uint64_t>(d.chunkPixels, M) + 63) / 64);
  const double chunks = double((M + d.chunkPixels - 1) / d.chunkPixels);
  const double perCU = chunks * double(tilesOf(d)) / double(computeUnits);
  const double rounds = std::max(1.0, std::ceil(perCU));
  const double deltasMB =
      double(d.groups) * d.ci * d.co * d.kH * d.kW * 1e-6;
  const double partialMB = 4.0 * deltasMB * chunks;
  // (pixels of whole 128-byte lines on both sides come, and go, faster)
  const bool lines = d.ci % 64 == 0 && d.co % 64 == 0;
  return 7.3 + (0.418 + 0.045 * std::min(perCU, 1.0) - (lines ? 0.026 : 0.0)) *
                   steps +
         (rounds - 1) * (3.5 + 0.4 * steps) +
         (lines ? 0.48 : 0.51) * std::min(partialMB, 14.4) +
         0.23 * std::max(partialMB - 14.4, 0.0) + 1.33 * deltasMB;
}

hipError_t launchWuTap(const WuTapDesc &d, int outType, const void *acts,
                       const void *deltas, void *workspace, void *out,
                       hipStream_t stream) {
  if (!wuTapTakes(d) || (outType != kHalf && outType != kFloat))
    return hipErrorInvalidValue;
  WuTapArgs a{};
  a.d = d;
  a.M = d.batch * d.outH * d.outW;
  a.taps = d.kH * d.kW;
  a.ciTiles = (d.ci + 127) / 128, a.coTiles = (d.co + 127) / 128;
  a.actPixelBytes = d.groups * d.ci * 2;
  a.deltaPixelBytes = d.groups * d.co * 2;
  a.actImageBytes = d.inH * d.inW * a.actPixelBytes;
  a.actBytes = uint64_t(d.batch) * a.actImageBytes;
  a.deltaBytes = uint64_t(a.M) * a.deltaPixelBytes;
  a.divOutW = makeFastDiv(d.outW), a.divOutH = makeFastDiv(d.outH);
  a.divTaps = makeFastDiv(a.taps), a.divCiTiles = makeFastDiv(a.ciTiles);
  a.divCoTiles = makeFastDiv(a.coTiles), a.divKW = makeFastDiv(d.kW);
  const uint32_t chunks = (a.M + d.chunkPixels - 1) / d.chunkPixels;
  a.chunks = chunks;
  a.tilesPerChunk = uint32_t(tilesOf(d));
  a.divTilesPerChunk = makeFastDiv(a.tilesPerChunk);
  const uint32_t blocks = chunks * a.tilesPerChunk;
  constexpr int kLds = kWuStages * kWuStageBytes + int(kWuTable) * 4;
  static_assert(kLds >= 64 * 1024, "room for the halves' exchange");
  static const hipError_t attr = [] {
    hipError_t e = hipSuccess;
    for (const void *k : {reinterpret_cast<const void *>(&wuTapKernel<false>),
                          reinterpret_cast<const void *>(&wuTapKernel<true>)})
      if (e == hipSuccess)
        e = hipFuncSetAttribute(
            k, hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    return e;
  }();
  if (attr != hipSuccess)
    return attr;
  const bool idle = (d.ci - 1) % 128 < 64 || (d.co - 1) % 128 < 64;
  const auto kernel = idle ? &wuTapKernel<true> : &wuTapKernel<false>;
  hipLaunchKernelGGL(kernel, dim3(blocks), dim3(kWuThreads), kLds, stream,
                     a, static_cast<const char *>(acts),
                     static_cast<const char *>(deltas),
                     static_cast<float *>(workspace));
  hipError_t e = hipGetLastError();
  if (e != hipSuccess)
    return e;
  WuSumArgs r{};
  r.groups = d.groups, r.chunks = chunks, r.taps = a.taps;
  r.ci = d.resultCi ? d.resultCi : d.ci, r.co = d.resultCo ? d.resultCo : d.co;
  r.ciTiles = a.ciTiles, r.coTiles = a.coTiles;
  r.tapsHere = std::min(a.taps, kWuSumSlots);
  r.parts = std::min({chunks, kWuSumSlots / r.tapsHere, kWuSumParts});
  r.ciBlocks = (r.ci + 15) / 16, r.coQuads = (r.co + 3) / 4;
  r.divParts = makeFastDiv(r.parts);
  r.divCoQuads = makeFastDiv(r.coQuads);
  const uint32_t tapBlocks = (a.taps + r.tapsHere - 1) / r.tapsHere;
  const uint64_t single =
      uint64_t(d.groups) * r.ciBlocks * r.coQuads * tapBlocks;
  r.ciPer = uint32_t(std::min<uint64_t>(
      {kWuSumSlots / (r.tapsHere * r.parts), r.ciBlocks,
       std::max<uint64_t>(1, single / kWuSumWorkgroups)}));
  r.ciGroups = (r.ciBlocks + r.ciPer - 1) / r.ciPer;
  r.divCiGroups = makeFastDiv(r.ciGroups);
  r.divTaps = makeFastDiv(r.tapsHere);
  r.divRun = makeFastDiv(16 * r.ciPer * r.tapsHere);
  const dim3 sumGrid(d.groups * r.ciGroups * r.coQuads, tapBlocks);
  const dim3 sumBlock((r.ciPer * r.tapsHere * r.parts * 16 + 63) / 64 * 64);
  if (outType == kHalf)
    hipLaunchKernelGGL(wuTapSumKernel<__half>, sumGrid, sumBlock, 0, stream,
                       static_cast<const float *>(workspace),
                       static_cast<__half *>(out), r);
  else
    hipLaunchKernelGGL(wuTapSumKernel<float>, sumGrid, sumBlock, 0, stream,
                       static_cast<const float *>(workspace),
                       static_cast<float *>(out), r);
  return hipGetLastError();
}

} // namespace mxk
