// Weight packing: from the external order [G][Co][Ci][kernel...] (or a matrix
// product's right-hand side, [G][Ci][Co]) to the order a matrix-core kernel
// reads.  One kernel for every layout, two threads per 16-byte vector of the
// packed weights; several packings of one set of weights - the phases of a
// convolution over a zero-stuffed input - and the block-diagonal weights of
// conv groups run as one all come out of a single launch.
//
// A training step packs its weights twice, so these launches are on its path;
// what they cost is latency: 31-bit indices taken apart with multiply-high
// divisions, the element loads of a thread all under way at once, one launch.
// (With 64-bit divisions and a launch per phase the four phases of a 3 x 3
// stride-2 layer of 200 -> 72 channels took 11.6 us, now 3.7.)
#include "device_types.hpp"
#include "kernels.hpp"

namespace mxk {
namespace {

// One wave per workgroup: each of a wave's loads touches up to 64 cache lines,
// which a compute unit takes one per cycle, so the waves are spread as far as
// they go.
constexpr uint32_t kPackThreads = 64;
constexpr uint32_t kPackParts = 2; // threads per vector

struct JobArgs {
  uint32_t firstVector; // of this job's threads
  uint32_t dstVector;   // where its packed weights start
  uint32_t steps;       // 16-byte vectors of a row, or k-steps of a block
  uint32_t blocks;      // rows, or blocks of channels, of a group
  uint32_t chunksPerTap, taps;
  FastDiv divSteps, divBlocks, divChunks;
  uint32_t selected, kW, kH, countH, countW;
  uint32_t firstD, stepD, firstH, stepH, firstW, stepW;
};

struct PackArgs {
  const void *src;
  uint2 *dst;
  uint32_t co, ci;     // of a group as the kernel runs it
  uint32_t srcCo, srcCi; // of a group as it is stored
  uint32_t fuse;       // stored groups in one of those
  uint32_t sourceTaps;
  uint32_t layout, chansTransposed;
  uint32_t total;
};

template <class T>
__device__ __forceinline__ void packVector(const PackArgs &a, const JobArgs &j,
                                           uint32_t part) {
  constexpr uint32_t kVec = 16 / sizeof(T);
  constexpr uint32_t kPart = kVec / kPackParts;
  const uint32_t id = part / kPackParts;
  // which channel, tap and first input channel this vector holds
  uint32_t n, tap, c0, g;
  if (a.layout == kPackRows) {
    const uint32_t row = j.divSteps(id), chunk = id - row * j.steps;
    g = j.divBlocks(row), n = row - g * j.blocks;
    tap = j.divChunks(chunk);
    c0 = (chunk - tap * j.chunksPerTap) * kVec;
  } else if (a.layout == kPackOperands16 || a.layout == kPackOperands32) {
    const uint32_t shift = a.layout == kPackOperands16 ? 4 : 5;
    const uint32_t lane = id & 63, q = id >> 6;
    const uint32_t block = j.divSteps(q), step = q - block * j.steps;
    g = j.divBlocks(block);
    n = ((block - g * j.blocks) << shift) + (lane & ((1u << shift) - 1));
    const uint32_t chunk = (step << (6 - shift)) + (lane >> shift);
    tap = j.divChunks(chunk);
    c0 = (chunk - tap * j.chunksPerTap) * kVec;
  } else {
    // resident patch: per k-step (a tap of a 128-byte channel slice) four
    // operands of the 32 channels of a block
    const uint32_t lane = id & 63, half = (id >> 7) & 1, low = (id >> 6) & 1;
    const uint32_t q = id >> 8;
    const uint32_t block = j.divSteps(q), step = q - block * j.steps;
    g = j.divBlocks(block);
    uint32_t within, chunk;
    if (a.layout == kPackPatch16) {
      // (K unit, column block) for fp16, (column block, half of the lane's 32
      // bytes) for fp8; lane = (K quarter, channel of the column block)
      within = (sizeof(T) == 2 ? low : half) * 16 + (lane & 15);
      chunk = (sizeof(T) == 2 ? half : low) * 4 + (lane >> 4);
    } else {
      within = lane & 31;
      chunk = half * 4 + (sizeof(T) == 2 ? low * 2 + (lane >> 5)
                                         : (lane >> 5) * 2 + low);
    }
    n = (block - g * j.blocks) * 32 + within;
    const uint32_t slice = j.divChunks(step); // (by the taps)
    tap = step - slice * j.taps;
    c0 = (slice * 8 + chunk) * kVec;
  }
  c0 += part % kPackParts * kPart;
  union {
    T e[kPart];
    uint2 u;
  } v;
  v.u = uint2{0, 0};
  if (n < a.co && tap < j.taps && c0 < a.ci) {
    if (j.selected) {
      const uint32_t row = tap / j.countW, w = tap - row * j.countW;
      const uint32_t plane = row / j.countH, h = row - plane * j.countH;
      tap = ((j.firstD + plane * j.stepD) * j.kH + j.firstH + h * j.stepH) *
                j.kW +
            j.firstW + w * j.stepW;
    }
    const T *src = static_cast<const T *>(a.src);
    // the element of c0 and the stride to the next channel's; channels that
    // are not there read the last one and are zeroed
    const T *from;
    uint32_t chans, stride = a.sourceTaps;
    uint32_t skip = 0; // leading channels of another group
    if (a.fuse > 1) {
      // block (x, y) of a fused group's channels is stored group x's where
      // x == y, else zero
      const uint32_t x = n / a.srcCo, lo = x * a.srcCi;
      skip = c0 < lo ? lo - c0 : 0;
      chans = lo + a.srcCi > c0 ? lo + a.srcCi - c0 : 0;
      from = src + (int64_t(g * a.fuse + x) * a.srcCo + n - x * a.srcCo) *
                       a.srcCi * a.sourceTaps +
             (int64_t(c0) - lo) * a.sourceTaps + tap;
    } else if (a.chansTransposed) {
      chans = a.ci - c0, stride = a.co;
      from = src + (uint64_t(g) * a.ci + c0) * a.co + n;
    } else {
      chans = a.ci - c0;
      from = src + ((uint64_t(g) * a.co + n) * a.ci + c0) * a.sourceTaps + tap;
    }
    if (skip < chans) {
      T e[kPart];
#pragma unroll
      for (uint32_t i = 0; i != kPart; ++i) {
        const uint32_t at = i < skip ? skip : i < chans ? i : chans - 1;
        e[i] = from[uint64_t(at) * stride];
      }
#pragma unroll
      for (uint32_t i = 0; i != kPart; ++i)
        v.e[i] = (i >= skip) & (i < chans) ? e[i] : T(0);
    }
  }
  a.dst[uint64_t(j.dstVector) * kPackParts + part] = v.u;
}

template <class T>
__global__ __launch_bounds__(kPackThreads) void
packWeightsKernel(PackArgs a, JobArgs job) {
  const uint32_t id = blockIdx.x * kPackThreads + threadIdx.x;
  if (id < a.total)
    packVector<T>(a, job, id);
}

/// Every job starts with a workgroup of its own.
struct ManyJobs {
  uint32_t count;
  JobArgs job[kIgemmMaxFused];
};
template <class T>
__global__ __launch_bounds__(kPackThreads) void
packManyWeightsKernel(PackArgs a, ManyJobs m) {
  const uint32_t at = blockIdx.x * kPackThreads;
  uint32_t i = 0;
  while (i + 1 < m.count && at >= m.job[i + 1].firstVector)
    ++i;
  const uint32_t id = at - m.job[i].firstVector + threadIdx.x;
  const uint32_t parts = m.job[i].steps * m.job[i].blocks * a.total;
  if (id < parts)
    packVector<T>(a, m.job[i], id);
}

} // namespace

hipError_t launchPackWeights(const PackSource &s, PackLayout layout,
                             const PackJob *jobs, size_t count, void *dst,
                             hipStream_t stream) {
  if (count == 0)
    return hipSuccess;
  if (count > kIgemmMaxFused || s.groups % s.fuse != 0 ||
      (s.elemBytes != 1 && s.elemBytes != 2 && s.elemBytes != 4))
    return hipErrorInvalidValue;
  const uint32_t vec = 16 / s.elemBytes;
  const uint32_t groups = s.groups / s.fuse;
  PackArgs a{};
  a.src = s.weights, a.dst = static_cast<uint2 *>(dst);
  a.co = s.co * s.fuse, a.ci = s.ci * s.fuse;
  a.srcCo = s.co, a.srcCi = s.ci, a.fuse = s.fuse, a.sourceTaps = s.taps;
  a.layout = uint32_t(layout), a.chansTransposed = s.chansTransposed ? 1 : 0;
  // vectors of a (block, k-step): one of a row, else 64 lanes' (x 4 operands)
  const uint32_t unit = layout == kPackRows ? 1
                        : layout == kPackPatch16 || layout == kPackPatch32
                            ? 256
                            : 64;
  ManyJobs m{};
  uint64_t first = 0;
  for (size_t i = 0; i != count; ++i) {
    const PackJob &x = jobs[i];
    JobArgs &j = m.job[m.count];
    const uint64_t vectors = uint64_t(groups) * x.blocks * x.steps * unit;
    const uint64_t parts = vectors * kPackParts;
    if (vectors == 0)
      continue;
    if (first + parts > 0x7fffffffull || x.dstBytes % 16 != 0 ||
        x.dstBytes / 16 + vectors > 0xffffffffull || x.ciPadded % vec != 0)
      return hipErrorInvalidConfiguration;
    j.firstVector = uint32_t(first), j.dstVector = uint32_t(x.dstBytes / 16);
    j.steps = x.steps, j.blocks = x.blocks;
    j.chunksPerTap = x.ciPadded / vec;
    j.taps = x.taps;
    j.divSteps = makeFastDiv(x.steps), j.divBlocks = makeFastDiv(x.blocks);
    j.divChunks = makeFastDiv(unit == 256 ? x.taps : j.chunksPerTap);
    if (x.select) {
      const IgemmTapSelection &t = *x.select;
      j.selected = 1, j.kW = t.kW, j.kH = t.kH;
      j.countH = t.countH, j.countW = t.countW;
      j.firstD = t.firstD, j.stepD = t.stepD;
      j.firstH = t.firstH, j.stepH = t.stepH;
      j.firstW = t.firstW, j.stepW = t.stepW;
    }
    ++m.count;
    first += (parts + kPackThreads - 1) / kPackThreads * kPackThreads;
    a.total = uint32_t(parts);
  }
  if (m.count == 0)
    return hipSuccess;
  const dim3 grid{uint32_t(first / kPackThreads)}, block{kPackThreads};
  auto go = [&](auto type) {
    using T = decltype(type);
    if (m.count == 1) {
      hipLaunchKernelGGL(packWeightsKernel<T>, grid, block, 0, stream, a,
                         m.job[0]);
    } else {
      // (what a job's rows or blocks times its steps are multiplied by)
      a.total = groups * unit * kPackParts;
      hipLaunchKernelGGL(packManyWeightsKernel<T>, grid, block, 0, stream, a,
                         m);
    }
    return hipGetLastError();
  };
  if (s.elemBytes == 1)
    return go(uint8_t{});
  if (s.elemBytes == 2)
    return go(uint16_t{});
  return go(uint32_t{});
}

} // namespace mxk
