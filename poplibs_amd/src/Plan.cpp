#include "Plan.hpp"
#include "poplar/exceptions.hpp"
#include "poplin/ConvUtil.hpp"
#include "poputil/exceptions.hpp"

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <sstream>
#include <vector>

namespace poplin {

namespace {

std::size_t product(const std::vector<std::size_t> &v) {
  std::size_t p = 1;
  for (auto x : v)
    p *= x;
  return p;
}

mxk::DimTransform toDim(const std::vector<std::size_t> &shape,
                        const ConvParams::InputTransform &t, unsigned d,
                        unsigned transformedSize) {
  return {uint32_t(shape[d]), t.truncationLower[d], t.truncationUpper[d],
          t.dilation[d],      t.paddingLower[d],    t.paddingUpper[d],
          uint32_t(t.flip[d] ? 1 : 0), transformedSize};
}

mxk::GenericDesc makeGenericDesc(const ConvParams &p) {
  mxk::GenericDesc g{};
  g.numDims = uint32_t(p.getNumFieldDims());
  g.batch = uint32_t(p.batchSize);
  g.groups = uint32_t(p.numConvGroups);
  g.inChansPerGroup = uint32_t(p.inputChannelsPerConvGroup);
  g.outChansPerGroup = uint32_t(p.outputChannelsPerConvGroup);
  g.kernelElems = 1;
  g.outElems = uint64_t(p.batchSize) * p.getNumOutputChans();
  for (unsigned d = 0; d != g.numDims; ++d) {
    g.in[d] = toDim(p.inputFieldShape, p.inputTransform, d,
                    p.getTransformedInputSize(d));
    g.kernel[d] = toDim(p.kernelShape, p.kernelTransform, d,
                        p.getTransformedKernelSize(d));
    g.outSize[d] = uint32_t(p.getOutputSize(d));
    g.outTruncLo[d] = p.outputTransform.truncationLower[d];
    g.outStride[d] = p.outputTransform.stride[d];
    g.outPadLo[d] = p.outputTransform.paddingLower[d];
    g.outPadHi[d] = p.outputTransform.paddingUpper[d];
    g.kernelElems *= uint32_t(p.kernelShape[d]);
    g.outElems *= g.outSize[d];
  }
  return g;
}

/// The subset the fast kernels take: up to two field dimensions; input with
/// truncation, dilation and zero padding; kernel with dilation only; output
/// with truncation and stride only.  Written as "row of the dilated input =
/// out*stride + k*dilation - pad; it holds input row r when it equals
/// r*inDil, valid for r inside [lo, hi)".
struct Simple2D {
  bool ok = false;
  std::string why;
  uint32_t inH = 1, inW = 1, outH = 1, outW = 1, kH = 1, kW = 1;
  int32_t padH = 0, padW = 0;
  uint32_t strideH = 1, strideW = 1, dilH = 1, dilW = 1;
  uint32_t loH = 0, hiH = 1, loW = 0, hiW = 1;
  uint32_t inDilH = 1, inDilW = 1;
  // A third, outermost dimension (depth).  One that the window does not
  // slide over in any interesting way (kernel 1, stride 1, nothing padded,
  // truncated or dilated) is folded into the batch instead.
  uint32_t inD = 1, outD = 1, kD = 1;
  int32_t padD = 0;
  uint32_t strideD = 1, dilD = 1, loD = 0, hiD = 1, inDilD = 1;
  std::size_t batch = 0; // the batch size times the folded depth
  // Kernel truncation, padding and flips: the kernel the window applies
  // (kD, kH, kW) is a selection of the taps of the stored one - tap j of it
  // is stored tap first + j * step (step 1, or -1 for a flipped dimension) -
  // and kernel padding only moves the window (folded into pad).  fullK*: the
  // stored extents.
  bool kernelSelected = false;
  uint32_t fullKD = 1, fullKH = 1, fullKW = 1;
  uint32_t selFirstD = 0, selFirstH = 0, selFirstW = 0;
  uint32_t selStepD = 1, selStepH = 1, selStepW = 1; // 1 or uint32_t(-1)
  // Zeros around the output field (outH, outW are the convolution's own).
  uint32_t outPadLoH = 0, outPadHiH = 0, outPadLoW = 0, outPadHiW = 0;
  uint32_t outPadLoD = 0, outPadHiD = 0;
  bool outputPadded() const {
    return outPadLoH || outPadHiH || outPadLoW || outPadHiW || outPadLoD ||
           outPadHiD;
  }
  bool hasDepth() const { return inD != 1 || outD != 1 || kD != 1; }
  bool inputDilated() const {
    return inDilH != 1 || inDilW != 1 || inDilD != 1;
  }
};

Simple2D asSimple2D(const ConvParams &p) {
  Simple2D s;
  const unsigned n = unsigned(p.getNumFieldDims());
  if (n > 3) {
    s.why = "more than three field dimensions";
    return s;
  }
  s.batch = p.batchSize;
  for (unsigned d = 0; d != n; ++d) {
    const auto &it = p.inputTransform, &kt = p.kernelTransform;
    const auto &ot = p.outputTransform;
    if (it.flip[d]) {
      s.why = "input flip";
      return s;
    }
    const bool kernelTransformed =
        kt.truncationLower[d] || kt.truncationUpper[d] || kt.paddingLower[d] ||
        kt.paddingUpper[d] || kt.flip[d];
    if (kt.truncationLower[d] + kt.truncationUpper[d] >= p.kernelShape[d] &&
        kernelTransformed) {
      s.why = "kernel truncated to nothing";
      return s;
    }
    // conv index = o*stride + outTruncLo; padded input = conv + k*dil;
    // dilated input = padded - padLo; input = dilated / inDil + truncLo when
    // that is whole.
    // (kernel padding shifts where the taps sit in the window: the lower
    // one, or - the flip comes last - the upper one of a flipped kernel)
    const int32_t pad =
        int32_t(it.paddingLower[d]) -
        int32_t(it.truncationLower[d] * it.dilation[d]) -
        int32_t(ot.truncationLower[d]) -
        int32_t(kt.flip[d] ? kt.paddingUpper[d] : kt.paddingLower[d]);
    const uint32_t kept = uint32_t(p.kernelShape[d] - kt.truncationLower[d] -
                                   kt.truncationUpper[d]);
    const uint32_t lo = it.truncationLower[d];
    const uint32_t hi = uint32_t(p.inputFieldShape[d]) - it.truncationUpper[d];
    // which of depth, height, width: the innermost dimension is the width
    const unsigned which = d + 3 - n;
    auto pick = [which](auto &dd, auto &hh, auto &ww) -> auto & {
      return which == 0 ? dd : which == 1 ? hh : ww;
    };
    pick(s.inD, s.inH, s.inW) = uint32_t(p.inputFieldShape[d]);
    pick(s.outD, s.outH, s.outW) = uint32_t(
        p.getOutputSize(d) - ot.paddingLower[d] - ot.paddingUpper[d]);
    pick(s.outPadLoD, s.outPadLoH, s.outPadLoW) = ot.paddingLower[d];
    pick(s.outPadHiD, s.outPadHiH, s.outPadHiW) = ot.paddingUpper[d];
    pick(s.kD, s.kH, s.kW) = kept;
    pick(s.fullKD, s.fullKH, s.fullKW) = uint32_t(p.kernelShape[d]);
    pick(s.selFirstD, s.selFirstH, s.selFirstW) =
        kt.flip[d] ? uint32_t(kt.truncationLower[d]) + kept - 1
                   : uint32_t(kt.truncationLower[d]);
    pick(s.selStepD, s.selStepH, s.selStepW) = kt.flip[d] ? ~0u : 1u;
    s.kernelSelected = s.kernelSelected || kernelTransformed;
    pick(s.padD, s.padH, s.padW) = pad;
    pick(s.strideD, s.strideH, s.strideW) = ot.stride[d];
    pick(s.dilD, s.dilH, s.dilW) = kt.dilation[d];
    pick(s.loD, s.loH, s.loW) = lo;
    pick(s.hiD, s.hiH, s.hiW) = hi;
    pick(s.inDilD, s.inDilH, s.inDilW) = it.dilation[d];
  }
  if (s.kD == 1 && s.strideD == 1 && s.padD == 0 && s.loD == 0 &&
      s.hiD == s.inD && s.inDilD == 1 && s.outD == s.inD &&
      s.outPadLoD == 0 && s.outPadHiD == 0) {
    s.batch *= s.inD;
    s.inD = s.outD = s.hiD = 1;
  }
  s.ok = true;
  return s;
}

/// Output tile (height, width) of the depthwise kernel: the input patch of a
/// tile - ((th-1)*stride + (k-1)*dilation + 1 rows, likewise columns, for up
/// to 16 channel vectors of 16 bytes - has to fit 52 KB so that three
/// workgroups share the 160 KB of a CU.  Width first: the candidate (at most
/// 16) that wastes the fewest pixels at the right edge; then the tallest tile
/// that fits.  {0, 0} when not even one pixel fits.
std::pair<unsigned, unsigned> chooseDepthwiseTile(const Simple2D &s,
                                                  std::size_t vecs) {
  const std::size_t vecBlock = std::min<std::size_t>(vecs, 16);
  const std::size_t budget = (52 * 1024) / 16; // 16-byte elements
  auto patch = [](unsigned t, unsigned stride, unsigned k, unsigned dil) {
    return std::size_t(t - 1) * stride + std::size_t(k - 1) * dil + 1;
  };
  for (unsigned maxW = 16; maxW >= 1; maxW /= 2) {
    unsigned bestW = 0;
    std::size_t bestWaste = ~std::size_t(0);
    for (unsigned tw = std::min(maxW, s.outW); tw > maxW / 2; --tw) {
      const std::size_t waste = (s.outW + tw - 1) / tw * tw - s.outW;
      if (waste < bestWaste) {
        bestWaste = waste;
        bestW = tw;
      }
    }
    if (bestW == 0)
      continue;
    const std::size_t pw = patch(bestW, s.strideW, s.kW, s.dilW);
    unsigned bestH = 0;
    for (unsigned th = 1; th <= std::min(16u, s.outH); ++th)
      if (patch(th, s.strideH, s.kH, s.dilH) *
              ((pw * vecBlock + 63) / 64 * 64) <=
          budget) // rows are padded to whole 64-element loads
        bestH = th;
    if (bestH)
      return {bestH, bestW};
  }
  return {0, 0};
}

/// Tile and strip of the LDS-tiled depthwise kernel where a thread forms a
/// strip of neighbouring pixels (mxk::depthwiseStripTakes): such layers cost
/// what their multiply-adds cost, so the tile is the one that keeps most of a
/// workgroup's 256 threads busy - rows x strips x channel vectors close to a
/// multiple of 256, few rows beyond the field's last, strips of seven pixels
/// where the tile's width is a multiple of seven and of four elsewhere
/// (ConvNeXt's 7 x 7 field: two strips of four, 224 threads, against one of
/// seven, 112) - within the LDS two workgroups of a CU can have.
/// Busy share of a workgroup's threads with strips of `px` pixels on a tile.
double stripFill(const mxk::DepthwiseDesc &d, unsigned th, unsigned tw,
                 unsigned px) {
  const unsigned vb = std::min(d.channels / 8, 16u);
  const unsigned strips = (tw + px - 1) / px;
  const double lanes = double(th) * strips * vb;
  return lanes / (std::ceil(lanes / 256.0) * 256.0) * double(tw) /
         (strips * px);
}

/// Strips of seven pixels where the tile's width is a multiple of seven and
/// that keeps at least as many threads busy as strips of four.
unsigned stripPixelsFor(const mxk::DepthwiseDesc &d, unsigned th,
                        unsigned tw) {
  return tw % 7 == 0 && stripFill(d, th, tw, 7) >= stripFill(d, th, tw, 4)
             ? 7
             : 4;
}

void chooseDepthwiseStripTile(mxk::DepthwiseDesc &d) {
  const unsigned vecs = d.channels / 8, vb = std::min(vecs, 16u);
  // (channel blocks of 16 vectors: the last block's share of busy lanes)
  const double chanFill =
      double(vecs) / double((vecs + vb - 1) / vb * vb);
  double best = 0;
  mxk::DepthwiseDesc chosen = d;
  for (unsigned tw = 1; tw <= std::min(16u, d.outW); ++tw)
    for (unsigned th = 1; th <= std::min(32u, d.outH); ++th) {
      mxk::DepthwiseDesc t = d;
      t.tileH = th, t.tileW = tw, t.stripPixels = stripPixelsFor(d, th, tw);
      if (mxk::depthwiseTileLdsBytes(t) > mxk::kDepthwiseTileLdsMost)
        break;
      const double edgeH =
          double(d.outH) / double((d.outH + th - 1) / th * th);
      const double edgeW =
          double(d.outW) / double((d.outW + tw - 1) / tw * tw);
      // (the patch's halo is loaded, not multiplied: a quarter's weight)
      const double halo = double(th) * tw / (double(th + 6) * (tw + 6));
      const double score = stripFill(d, th, tw, t.stripPixels) * edgeH *
                           edgeW * chanFill * (0.75 + 0.25 * halo);
      if (score > best)
        best = score, chosen = t;
    }
  d = chosen;
}

} // namespace

namespace {

// Cost model of the matrix-core kernels, in microseconds, from kernel traces
// and in-kernel cycle stamps on MI355X at the ~2.0 GHz the chip holds under
// MFMA load.  A k-step is 128 bytes of K per tile row.
constexpr double kLaunchUs = 2.0; // dispatch + drain of any kernel

/// Rounds of workgroups a launch makes with `perCU` workgroups per CU: whole
/// ones where one workgroup owns a CU (equal tiles all end together), softer
/// where two share it.
double roundsOf(std::size_t workgroups, std::size_t perCU) {
  const double slots = double(gfx950::numCUs) * double(perCU);
  if (double(workgroups) <= slots)
    return 1.0;
  const double whole = std::ceil(double(workgroups) / slots);
  return perCU == 1 ? whole : std::min(whole, double(workgroups) / slots + 0.5);
}

/// igemmKernel: 1.45 us start-up + 1.5 us epilogue, 0.345 us per k-step of a
/// 128 x 128 tile (0.24 for 128 x 64); further rounds on a CU pay another
/// 1.5 us (nothing overlaps the next workgroup's start-up); two workgroups
/// sharing a CU take 2.1 times one's time between them; K split adds
/// splitPenaltyUs of its `partialBytes` of fp32 tiles.
/// What K split over workgroups adds: the second kernel with its launch, and
/// the fp32 partial tiles' way out and in again at what a stream of that size
/// reaches (N = 32, 14 x 14, 1 x 1, 1024 -> 256 in two parts, 12.8 MB of
/// tiles: 16.4 us where the tiles' k-steps are estimated at 7.7; 7 x 7, 3 x 3,
/// 512 -> 512 in four, 12.8 MB: 18.7 against 11.2; N = 1, 14 x 14, 3 x 3,
/// 256 -> 256 in nine, 1.8 MB: 9.2 against 6.3).
double splitPenaltyUs(std::size_t partialBytes) {
  return 4.5 + 2.0 * double(partialBytes) / 6.4e6;
}

/// What a k-step is: fp16's or fp8's; fp32's (a 128 x 128 k-step of 32 values
/// is 2 048 cycles of MFMAs); fp32's where the taps are looked up in ranges
/// (more than 32 of them, a weight update pass mostly), which the loading
/// threads take as long again for: N = 8, 16 x 16, 3 x 3, 96 -> 96 147 us in
/// 64 k-steps of 128 x 128, 88 in 128 x 64.
enum StepKind { kStep16, kStep32, kStep32Ranges };
StepKind stepKindOf(bool fp32, std::size_t taps) {
  return !fp32 ? kStep16 : taps > 32 ? kStep32Ranges : kStep32;
}

double estimateStreaming(std::size_t workgroups, std::size_t kSteps,
                         std::size_t perCU, unsigned blockN, unsigned splitK,
                         std::size_t partialBytes, StepKind kind) {
  const double rounds = roundsOf(workgroups, perCU);
  const double step = kind == kStep32Ranges ? (blockN == 128 ? 2.1 : 1.2)
                      : kind == kStep32     ? (blockN == 128 ? 1.0 : 0.52)
                                            : (blockN == 128 ? 0.345 : 0.24);
  double tile = 2.95 + step * double(kSteps);
  if (perCU == 1 && rounds > 1)
    tile += 1.5;
  if (perCU == 2)
    tile *= double(workgroups) > double(gfx950::numCUs) ? 2.1 : 1.0;
  return kLaunchUs + rounds * tile +
         (splitK > 1 ? splitPenaltyUs(partialBytes) : 0.0);
}

/// ... nor is it faster than the chip's power lets the matrix cores run, the
/// work on padding counted: 950 TFLOP/s on a plain product in 128 x 128 tiles
/// (4096 x 4096 x 4096), 800 where taps are gathered (N = 64, 56 x 56, 3 x 3
/// stride 2, 256 -> 512: 740), 720 in 128 x 64 tiles (N = 71, 35 x 35, 3 x 3,
/// 624 -> 136: 730); twice that in fp8, whose k-steps hold twice as much.
double streamingPowerUs(std::size_t workgroups, std::size_t kSteps,
                        unsigned blockN, bool oneTap) {
  const double rate = blockN == 64 ? 7.2e8 : oneTap ? 9.5e8 : 8.0e8;
  return double(workgroups) * double(kSteps) * 128.0 * blockN * 64.0 * 2.0 /
         rate;
}

/// igemmWideKernel: 10 us per round around the loop (256 x 256 outputs leave
/// at its end), 1.3 us per k-step of a workgroup, and where all CUs are busy
/// 1.7 us - the chip's power (4096 x 4096 x 4096 119 us, 4096 x 1024 x 4096
/// 38, 2048 x 4096 x 4096 on half the CUs 90, N = 64, 56 x 56, 3 x 3 stride 2,
/// 256 -> 512 in 392 tiles 124); four fifths of it for tiles of 192 channels.
double estimateWide(std::size_t workgroups, std::size_t kSteps,
                    unsigned blockN) {
  const double rounds = roundsOf(workgroups, 1);
  const double step =
      std::max(1.3 * rounds, 1.7 * double(workgroups) / gfx950::numCUs);
  return kLaunchUs + 10.0 * rounds +
         step * double(kSteps) * (blockN == 192 ? 0.8 : 1.0);
}

/// What the estimates of large problems leave out where K is short - a tile's
/// start and its outputs' way out, which one of 256 pixels waits for alone and
/// two of 128 cover for each other: a call with `tiles` of `blockM` x `blockN`,
/// `kSteps` each, and `mb` megabytes of outputs and weights.  Fitted to 700 random layers
/// and products of 4 to 140 GFLOP, within 9 to 16 % (standard deviation).
double fillingUs(unsigned blockM, unsigned blockN, unsigned stages,
                 std::size_t tiles, std::size_t kSteps, double mb) {
  struct Fit {
    double call, round, stepRound, step, byte;
  };
  const Fit f = blockM == 256 ? blockN == 256 ? Fit{3.3, 7.45, 1.04, 1.69, 0.09}
                                              : Fit{2.7, 5.7, 0.87, 1.36, 0.11}
                : blockN == 64  ? Fit{3.0, 0.84, 0.30, 0.34, 0.095}
                : stages == 2   ? Fit{2.9, 0.0, 0.56, 0.45, 0.21}
                                : Fit{1.5, 2.5, 0.36, 0.51, 0.12};
  const double perCU = double(tiles) / double(gfx950::numCUs);
  // (two narrow tiles share a CU: rounds of half a tile each)
  const bool shared = blockM == 128 && (blockN == 64 || stages == 2);
  const double rounds =
      shared ? std::max(1.0, std::ceil(2.0 * perCU) / 2.0) : std::ceil(perCU);
  return f.call + f.round * (shared ? std::max(perCU, 0.5) : rounds) +
         double(kSteps) * std::max(f.stepRound * rounds, f.step * perCU) +
         f.byte * mb;
}

/// A call of igemmFlexKernel and of the kernels it is weighed against, on one
/// scale: `tiles` workgroups of `kSteps` each, megabytes out and in (weights
/// included).  Per call, per round of workgroups, per k-step - of the longest
/// CU, `lone` times that where the chip is not full - and per megabyte.  Fitted
/// to 2 493 random layers and products of 0.15 to 137 GFLOP (fp16; 1 to 128
/// images of 7 to 64 squared, 1 x 1 to 5 x 5, up to 768 channels; products of up
/// to 4096 x 8192 x 8192), all tiles of each: igemmFlexKernel within 10 %
/// (two workgroups to a CU: 17 %), the tile picked by it 1.1 % behind the best;
/// the others within 6 to 14 %.
struct CallFit {
  double call, round, step, lone, ragged, out, in;
};
double callUs(const CallFit &f, bool shared, std::size_t tiles,
              std::size_t kSteps, bool ragged, double outMB, double inMB) {
  const double perCU = double(tiles) / double(gfx950::numCUs);
  // (two to a CU: rounds of half as much each)
  const double rounds = shared ? std::max(1.0, std::ceil(2.0 * perCU) / 2.0)
                               : std::ceil(perCU);
  return f.call + f.round * (shared ? std::max(perCU, 0.5) : rounds) +
         double(kSteps) * std::max(f.lone * rounds, perCU) * f.step *
             (1.0 + (ragged ? f.ragged : 0.0)) +
         f.out * outMB + f.in * inMB;
}
double estimateFlex(unsigned blockM, unsigned blockN, bool shared,
                    std::size_t tiles, std::size_t kSteps, bool ragged,
                    double outMB, double inMB) {
  // (odd multiples of 32 channels load as many rows as the next even one; two
  // stages, and 64 channels under a tall tile, cost a step more)
  const double edge = (blockM + (blockN + 63) / 64 * 64) / 256.0;
  const double area = blockM * blockN / 16384.0;
  const double base = shared ? 0.127 + 0.225 * edge + 0.063 * area
                             : 0.167 + 0.073 * edge + 0.189 * area;
  const double more = shared                             ? 1.0
                      : blockM + blockN >= 416           ? 1.15
                      : blockN == 64 && blockM > 128 ? 1.10
                                                         : 1.0;
  return callUs(shared ? CallFit{3.26, 0.0, base, 1.015, 0.035 * edge / base,
                                 0.25, 0.159}
                       : CallFit{1.75, 2.37 + 0.45 * area, more * base, 0.80,
                                 0.024 * edge / base, 0.129, 0.078},
                shared, tiles, kSteps, ragged, outMB, inMB);
}
/// igemmKernel (patch 0) and the resident patch, K whole.
double estimateBesideFlex(unsigned patch, unsigned blockN, unsigned stages,
                          std::size_t tiles, std::size_t kSteps, bool ragged,
                          double outMB, double inMB) {
  const bool shared = !patch && (blockN == 64 || stages == 2);
  const CallFit f =
      patch == 1     ? CallFit{0.52, 2.98, 0.172, 0.86, 0.0, 0.34, 0.34}
      : patch == 2   ? CallFit{1.74, 1.92, 0.291, 0.97, 0.07, 0.15, 0.104}
      : blockN == 64 ? CallFit{2.58, 0.0, 0.313, 0.91, 0.17, 0.38, 0.083}
      : stages == 2  ? CallFit{2.98, 0.99, 0.492, 0.96, 0.04, 0.095, 0.07}
                     : CallFit{2.02, 1.63, 0.412, 0.89, 0.16, 0.175, 0.09};
  return callUs(f, shared, tiles, kSteps, ragged, outMB, inMB);
}
/// ... and pointwiseKernel.
double pointwiseBesideFlex(double pixels, double co, double macs, double outMB,
                           double inMB, double weightsMB) {
  return std::max(4.9, 4.14 + 0.02 * outMB + 0.083 * inMB +
                           0.112 * weightsMB + 2.51e-9 * macs +
                           7.95e-6 * pixels * std::ceil(co / 64.0));
}
/// Long sums over few outputs (K of 2 000 and more, up to 800 tiles of 128 x 64):
/// a call of igemmFlexKernel with K in `parts`, one round of workgroups of `kSteps`
/// each and the kernel that adds the parts, and of igemmKernel, K whole or in
/// parts.  Fitted to 569 random layers and products of 0.4 to 60 GFLOP, all tiles
/// and up to two numbers of parts each, within 8 % (igemmKernel 6 to 11); the tile
/// picked by it is 1.4 % behind the best.
double estimateFlexParts(unsigned blockM, unsigned blockN,
                         std::size_t workgroups, std::size_t kSteps,
                         std::size_t parts, bool ragged, double partialMB) {
  const double perCU = double(workgroups) / double(gfx950::numCUs);
  const double edge = (blockM + (blockN + 63) / 64 * 64) / 256.0;
  const double area = blockM * blockN / 16384.0;
  const double step = (0.175 + 0.044 * edge + 0.145 * area) *
                          (blockM + blockN >= 416 ? 1.15 : 1.0) +
                      (ragged ? 0.073 * edge : 0.0);
  return 5.9 + 1.03 * area + 0.0049 * blockM +
         double(kSteps) * step * (0.895 + 0.105 * perCU) +
         0.45 * std::min(partialMB, 15.0) +
         0.24 * std::max(partialMB - 15.0, 0.0) + 0.05 * double(parts);
}
double estimateBesideFlexParts(unsigned blockN, std::size_t parts,
                               std::size_t workgroups, std::size_t kSteps,
                               bool ragged, double outMB, double inMB) {
  if (parts == 1)
    return callUs(CallFit{1.44, 0.05, 0.272, 0.94, 0.23, 0.83, 0.18}, true,
                  workgroups, kSteps, ragged, outMB, inMB);
  // (a part's sums are fp32)
  const double partialMB = 2.0 * outMB * double(parts);
  return blockN == 64
             ? callUs(CallFit{4.86, 2.1, 0.282, 0.95, 0.31, 0.52, 0.0}, false,
                      workgroups, kSteps, ragged, partialMB, inMB)
             : callUs(CallFit{1.62, 0.3, 0.351, 1.06, 0.28, 0.59, 0.097}, false,
                      workgroups, kSteps, ragged, partialMB, inMB);
}

/// The same two for up to 128 pixels, one tile of rows, where the weights' way from
/// memory counts beside the products, and rows that start in the middle of a line
/// (`ragged`) cost a k-step more.  Fitted to 855 random products and layers of 4 to
/// 128 pixels with 3 MB to 1.7 GB of weights that no cache holds, igemmFlexKernel
/// within 5 %, igemmKernel 3 to 4.
double besideBytes(double computeUs, double bytesUs) {
  return std::sqrt(std::hypot(computeUs * computeUs, bytesUs * bytesUs));
}
double estimateFlexPartsOfFewRows(unsigned blockM, unsigned blockN,
                                  std::size_t kSteps, std::size_t parts,
                                  double partialMB, double weightsMB) {
  const double area = blockM * blockN / 16384.0;
  return 4.375 +
         besideBytes(double(kSteps) * (0.21 + 0.412 * area),
                     0.151 * weightsMB) +
         0.901 * partialMB + 0.097 * double(parts);
}
double estimateBesideFlexPartsOfFewRows(unsigned blockN, std::size_t parts,
                                        std::size_t workgroups,
                                        std::size_t kSteps, std::size_t rows,
                                        bool ragged, double partialMB,
                                        double weightsMB) {
  struct Fit {
    double call, lone, step, byte, partial, ragged, whole;
  };
  const Fit f =
      blockN == 64
          ? parts == 1 ? Fit{2.926, 0.984, 0.359, 0.222, 0.256, 0.257, 0.113}
                       : Fit{7.241, 1.013, 0.364, 0.192, 0.098, 0.225, 0.101}
      : parts == 1 ? Fit{4.253, 0.98, 0.408, 0.151, 0.389, 0.426, 0.253}
                   : Fit{6.55, 0.941, 0.407, 0.156, 0.673, 0.487, 0.333};
  const double perCU = double(workgroups) / double(gfx950::numCUs);
  const double step =
      f.step + double(rows) / 128.0 * (ragged ? f.ragged : f.whole);
  return f.call +
         besideBytes(double(kSteps) * std::max(f.lone, perCU) * step,
                     f.byte * weightsMB) +
         f.partial * partialMB;
}

/// igemmFlexKernel is taken where it is estimated at less than these shares of
/// what is planned.  Over the layers of the fit, at the share and (in brackets)
/// wherever the estimate is lower at all: tiles of 128 x 128, two to a CU, 1.155
/// times as fast on average (1.17), one round of them 1.0075 (under 1), of 128 x
/// 64 1.013 (1.01), resident patch of 16-pixel blocks 1.13 (1.15), of 32 1.03,
/// pointwise layers 1.014 (1.02, one in seven slower); at the share 7 of 1 400 are
/// slower by more than 3 %, the worst 0.85 times as fast, in brackets 190.  Of
/// 1 105 other layers and products with three calls' tensors in turn, those that
/// the rules below leave aside taken out: 1.25 (484), 1.04 (38), 1.16 (57), 1.30 (96),
/// 1.38 (13), 1.23 (79), tiles of 256 x 192 and 256 x 256 1.19 and 1.14 (338); 13
/// slower by more than 3 %, the worst 0.86.
double flexShare(bool pointwise, unsigned patch, unsigned blockN,
                 unsigned stages) {
  return pointwise ? 0.9 : patch ? 0.82 : blockN == 64 || stages == 4 ? 0.85 : 0.88;
}

/// igemmPatchKernel (mode 1) and igemmPatch16Kernel (mode 2, seven blocks of 16
/// pixels whatever the tile's height): start and end of a workgroup and its
/// k-steps, again for every further round of workgroups on a CU, and the way
/// out of `outMB` megabytes of outputs.  Fitted to 17 000 measurements of 3 800
/// random layers (fp16, 1 to 128 images, fields of 7 to 64, 32 to 768 channels,
/// two to 25 taps; 5 500 in fp8), mode 2 within 10 % (fp8 3 %), mode 1 within 8
/// % and, for tiles of 64, of which two may share a CU, 17 %.
double estimatePatch(std::size_t workgroups, std::size_t kSteps, unsigned mode,
                     unsigned blockM, bool quarter, double outMB) {
  struct Fit {
    double first, step, round, roundStep, byte;
  };
  static constexpr Fit kFits[2][3] = {
      {{1.97, 0.173, 2.92, 0.163, 0.0},
       {2.48, 0.286, 1.88, 0.377, 0.2},
       {1.98, 0.259, 1.99, 0.281, 0.205}},
      {{1.95, 0.154, 2.93, 0.129, 0.0},
       {2.26, 0.280, 1.54, 0.377, 0.17},
       {1.41, 0.283, 1.35, 0.312, 0.18}}};
  const Fit &f = kFits[quarter][mode == 2 ? 2 : blockM == 128 ? 1 : 0];
  return kLaunchUs + f.first + f.step * double(kSteps) +
         (roundsOf(workgroups, 1) - 1.0) *
             (f.round + f.roundStep * double(kSteps)) +
         f.byte * outMB;
}

/// What K split adds to it (the same measurements): the second kernel, and
/// the fp32 partial tiles out and in again, mostly from the caches.
double patchSplitUs(std::size_t partialBytes) {
  return 2.75 + 0.29e-6 * double(partialBytes);
}

/// igemmSmallKernel, by its tile (kIgemmSmallTiles): a workgroup that has a CU
/// to itself takes `first` and `group` for every further group of k-steps its
/// waves go through; where there are more of them than half the CUs, each
/// workgroup adds `tile` + `step` per k-step to its CU's time (times 1 +
/// `window` where a window is worked out).  Fitted to 330 random layers and
/// products of up to 6 GFLOP, and to 150 more in fp32, four tiles each: the
/// tile picked by it is on average within 3 % of the best of the four.
/// Nor is a launch faster than a CU's share of the operands arrives, at 60 KB
/// per us: a product of a few rows, bound by its weights, wants tiles enough
/// for every CU (16 x 4096 x 4096: 256 tiles of 16 x 16 take 7.9 us, 128 of
/// 16 x 32 10.3).
double estimateSmall(const mxk::IgemmDesc &d, int inType) {
  struct Fit {
    double first, group, tile, step, window;
    unsigned stepsPerGroup;
  };
  static constexpr Fit kHalfFits[mxk::kIgemmSmallTiles + 1] = {
      {},
      {0.69, 1.56, 0.123, 0.0246, 0.02, 4},
      {1.04, 2.26, 0.213, 0.0379, 0.0, 4},
      {1.37, 1.45, 0.250, 0.0537, 0.0, 2},
      {2.04, 0.99, 0.661, 0.0337, 0.71, 1}};
  static constexpr Fit kFloatFits[mxk::kIgemmSmallTiles + 1] = {
      {},
      {0.63, 0.73, 0.171, 0.0376, 0.0, 4},
      {0.97, 0.70, 0.329, 0.0652, 0.0, 4},
      {1.61, 2.74, 0.605, 0.0652, 0.0, 2},
      {2.74, 2.48, 0.867, 0.0771, 0.0, 1}};
  const Fit &f = inType == mxk::kFloat ? kFloatFits[d.small]
                                       : kHalfFits[d.small];
  const unsigned eb = inType == mxk::kFloat ? 4 : inType == mxk::kHalf ? 2 : 1;
  const double steps =
      std::ceil(double(d.kH) * d.kW * d.inChansPerGroup * eb / 64.0);
  const double perCU =
      double(mxk::igemmSmallTileCount(d)) / double(gfx950::numCUs);
  const double perWave = std::ceil(steps / mxk::igemmSmallWaves(d, inType));
  const double window =
      d.kH * d.kW > 1 || d.inDilH != 1 || d.inDilW != 1 ? f.window : 0.0;
  const double pixelBlocks =
      std::min(double(mxk::igemmSmallTilePixels(d.small)) / 16.0,
               std::ceil(double(d.batch) * d.outH * d.outW / 16.0));
  const double arriveUs =
      2.6 + (perCU <= 2.0 ? std::ceil(perCU) : perCU) * steps *
                (pixelBlocks + mxk::igemmSmallTileChans(d.small) / 16.0) /
                60.0;
  const double computeUs =
      2.1 + f.first +
      f.group * (std::ceil(perWave / f.stepsPerGroup) - 1.0) *
          (1.0 + 0.5 * window) +
      std::max(0.0, perCU - 0.5) * (f.tile + f.step * steps * (1.0 + window));
  return std::max(arriveUs, computeUs);
}

/// What both of the above miss where tiles come by the thousand, as layers of
/// many pixels and few channels make them: more than 8 tiles of 16 x 16 to a CU
/// and at most 64 k-steps (fp8 and fp32: more than 3 tiles).  The time of a
/// call that is repeated on a stream: a CU turns workgroups over, and each of
/// igemmSmallKernel's adds `tile`, `wave` per wave and `step` per k-step to its
/// CU's time (times 1 + `window` or 1 + `dilated` where the input is looked up
/// so); a single one takes `first` and `group` per further group of its waves'
/// k-steps.  Fitted to 7700 random layers, all four tiles, with a standard
/// deviation of 13 %.  Below kCallUs the host's share of the call hides what
/// the kernel takes.
constexpr double kCallUs = 5.0;
double estimateManySmall(const mxk::IgemmDesc &d, int inType) {
  struct Fit {
    double first, group, start, tile, wave, step, window, dilated, share;
    unsigned stepsPerGroup;
  };
  // fp16, fp32, fp8
  static constexpr Fit kFits[3][mxk::kIgemmSmallTiles + 1] = {
      {{},
       {4.08, 0.92, 3.36, 0.075, 0.018, 0.023, 0.0, 0.14, 0.011, 4},
       {4.69, 1.21, 3.19, 0.032, 0.088, 0.024, 0.0, 0.04, 0.014, 4},
       {4.68, 0.77, 3.38, 0.077, 0.075, 0.040, 0.0, 0.07, 0.023, 2},
       {4.83, 0.64, 3.55, 0.165, 0.114, 0.055, 0.14, 0.33, 0.038, 1}},
      {{},
       {4.80, 1.57, 3.39, 0.102, 0.023, 0.030, 0.09, 0.25, 0.009, 4},
       {4.95, 2.68, 3.41, 0.119, 0.092, 0.044, 0.015, 0.16, 0.019, 4},
       {5.07, 2.41, 3.58, 0.07, 0.115, 0.078, 0.10, 0.24, 0.010, 2},
       {5.39, 2.30, 3.95, 0.126, 0.159, 0.145, 0.057, 0.22, 0.007, 1}},
      {{},
       {4.95, 1.32, 3.43, 0.091, 0.019, 0.028, 0.024, 0.5, 0.006, 4},
       {4.95, 2.58, 3.43, 0.012, 0.138, 0.028, 0.0, 0.5, 0.018, 4},
       {5.01, 1.99, 3.50, 0.024, 0.105, 0.068, 0.0, 0.5, 0.019, 2},
       {5.31, 1.84, 3.97, 0.174, 0.099, 0.117, 0.194, 0.5, 0.018, 1}}};
  const Fit &f = kFits[inType == mxk::kHalf ? 0 : inType == mxk::kFloat ? 1 : 2]
                      [d.small];
  const unsigned eb = inType == mxk::kFloat ? 4 : inType == mxk::kHalf ? 2 : 1;
  const double steps =
      std::ceil(double(d.kH) * d.kW * d.inChansPerGroup * eb / 64.0);
  const double perCU =
      double(mxk::igemmSmallTileCount(d)) / double(gfx950::numCUs);
  const double waves = mxk::igemmSmallWaves(d, inType);
  const double groups =
      std::ceil(std::ceil(steps / waves) / double(f.stepsPerGroup));
  const bool dilated = d.inDilH != 1 || d.inDilW != 1;
  const double lookup = dilated           ? f.dilated
                        : d.kH * d.kW > 1 ? f.window
                                          : 0.0;
  // (a stuffed input under a single tap: most chunks meet none of it)
  const double singleTap = dilated && d.kH * d.kW == 1 ? 1.25 : 1.0;
  return std::max({kCallUs,
                   f.first +
                       f.group * (groups - 1.0) *
                           (1.0 + (dilated ? f.dilated : 0.0)) +
                       f.share * std::min(perCU, 1.0) * steps,
                   f.start + perCU * singleTap *
                                 (f.tile + f.wave * waves +
                                  f.step * steps * (1.0 + lookup))});
}
/// What the host's share of a call and the launch's start add to what
/// estimateSmall and the others count from.
constexpr double kCallOverKernelUs = 1.5;
/// Whether estimateManySmall holds for a layer.
bool manySmallTiles(mxk::IgemmDesc d, int inType) {
  d.small = 1;
  const std::uint64_t tiles = mxk::igemmSmallTileCount(d);
  if (inType != mxk::kHalf)
    return tiles > 3 * gfx950::numCUs;
  return tiles > 8 * gfx950::numCUs &&
         std::uint64_t(d.kH) * d.kW * d.inChansPerGroup * 2 <= 64 * 64;
}
/// ... and igemmKernel's on the same scale: one tile alone, or a CU's tiles one
/// behind the other.  `ragged`: channels that fill no whole k-steps.
struct ManyTiles {
  bool fp32;
  unsigned blockN, stages;
  double aloneUs(double kSteps) const {
    if (blockN == 64)
      return fp32 ? 4.65 + 0.97 * kSteps : 4.8 + 0.19 * kSteps;
    return fp32 ? 5.84 + 1.98 * kSteps : stages == 2 ? 0 : 5.5 + 0.34 * kSteps;
  }
  double startUs() const {
    return blockN == 64 ? (fp32 ? 4.1 : 3.4) : fp32 ? 6.5 : 3.9;
  }
  double tileUs(double kSteps, bool ragged) const {
    if (blockN == 64)
      return fp32 ? 1.4 + (1.05 + 0.05 * ragged) * kSteps
                  : 1.1 + (0.3 + 0.05 * ragged) * kSteps;
    if (stages == 4) // (one round of them: aloneUs)
      return fp32 ? 0.0 : 0.14 * ragged * kSteps;
    return fp32 ? 1.86 + 2.28 * kSteps
                : 1.75 + (0.475 + 0.03 * ragged) * kSteps;
  }
};

} // namespace

namespace {

/// Conv groups to run as one (see mxconv_plan::convGroupsPerGroup), 1 = each
/// by itself.  By the planner's own choice: layers whose groups have fewer
/// input channels than half a 128-byte slice and few output channels - the
/// smallest number of groups that makes a whole slice, where that keeps the
/// fused group within 256 output channels (32 groups of 4 -> 4 channels run
/// as 2 groups of 64 -> 64: 16 times the multiply-adds, on matrix cores that
/// stood idle behind 16-byte vectors half empty and 64-channel tiles with 4
/// channels in them).  A `convGroupsPerGroup` plan constraint is taken where
/// it can be (it divides the groups and the fused channels are whole 16-byte
/// vectors) and means "by itself" elsewhere: the reference accepts values
/// that only its own vertices give a meaning to.
///
/// A weight update pass (its parameters are getWeightUpdateParams of the
/// layer's: batch = the layer's input channels, input channels = its batch)
/// is planned for the layer with that many groups taken as one - the same
/// rule on the layer's channels - and the diagonal blocks of the fused
/// layer's weight deltas are what the pass hands back
/// (mxconv_plan::wuGroupsPerGroup).
unsigned chooseConvGroupsPerGroup(const ConvParams &p,
                                  const ConvOptions &options) {
  const auto &pc = options.planConstraints;
  const bool wu = isWeightUpdatePass(options.pass);
  switch (options.pass) {
  case Pass::NONE:
  case Pass::INFERENCE_FWD:
  case Pass::TRAINING_FWD:
  case Pass::TRAINING_BWD:
  case Pass::TRAINING_WU:
    break;
  default:
    return 1;
  }
  const std::size_t groups = p.numConvGroups;
  const std::size_t ci = wu ? p.batchSize : p.inputChannelsPerConvGroup;
  const std::size_t co = p.outputChannelsPerConvGroup;
  const std::size_t eb = p.inputType.size();
  if (groups < 2 || ci == 0 || co == 0 || (ci == 1 && co == 1) ||
      (!pc.kernel.empty() && pc.kernel != "igemm") || p.batchSize == 0 ||
      p.inputChannelsPerConvGroup == 0)
    return 1;
  auto usable = [&](std::size_t f) {
    return f >= 1 && groups % f == 0 && (f * ci * eb) % 16 == 0;
  };
  if (pc.convGroupsPerGroup != 0)
    return usable(pc.convGroupsPerGroup) ? pc.convGroupsPerGroup : 1u;
  // (one input channel per group with several output channels - a depthwise
  // layer with a channel multiplier - included: 64 groups of 1 -> 2 channels
  // run as one of 64 -> 128)
  if (ci * eb >= 64)
    return 1;
  for (std::size_t f = 2; f <= groups; ++f)
    if (usable(f) && f * ci * eb >= 128)
      return f * co <= 256 ? unsigned(f) : 1u;
  // (too few groups for a whole slice: all of them, where that makes two
  // vectors of channels or more)
  if (usable(groups) && groups * ci * eb >= 32 && groups * co <= 256)
    return unsigned(groups);
  return 1;
}

mxconv_plan makePlanWith(const ConvParams &params,
                         const ConvOptions &optionsIn,
                         unsigned convGroupsPerGroup);

/// fp32 layers: wuWindowKernel's fp32 sibling wherever it takes the layer and
/// nothing names a tile for the pass's own convolution.  Over 14 150 random
/// layers (1 to 64 images of 5 to 64 squared, up to 512 channels and 10 GFLOP)
/// it is 3.8 times as fast (geometric mean), slower for 24 of them.  Those, and
/// 498 of 6 350 of up to 1024 channels and 60 GFLOP, are 3 x 3 layers, all but
/// three of more than 200 channels, most with rows that fill the kernel's units
/// of eight columns to 75 % or less (61 images of 7 x 7 at stride 2, 389 -> 442
/// 108.7 us, the convolution 67.7; 36 of 9 x 9, 699 -> 619 475 against 236).  They
/// stay with the kernel all the same: the convolution adds its pixels in one
/// chain, or a few, and its error against 64 bits was 1.7 to 3.4 times the
/// kernel's for six of them (those two 4.7e-7 against 1.8e-7 and 9.0e-7 against
/// 3.2e-7).
bool floatWindowAsked(const PlanConstraints &pc) {
  return pc.deltaWindow == 1 ||
         (!pc.blockM && !pc.blockN && !pc.blockK && !pc.splitK && !pc.stages &&
          pc.patch < 0 && pc.pointwise < 0 && pc.smallTile < 0);
}

/// The weight deltas of `layer` (channels of a group as the layer has them, in
/// resultCi and resultCo) by wuWindowKernel, where that is named or estimated
/// to be faster than what `plan` has; `fuse`: groups that plan takes as one.
/// Both estimates as they are: of 187 random layers that both kernels take (4 to
/// 64 images of 7 to 64 squared, 24 to 512 channels, 1 x 1 and 3 x 3, up to 40
/// GFLOP) the choice is on average 0.4 % slower than the faster of the two, 0.6 %
/// in total time; this one's times 1.08 1.3 and 1.5 %, 1.04 0.7 and 0.8, 0.96 0.8
/// and 1.4, 0.93 1.2 and 2.1 (over 300 layers wuTapKernel for all 55 %, this one
/// for all 1.8 %).
void windowWeightDeltas(mxconv_plan &plan, const mxk::WuTapDesc &layer,
                        unsigned fuse) {
  const auto &pc = plan.options.planConstraints;
  const int asked = pc.deltaWindow;
  if (asked == 0 || pc.weightDeltas == 0 ||
      (pc.weightDeltas == 1 && asked != 1))
    return;
  mxk::WuTapDesc w = layer;
  w.chunkPixels = 64;
  w.ci = w.resultCi, w.co = w.resultCo;
  double us = mxk::wuWindowChoose(w, gfx950::numCUs);
  if (!w.windowCo && w.elemBytes == 4)
    return;
  if (!w.windowCo) {
    // (channels filled up to whole vectors, in copies, as wuTapKernel's are)
    w = layer;
    w.chunkPixels = 64;
    w.ci = (w.resultCi + 7) / 8 * 8, w.co = (w.resultCo + 7) / 8 * 8;
    us = mxk::wuWindowChoose(w, gfx950::numCUs);
    if (!w.windowCo)
      return;
  }
  auto copiesUs = [](const mxk::WuTapDesc &d) {
    double sum = 0.0;
    if (d.resultCi != d.ci)
      sum += 2.6 + double(d.batch) * d.inH * d.inW * d.groups * d.ci * 0.8e-6;
    if (d.resultCo != d.co)
      sum += 2.6 + double(d.batch) * d.outH * d.outW * d.groups * d.co * 0.8e-6;
    return sum;
  };
  us += copiesUs(w);
  if (asked != 1 && plan.denseWeightUpdate) {
    double otherUs;
    if (plan.denseForward.windowCo) {
      otherUs = plan.windowUs;
    } else {
      otherUs = mxk::wuTapEstimateUs(plan.denseForward, gfx950::numCUs) +
                copiesUs(plan.denseForward);
    }
    // (the diagonal blocks of groups taken as one are a launch of their own)
    if (fuse > 1)
      otherUs += 2.2;
    if (us >= otherUs)
      return;
  }
  plan.denseWeightUpdate = true;
  plan.denseForward = w;
  plan.windowUs = us;
  plan.wuOwnGroups = fuse > 1;
}

/// A weight update pass of fewer than 1024 pixels that was planned for
/// wuTapKernel: back to the pass's own convolution where that is estimated to
/// be faster.  Fitted to 2472 random layers of 1 to 64 images, kernels of up to
/// 49 taps, 1 to 800 channels and up to 32 groups: what is picked by the two
/// estimates is on average 0.4 % slower than the faster of the two; the kernel
/// for all of them would be 2.5 % slower, the convolution takes 2.6 times it.
///  * A batch that is no whole vector is the convolution's padded copy and two
///    rearrangements more; only kernels of 25 taps and more over many poorly
///    filled groups are faster so (3 images of 7 x 7, 7 x 7, 32 groups of 48 ->
///    64 39.1 us, the kernel 52.6; but 4 of 14 x 14, 3 x 3, 32 -> 48 23.8
///    against 9.1, one of 10 x 10, 504 -> 144 25.9 against 10.2).
///  * With whole vectors of images it takes fewer taps to bring it ahead: 8
///    images of 8 x 8, 5 x 5, 256 -> 256 12.3 against 22.7, 3 x 3, 512 -> 256
///    12.5 against 17.8, 3 x 3, 64 -> 64 11.7 against 9.7.
void settleFewPixelWeightDeltas(mxconv_plan &plan) {
  const mxk::WuTapDesc &f = plan.denseForward;
  const std::size_t pixels = std::size_t(f.batch) * f.outH * f.outW;
  if (!plan.denseWeightUpdate || pixels >= 1024 || f.elemBytes == 4 ||
      plan.options.planConstraints.weightDeltas == 1 ||
      plan.options.planConstraints.deltaWindow == 1)
    return;
  plan.denseWeightUpdate = false;
  const mxconv_plan::DetailedEstimate e = plan.detailedEstimate();
  const bool wholeVectors =
      f.batch % (16 / plan.params.inputType.size()) == 0;
  const bool fused = plan.wuGroupsPerGroup > 1;
  const double tensorsMB =
      double(plan.inputBytes() + plan.weightBytes()) * 1e-6;
  const double resultMB = double(plan.outputBytes()) * 1e-6;
  const double partialBytes = double(mxk::wuTapWorkspaceBytes(f));
  const double rounds =
      std::ceil(partialBytes / 65536.0 / double(gfx950::numCUs));
  const double steps = std::ceil(
      double(std::min<std::size_t>(f.chunkPixels, pixels)) / 64.0);
  const double kernelUs =
      f.windowCo ? plan.windowUs :
      std::max(8.9, 6.8 + rounds * (0.6 + 0.52 * steps) +
                        0.12e-6 * partialBytes + 1.5 * resultMB +
                        (fused ? 2.2 + 0.17 * resultMB : 0.0));
  const double blocksUs = fused ? 2.1 + 0.5 * resultMB : 0.0;
  const double convolutionUs =
      wholeVectors
          ? std::max(11.8, 3.9 + 1.39 * e.totalUs() + 1.26 * tensorsMB +
                               blocksUs)
          : std::max(20.0, 11.7 + 1.3 * e.totalUs() + 2.5 * tensorsMB +
                               blocksUs);
  plan.denseWeightUpdate = !e.known || kernelUs <= convolutionUs;
  plan.wuOwnGroups = plan.wuOwnGroups && plan.denseWeightUpdate;
}

} // namespace

mxconv_plan makePlan(const ConvParams &params, const ConvOptions &optionsIn) {
  const unsigned fuse =
      chooseConvGroupsPerGroup(params.canonicalize(), optionsIn);
  if (fuse > 1 && isWeightUpdatePass(optionsIn.pass)) {
    // the weight update pass of the layer with `fuse` groups taken as one
    ConvParams fused = params;
    fused.numConvGroups /= fuse;
    fused.batchSize *= fuse;
    fused.outputChannelsPerConvGroup *= fuse;
    mxconv_plan plan = makePlanWith(fused, optionsIn, 1);
    plan.wuGroupsPerGroup = fuse;
    if (plan.wuOwnTensors) {
      // (wuWindowKernel takes the layer's own groups, as many to a tile as
      // have room in it)
      mxk::WuTapDesc own = plan.wuLayer;
      own.groups *= fuse;
      own.resultCi /= fuse, own.resultCo /= fuse;
      windowWeightDeltas(plan, own, fuse);
    }
    settleFewPixelWeightDeltas(plan);
    return plan;
  }
  if (fuse > 1) {
    // (only the matrix-core kernels run groups as one)
    mxconv_plan plan = makePlanWith(params, optionsIn, fuse);
    if (plan.kernel == mxconv_plan::Kernel::IGEMM)
      return plan;
  }
  mxconv_plan plan = makePlanWith(params, optionsIn, 1);
  settleFewPixelWeightDeltas(plan);
  return plan;
}

namespace {

/// The kernels of LDS halo tiles and of rings of rows (3 x 3 taps, input
/// dilations, other element types; 5 x 5 and 7 x 7 halves where a plan names one
/// of them or `columns` 0).
void chooseDepthwiseTileOrRing(mxk::DepthwiseDesc &d, const PlanConstraints &pc,
                               bool inputDilated, int dwType) {
  // 7 x 7 taps at unit stride: a thread forms a strip of neighbouring
  // pixels, and the tile is chosen to fill the workgroup's 256 threads.
  if (mxk::depthwiseStripTakes(d) && !(pc.tileH || pc.tileW))
    chooseDepthwiseStripTile(d);
  // An explicit tile asks for the LDS-tiled kernel.
  d.dense3x3 = !inputDilated && !(pc.tileH || pc.tileW) &&
               mxk::depthwise3x3Takes(d, dwType);
  // Layers that give every CU a band of at least four output rows go to
  // the persistent kernel with a ring of input rows in LDS: its start-up
  // (seven rows before the first output; 3.5 us for the smallest layer
  // against 2.9 us) wants rows to spread over.  Layers of more channels
  // than the small-workgroup kernel takes (224) always do: the kernel of
  // LDS halo tiles needs 5 to 8 us for the smallest of them.
  if (!inputDilated && !(pc.tileH || pc.tileW) && pc.rowRing != 0) {
    d.cus = gfx950::numCUs;
    const mxk::DepthwiseRowsLaunch l = mxk::depthwiseRowsLaunchShape(d);
    const bool takes = mxk::depthwiseRowsTakes(d, dwType);
    if (pc.rowRing == 1 && !takes)
      throw poplar::invalid_option(
          "planConstraints gfx950 rowRing: that kernel takes 3x3 or 5x5 "
          "taps, stride 1 or 2, channels in vectors of 8, at most 2048 "
          "(5x5: 1224) to a pixel");
    // 5 x 5 taps (25 multiply-adds per output and channel: the vector ALU
    // shares the bound): strips of four columns or more, and at stride 2
    // bands of six rows or more - N = 32, 56 x 56, 144 channels, stride 2
    // 26.0 -> 13.1 us and 14 x 14, 480 channels 14.7 -> 9.3, but 28 x 28,
    // 240 channels, stride 2 8.1 -> 9.3 and 7 x 7, 1152 channels (strips of
    // one column) 10.6 -> 12.6.
    const bool five = d.kH == 5;
    // Layers of less than 6 MB take it with strips of two columns and any
    // band: a tile's patch and its rounds of pixels are a longer chain than
    // the ring's first rows (of 48 such layers, stride 2 but one, all were
    // faster, by 23 % at the median: N = 10, 29 x 29, 40 channels 8.8 ->
    // 5.1, N = 3, 23 x 23, 416 8.1 -> 5.0, N = 37, 9 x 9, 640 7.7 -> 6.4).
    const double bytes = 2.0 * d.batch * d.channels *
                         (double(d.inH) * d.inW + double(d.outH) * d.outW);
    const bool fiveWorth =
        ((l.colsOut >= 4 || l.strips == 1) &&
         (d.strideH == 1 || l.rowsOut >= 6)) ||
        (l.colsOut >= 2 && bytes < 6e6);
    if (takes &&
        (pc.rowRing == 1 ||
         (five ? fiveWorth
               : !d.dense3x3 || (l.workgroups * 2 >= gfx950::numCUs &&
                                 l.rowsOut >= 4))))
      d.dense3x3 = 2;
  } else if (pc.rowRing == 1) {
    throw poplar::invalid_option(
        "planConstraints gfx950 rowRing: the layer is not one the "
        "depthwise 3x3 kernels take");
  }
  if (!inputDilated && (pc.tileH || pc.tileW)) {
    d.tileH = pc.tileH ? pc.tileH : d.tileH;
    d.tileW = pc.tileW ? pc.tileW : d.tileW;
    if (mxk::depthwiseStripTakes(d))
      d.stripPixels = stripPixelsFor(d, d.tileH, d.tileW);
    if (mxk::depthwiseTileLdsBytes(d) >
        (d.stripPixels ? mxk::kDepthwiseTileLdsMost : 64 * 1024))
      throw poplar::invalid_option(
          "planConstraints gfx950 tileH x tileW: the input patch of such a "
          "tile does not fit 64 KB of LDS");
  }
}

mxconv_plan makePlanWith(const ConvParams &params,
                         const ConvOptions &optionsIn,
                         unsigned convGroupsPerGroup) {
  mxconv_plan plan;
  plan.params = params;
  plan.canonical = params.canonicalize(); // validates
  plan.options = optionsIn;
  ConvOptions &options = plan.options;
  // What the kernels are planned for: the canonical parameters, with
  // `convGroupsPerGroup` groups taken as one further down.
  ConvParams planned = plan.canonical;
  const ConvParams &p = planned;

  if (p.getNumFieldDims() > mxk::kMaxDims)
    throw poputil::poplibs_error("At most " + std::to_string(mxk::kMaxDims) +
                                 " field dimensions are supported");

  // validateLayerParams: partials at least as wide as the output; quarter
  // inputs produce half outputs.  This build always accumulates in fp32, which
  // satisfies every partials type the reference would settle on.
  for (poplar::Type *t : {&options.partialsType, &options.interTilePartialsType,
                          &options.interIpuPartialsType})
    if (t->size() < params.outputType.size())
      *t = params.outputType;
  if (params.inputType == poplar::QUARTER && params.outputType != poplar::HALF)
    throw poputil::poplibs_error(
        "When the input type for a convolution is quarter, the output type "
        "must be half, not " +
        params.outputType.toString());
  if (params.outputType == poplar::QUARTER)
    throw poputil::poplibs_error("Unsupported convolution output element type "
                                 "(must be float or half)");

  plan.inputElems = params.batchSize * params.getNumInputChans() *
                    product(params.inputFieldShape);
  plan.outputElems = params.batchSize * params.getNumOutputChans() *
                     product(params.getOutputFieldShape());
  plan.weightElems = params.numConvGroups * params.outputChannelsPerConvGroup *
                     params.inputChannelsPerConvGroup *
                     product(params.kernelShape);
  plan.biasElems = params.getNumOutputChans();
  plan.generic = makeGenericDesc(p);
  plan.zeroConv = isZeroConvolution(p);
  plan.madeForWeightUpdate = isWeightUpdatePass(options.pass);

  using Kernel = mxconv_plan::Kernel;
  using Method = PlanConstraints::Method;
  // The weight update pass of a depthwise layer (getWeightUpdateParams of
  // it): one "image" (the layer's single input channel per group), one output
  // channel per group, the layer's batch as input channels.  Its output field
  // is the layer's kernel, its kernel the layer's output field, its kernel
  // dilation the layer's stride and its stride the layer's kernel dilation.
  {
    const Simple2D w = asSimple2D(p);
    if (isWeightUpdatePass(options.pass) &&
        options.planConstraints.weightDeltas != 0 && w.ok && !w.hasDepth() &&
        !w.outputPadded() && !w.kernelSelected && w.batch == 1 &&
        !plan.zeroConv &&
        !w.inputDilated() && p.batchSize == 1 &&
        p.outputChannelsPerConvGroup == 1 &&
        (params.inputType == poplar::HALF ||
         params.inputType == poplar::FLOAT) &&
        p.numConvGroups % (16 / params.inputType.size()) == 0 &&
        p.numConvGroups * p.inputChannelsPerConvGroup *
                std::size_t(w.inH) * w.inW * params.inputType.size() <
            (1ull << 31)) {
      plan.depthwiseWeightUpdate = true;
      mxk::DepthwiseDesc &f = plan.depthwiseForward;
      f.elemBytes = uint32_t(params.inputType.size());
      f.batch = uint32_t(p.inputChannelsPerConvGroup);
      f.channels = uint32_t(p.numConvGroups);
      f.inH = w.inH, f.inW = w.inW;
      f.outH = w.kH, f.outW = w.kW, f.kH = w.outH, f.kW = w.outW;
      f.padH = w.padH, f.padW = w.padW;
      f.strideH = w.dilH, f.strideW = w.dilW;
      f.dilH = w.strideH, f.dilW = w.strideW;
      f.loH = w.loH, f.hiH = w.hiH, f.loW = w.loW, f.hiW = w.hiW;
      // 3x3 layers that give every CU a band of rows: the persistent kernel
      // with the rows of both tensors in LDS rings (as for the forward pass),
      // where strips of columns are not estimated to be faster
      f.cus = gfx950::numCUs;
      const mxk::DepthwiseRowsLaunch l =
          mxk::depthwiseRowsDeltaLaunchShape(f);
      if (options.planConstraints.rowRing != 0 &&
          params.inputType == poplar::HALF &&
          mxk::depthwiseRowsDeltaTakes(f) &&
          (options.planConstraints.rowRing == 1 ||
           // (strips of fewer than four columns read mostly halo: N = 32,
           // 7 x 7, 960 channels 20.5 us against 13.1)
           (l.workgroups * 2 >= gfx950::numCUs && l.rowsOut >= 4 &&
            (l.colsOut >= 4 || l.strips == 1))))
        f.dense3x3 = 2;
      // Strips of columns for the others from some amount of work on, more of it
      // where channels are few and many slots' sums meet: below, the kernel's
      // longer program and the meeting cost up to 4 us more than they save.  Of
      // 260 layers around the lines (1 to 128 images of 7 to 112 squared, 8 to
      // 1040 channels) the choice is 0.7, 0.9 and 0.9 % behind the faster of the
      // two for 3, 5 and 7 taps a side; with lines at 8e6, 20e6 and 43e6 products
      // 4.4, 3.1 and 1.6 %, at 8e6 and 14e6 whatever the channels 2.2 (5 x 5) and
      // 3.6 % (7 x 7, N = 16, 11 x 11 stride 2, 568 channels 14.4 us, 11.6 so).
      const double products =
          double(f.batch) * f.outH * f.outW * f.channels * f.kH * f.kW;
      const double enough =
          f.kH == 3   ? 1e6 * std::max(1.0, 192.0 / f.channels)
          : f.kH == 5 ? 10e6 * std::max(1.0, 32.0 / f.channels)
                      : 30e6 * std::max(1.0, 16.0 / f.channels);
      const int asked = options.planConstraints.columns;
      const bool takes = params.inputType == poplar::HALF &&
                         options.planConstraints.rowRing != 1 &&
                         mxk::depthwiseColumnDeltasTakes(f);
      if (asked > 0 && !takes)
        throw poplar::invalid_option(
            "planConstraints gfx950 columns: the weight deltas' kernel takes "
            "half tensors, 3x3, 5x5 or 7x7 taps at stride 1 or 2, without "
            "rowRing 1");
      // (Rings whatever the estimates say where the tensors are more than the
      // 256 MB cache in front of HBM holds: both were fitted to smaller ones.  Of
      // 69 layers of 0.26 to 2.7 GB what they picked took 0.79 to 1.42 times the
      // rings' time, 1.02 on average, 170 x 65 x 65, 136 channels 109 us, 77 in
      // rings.)
      const double tensors =
          2.0 * f.batch * f.channels *
          (double(f.inH) * f.inW + double(f.outH) * f.outW);
      const bool ringsKept = f.dense3x3 == 2 && tensors > 256e6;
      if (takes && (asked > 0 ||
                    (asked != 0 && products >= enough && !ringsKept))) {
        // The rings win where a few channels make long strips and the tensors
        // are large (32 x 112 x 112 stride 2, 96 channels 23.3 us against 27.3 in
        // strips; 64 x 56 x 56, 144 27.4 and 30.1; but 32 x 56 x 56, 144 19.2 and
        // 17.2, where the two estimates are 0.1 us apart): every workgroup leaves
        // a tile of all channels, whose sums their columns meet for in LDS (9 x 17
        // x 17, 856 channels 19.8 us, 10.4 in strips; 32 x 14 x 14, 504 16.8 and
        // 10.0; 11 x 56 x 56, 320 18.4 and 14.4).  Of 80 layers that the rings
        // take the choice is 1.0 % behind the best.
        const double ringUs = f.dense3x3 == 2
                                  ? mxk::depthwiseRowsDeltaEstimateUs(f)
                                  : 0.0;
        mxk::DepthwiseDesc c = f;
        mxk::chooseDepthwiseColumnDeltas(c, asked > 0 ? uint32_t(asked) : 0);
        if (asked > 0 || f.dense3x3 != 2 ||
            mxk::depthwiseColumnDeltasEstimateUs(c) <= ringUs) {
          f = c;
          f.dense3x3 = 0;
        }
      }
    }
  }
  // The weight update pass of a dense layer with an undilated kernel and
  // input: batch = the layer's input channels, input channels = its batch,
  // kernel = its output field, output field = its kernel, kernel dilation =
  // its stride.  (Opt out:
  // planConstraints gfx950 kernel names one.)
  {
    const Simple2D w = asSimple2D(p);
    const int asked = options.planConstraints.weightDeltas;
    if (isWeightUpdatePass(options.pass) && asked != 0 && w.ok &&
        !w.hasDepth() && !w.outputPadded() && !w.kernelSelected &&
        !plan.zeroConv && !plan.depthwiseWeightUpdate && !w.inputDilated() &&
        w.batch == p.batchSize && w.strideH == 1 && w.strideW == 1 &&
        (params.inputType == poplar::HALF ||
         (params.inputType == poplar::FLOAT &&
          floatWindowAsked(options.planConstraints))) &&
        (asked == 1 ||
         (options.planConstraints.kernel.empty() &&
          options.planConstraints.method == PlanConstraints::Method::ANY))) {
      const bool half = params.inputType == poplar::HALF;
      mxk::WuTapDesc &f = plan.denseForward;
      f.elemBytes = uint32_t(params.inputType.size());
      f.batch = uint32_t(p.inputChannelsPerConvGroup);
      f.inH = w.inH, f.inW = w.inW;
      f.outH = w.kH, f.outW = w.kW, f.kH = w.outH, f.kW = w.outW;
      f.padH = w.padH, f.padW = w.padW;
      f.strideH = w.dilH, f.strideW = w.dilW; // (the layer's stride)
      f.loH = w.loH, f.hiH = w.hiH, f.loW = w.loW, f.hiW = w.hiW;
      f.groups = uint32_t(p.numConvGroups);
      // (channels that are no whole 16-byte vectors: the kernel gets copies
      // with theirs filled up)
      f.resultCi = uint32_t(p.batchSize);
      f.resultCo = uint32_t(p.outputChannelsPerConvGroup);
      const uint32_t vector = half ? 8 : 1;
      f.ci = (f.resultCi + vector - 1) / vector * vector;
      f.co = (f.resultCo + vector - 1) / vector * vector;
      f.chunkPixels = mxk::wuTapChunkPixels(f, gfx950::numCUs);
      plan.wuOwnTensors = true;
      plan.wuLayer = f;
      // Of 1024 pixels or more: 16 channels and more and, in a grouped layer,
      // a quarter of the kernel's 128 x 128 tile per (group, tap): every group
      // brings its own tiles, and poorly filled ones lose to the pass's own
      // convolution (N = 32, 28 x 28, 3 x 3: 32 groups of 16 -> 16 channels 420 against
      // 117 us, 8 groups of 32 -> 32 78 against 49, 2 groups of 64 -> 64 26
      // against 26.5, 4 groups of 64 -> 64 41 against 34 and 2 such groups on
      // 56 x 56 70 against 52; without groups 16 -> 16 on 56 x 56 ties at
      // 39 us and 32 -> 64 wins with 18 against 25).  What is refused here goes
      // to wuWindowKernel where that takes it, without a comparison: of 12 640
      // random half layers of that kind (2 to 64 groups, or fewer than 16
      // channels on a side) the plan took 0.31 of the convolution's time, and
      // 0.86 at most.
      const std::size_t tileArea = std::size_t((f.ci + 127) / 128 * 128) *
                                   ((f.co + 127) / 128 * 128);
      const bool filled =
          f.groups == 1 || std::size_t(f.ci) * f.co * 4 > tileArea;
      // Of fewer pixels: by estimate, once both are planned
      // (settleFewPixelWeightDeltas).
      const bool worth = std::size_t(f.batch) * f.outH * f.outW < 1024 ||
                         (f.resultCi >= 16 && f.resultCo >= 16 && filled);
      plan.denseWeightUpdate =
          half && (asked == 1 || worth) && mxk::wuTapTakes(f);
      // ... or by the kernel that gathers pixels in registers
      windowWeightDeltas(plan, f, 1);
    }
    if (asked == 1 && isWeightUpdatePass(options.pass) &&
        !plan.denseWeightUpdate && !plan.depthwiseWeightUpdate)
      throw poplar::invalid_option(
          "planConstraints gfx950 weightDeltas: no weight-delta kernel takes "
          "this layer's own tensors (half inputs, nothing dilated, truncated, "
          "padded or flipped on the kernel side)");
    if (options.planConstraints.deltaWindow == 1 &&
        isWeightUpdatePass(options.pass) &&
        !(plan.denseWeightUpdate && plan.denseForward.windowCo))
      throw poplar::invalid_option(
          "planConstraints gfx950 deltaWindow: that kernel takes weightDeltas "
          "1 of half and float layers whose kernel has one or three columns and whose "
          "stride along a row is one or two");
  }
  const auto &pc = options.planConstraints;
  if (convGroupsPerGroup > 1) {
    planned.numConvGroups /= convGroupsPerGroup;
    planned.inputChannelsPerConvGroup *= convGroupsPerGroup;
    planned.outputChannelsPerConvGroup *= convGroupsPerGroup;
  }
  const Simple2D s = asSimple2D(p);
  const bool halfIn = params.inputType == poplar::HALF;
  const bool quarterIn = params.inputType == poplar::QUARTER;
  const bool floatIn = params.inputType == poplar::FLOAT;
  const std::size_t ci = p.inputChannelsPerConvGroup;
  const std::size_t co = p.outputChannelsPerConvGroup;
  // The matrix-core kernel reads whole 16-byte vectors of channels; other
  // channel counts are padded with zeros (input: a copy per launch; weights:
  // when they are packed).
  const std::size_t vecElems = 16 / params.inputType.size();
  const std::size_t ciPadded = (ci + vecElems - 1) / vecElems * vecElems;

  // The matrix-core kernel addresses its input with 32-bit offsets from the
  // first image a tile reads.
  auto inputAddressable = [&] {
    mxk::IgemmDesc g{};
    g.blockM = 128; // (the tiles of 256 pixels ask for themselves)
    g.batch = uint32_t(s.batch), g.groups = uint32_t(p.numConvGroups);
    g.inChansPerGroup = uint32_t(ciPadded);
    g.inD = s.inD, g.inH = s.inH, g.inW = s.inW;
    g.outD = s.outD, g.outH = s.outH, g.outW = s.outW;
    g.padD = s.padD, g.padH = s.padH, g.padW = s.padW;
    return s.batch < (1ull << 31) &&
           mxk::igemmAddressable(
               g, halfIn ? mxk::kHalf : floatIn ? mxk::kFloat : mxk::kQuarter);
  };

  // Which kernels can take this convolution at all?
  std::string igemmWhyNot, dwWhyNot;
  static const char *const tooLittleWork =
      "too little work to pay for a padded copy of the input (channels per "
      "group not a multiple of a 16-byte vector)";
  std::pair<unsigned, unsigned> dwTile{0, 0};
  if (plan.zeroConv)
    igemmWhyNot = dwWhyNot = "all outputs are zero";
  else if (!s.ok)
    igemmWhyNot = dwWhyNot = s.why;
  else {
    if (!(halfIn || quarterIn || floatIn))
      igemmWhyNot = "matrix-core kernel takes float, half or quarter inputs";
    else if (ciPadded != ci && (ci == 0 || (ci == 1 && co == 1)))
      // (one channel per group is vector-ALU work)
      igemmWhyNot = "input channels per group not a multiple of a 16-byte "
                    "vector";
    else if (ciPadded != ci && pc.kernel != "igemm" &&
             2.0 * double(s.batch) * s.outD * s.outH * s.outW * s.kD * s.kH *
                     s.kW * ci * co * p.numConvGroups <
                 double(1u << 22) &&
             // The generic kernel's time is its chain of products, of which a
             // thread has all of an output's: 4 us and 0.09 a product in fp16,
             // 0.075 in fp32, 0.36 in fp8; windows three to five times that.
             // The matrix cores take 6 to 8 with the copy (fp32 8 to 14).  By
             // the work alone, as before: fp16 1 x 1, 263 -> 440 channels, ten
             // pixels 30.6 us, now 6; 5 x 5, 12 -> 6, 4 x 5 x 5 51 -> 8; fp8
             // 1 x 1, 227 -> 6 73 -> 7; of 110 random layers below that line
             // the 61 that leave it are 0.98 to 37 times as fast (3.6 at the
             // geometric mean).
             s.kD * s.kH * s.kW * ci <=
                 (s.kD * s.kH * s.kW > 1 ? 36u : quarterIn ? 8u : 64u))
      igemmWhyNot = tooLittleWork;
    else if (std::size_t(s.outH) * s.strideH + std::size_t(s.kH) * s.dilH +
                     std::size_t(std::abs(s.padH)) >=
                 32768 ||
             std::size_t(s.outW) * s.strideW + std::size_t(s.kW) * s.dilW +
                     std::size_t(std::abs(s.padW)) >=
                 32768)
      igemmWhyNot = "field too large for 16-bit window origins";
    else if (s.hasDepth() &&
             ((s.inputDilated() &&
               !((s.inDilD == 1 || s.strideD == 1) &&
                 (s.inDilH == 1 || s.strideH == 1) &&
                 (s.inDilW == 1 || s.strideW == 1) &&
                 std::size_t(s.inDilD) * s.inDilH * s.inDilW <=
                     mxk::kIgemmMaxFused))))
      igemmWhyNot = "three field dimensions with a dilated input that does "
                    "not come apart into phases";
    else if (s.inputDilated() &&
             (std::size_t(s.inW) * p.getNumInputChans() *
                      params.inputType.size() >=
                  (1u << 24) ||
              s.inDilH >= (1u << 24) || s.inDilW >= (1u << 24)))
      igemmWhyNot = "input rows too long for the arithmetic tap addressing";
    else if (!s.inputDilated() && std::size_t(s.kD) * s.kH * s.kW > 32 &&
             (s.kD > 255 || s.kH > 255 || s.kW > 32767))
      igemmWhyNot = "kernel extent above 255 (32 767 in the last dimension)";
    else if (!inputAddressable() ||
             s.batch * s.outD * s.outH * s.outW >= (1ull << 31) ||
             p.numConvGroups * ((co + 127) / 128 * 128) * s.kD * s.kH * s.kW *
                     (ciPadded + vecElems * 8) * params.inputType.size() >=
                 (1ull << 31))
      igemmWhyNot = "tensor too large for 32-bit buffer addressing";
    if (s.hasDepth())
      dwWhyNot = "three field dimensions";
    else if (s.kernelSelected)
      dwWhyNot = "kernel truncation, padding or flip";
    else if (s.outputPadded())
      dwWhyNot = "output padding";
    else if (quarterIn && s.inputDilated())
      dwWhyNot = "depthwise kernel takes a dilated input as half or float";
    else if (ci != 1 || co != 1)
      dwWhyNot = "not one channel per group";
    else if (p.numConvGroups % vecElems != 0)
      dwWhyNot = "channel count not a multiple of a 16-byte vector";
    else if (std::size_t(s.inH) * s.inW * p.numConvGroups *
                     params.inputType.size() >=
                 (1ull << 30) ||
             std::size_t(s.outH) * s.outW * p.numConvGroups * 4 >=
                 (1ull << 30))
      dwWhyNot = "image too large for 32-bit buffer addressing";
    else if (!s.inputDilated() &&
             (dwTile = chooseDepthwiseTile(s, p.numConvGroups / vecElems))
                     .first == 0)
      dwWhyNot = "input patch of a single output pixel exceeds the LDS budget";

  }

  // Choose.  PopLibs method names map onto the kernels that take their role:
  // AMP -> matrix cores; HMAC / VMAC / SLIC -> vector-ALU direct kernel.
  Kernel chosen = Kernel::GENERIC;
  std::string reason;
  auto require = [&](const std::string &whyNot, const char *what) {
    if (!whyNot.empty())
      throw poplar::invalid_option(
          std::string("planConstraints ask for the ") + what +
          " kernel, which cannot take this convolution: " + whyNot);
  };
  if (pc.kernel == "generic") {
    reason = "forced by planConstraints";
  } else if (pc.kernel == "igemm") {
    require(igemmWhyNot, "igemm");
    chosen = Kernel::IGEMM;
    reason = "forced by planConstraints";
  } else if (pc.kernel == "depthwise") {
    require(dwWhyNot, "depthwise");
    chosen = Kernel::DEPTHWISE;
    reason = "forced by planConstraints";
  } else if (pc.method == Method::AMP && igemmWhyNot.empty()) {
    chosen = Kernel::IGEMM;
    reason = "method AMP -> matrix cores";
  } else if ((pc.method == Method::HMAC || pc.method == Method::VMAC ||
              pc.method == Method::SLIC) &&
             dwWhyNot.empty()) {
    chosen = Kernel::DEPTHWISE;
    reason = "method " + std::string(pc.method == Method::HMAC   ? "HMAC"
                                     : pc.method == Method::VMAC ? "VMAC"
                                                                 : "SLIC") +
             " -> vector-ALU direct kernel";
  } else if (pc.method == Method::HMAC || pc.method == Method::VMAC ||
             pc.method == Method::SLIC || pc.method == Method::OUTER_PRODUCT) {
    reason = "vector-ALU method requested; generic direct kernel";
  } else if (dwWhyNot.empty()) {
    chosen = Kernel::DEPTHWISE;
    reason = "one channel per group: memory-bound, vector-ALU direct kernel";
  } else if (igemmWhyNot.empty()) {
    chosen = Kernel::IGEMM;
    reason = "dense channels: implicit GEMM on the matrix cores";
  } else {
    reason = "generic direct kernel (" + igemmWhyNot + ")";
  }
  // An input of 1 to 4 channels (an image, a waveform): the matrix-core
  // kernel that takes the kW * Ci neighbouring elements under a kernel row in
  // chunks of 8, four to a k-step, instead of padding the channels to a whole
  // vector - no copy of the input, K = 192 instead of 392 for N = 32,
  // 224 x 224, 7 x 7 stride 2, 3 -> 64 (58 -> 19 us).  Layers of too little
  // work for a padded copy take it too: it makes none (one 121 x 121 image,
  // 3 x 3 stride 2, 3 -> 16: 17 us on the generic kernel, 4 on this one).
  {
    mxk::ThinInputDesc &t = plan.thinInput;
    t.batch = uint32_t(s.batch), t.inChans = uint32_t(ci);
    t.outChans = uint32_t(co);
    t.inH = s.inH, t.inW = s.inW, t.outH = s.outH, t.outW = s.outW;
    t.kH = s.kH, t.kW = s.kW, t.padH = s.padH, t.padW = s.padW;
    t.strideH = s.strideH, t.strideW = s.strideW;
    t.loH = s.loH, t.hiH = s.hiH, t.loW = s.loW, t.hiW = s.hiW;
    const bool shapeOk =
        !plan.zeroConv && s.ok && !s.hasDepth() && !s.inputDilated() &&
        !s.kernelSelected && !s.outputPadded() && s.dilH == 1 &&
        s.dilW == 1 && p.numConvGroups == 1 && s.batch < (1ull << 31) &&
        mxk::thinInputTakes(t,
                            halfIn    ? mxk::kHalf
                            : floatIn ? mxk::kFloat
                                      : mxk::kQuarter,
                            params.outputType == poplar::HALF ? mxk::kHalf
                                                              : mxk::kFloat);
    const bool unconstrained =
        pc.kernel.empty() && !pc.blockM && !pc.blockN && !pc.blockK &&
        !pc.splitK && !pc.stages && pc.patch < 1 && pc.pointwise != 1 &&
        (pc.method == Method::ANY || pc.method == Method::AMP);
    if (pc.thinInput == 1 && !shapeOk)
      throw poplar::invalid_option(
          "planConstraints gfx950 thinInput: that kernel takes 2-D "
          "convolutions of half inputs with 1 to 4 channels in one group "
          "(kW * Ci <= 32, at most 28 chunks of 8 elements over the kernel "
          "rows; 16, 32, 48 or 64 output "
          "channels; nothing dilated or flipped, no kernel truncation or "
          "padding, no output padding, no negative padding of the columns)");
    if (shapeOk && pc.thinInput != 0 &&
        (pc.thinInput == 1 ||
         (unconstrained &&
          (chosen == Kernel::IGEMM || igemmWhyNot == tooLittleWork)))) {
      plan.thinInputOn = true;
      mxk::chooseThinInputTiles(t, gfx950::numCUs);
      reason = chosen != Kernel::IGEMM && pc.thinInput == 1
                   ? "forced by planConstraints"
                   : "few input channels: a kernel row's pixels as one k-step "
                     "on the matrix cores";
      chosen = Kernel::IGEMM;
    }
  }
  plan.kernel = chosen;
  plan.reason = reason;

  if (plan.thinInputOn) {
    plan.weightPackedElems = mxk::thinInputPackedElems(plan.thinInput);
    plan.workspaceBytes = 0;
  } else if (chosen == Kernel::IGEMM) {
    mxk::IgemmDesc &g = plan.igemm;
    g.batch = uint32_t(s.batch);
    g.groups = uint32_t(p.numConvGroups);
    g.inChansPerGroup = uint32_t(ciPadded);
    g.inD = s.inD, g.outD = s.outD, g.kD = s.kD, g.padD = s.padD;
    g.strideD = s.strideD, g.dilD = s.dilD, g.loD = s.loD, g.hiD = s.hiD;
    g.outChansPerGroup = uint32_t(co);
    g.inH = s.inH, g.inW = s.inW, g.outH = s.outH, g.outW = s.outW;
    g.kH = s.kH, g.kW = s.kW, g.padH = s.padH, g.padW = s.padW;
    g.strideH = s.strideH, g.strideW = s.strideW;
    g.dilH = s.dilH, g.dilW = s.dilW;
    g.loH = s.loH, g.hiH = s.hiH, g.loW = s.loW, g.hiW = s.hiW;
    g.inDilH = s.inDilH, g.inDilW = s.inDilW;
    if (s.kernelSelected) {
      plan.kernelSelected = true;
      plan.igemmTaps = {s.fullKW,
                        s.selFirstH, s.selStepH, s.kH,
                        s.selFirstW, s.selStepW, s.kW,
                        s.fullKH, s.selFirstD, s.selStepD, s.kD};
    }
    if (s.outputPadded()) {
      // the convolution writes the inside of the padded field; the launch
      // fills the field with zeros (or the bias) first
      g.outFullH = s.outH + s.outPadLoH + s.outPadHiH;
      g.outFullW = s.outW + s.outPadLoW + s.outPadHiW;
      g.outFullD = s.outD + s.outPadLoD + s.outPadHiD;
      g.outOffH = s.outPadLoH, g.outOffW = s.outPadLoW;
      g.outOffD = s.outPadLoD;
      plan.outputPadded = true;
      plan.outputPadLoH = s.outPadLoH, plan.outputPadHiH = s.outPadHiH;
      plan.outputPadLoW = s.outPadLoW, plan.outputPadHiW = s.outPadHiW;
      plan.outputPadLoD = s.outPadLoD, plan.outputPadHiD = s.outPadHiD;
    }
    // Tile shape.  M = batch * outH * outW pixels, N = out channels of one
    // group, K = kH * kW * in channels.  A 128-pixel tile keeps the A
    // fragment reuse high; N is 128 unless the group has at most 64 output
    // channels, when a narrower tile avoids computing padding.
    g.blockM = pc.blockM ? pc.blockM : 128;
    g.blockN = pc.blockN ? pc.blockN : (co <= 64 ? 64 : 128);
    const unsigned stepElems = unsigned(128 / params.inputType.size());
    g.blockK = pc.blockK ? pc.blockK : stepElems;
    // More than 64 output channels on few pixels (the deep 1 x 1 layers at
    // the end of a ResNet): 128 x 128 tiles leave CUs idle or need K split
    // over workgroups with a second kernel; twice as many 128 x 64 tiles, two
    // workgroups to a CU, fill the chip with K whole.  Weighed by the same
    // estimates (N = 32, 14 x 14, 1024 -> 256: 8.9 -> 7.1 us; 7 x 7, 2048 ->
    // 512: 12.8 -> 10.2; but 14 x 14, 1024 -> 512, 392 narrow tiles: 10.2
    // against 12.1, and the estimate keeps the wide tile there).
    const StepKind stepKind =
        stepKindOf(floatIn, std::size_t(s.kD) * s.kH * s.kW);
    bool narrowWhole = false;    // ... chosen: K stays whole
    std::size_t narrowSplit = 0; // ... or narrow tiles with K in this many parts
    if (!pc.blockN && !pc.splitK && !pc.stages && co > 64 &&
        g.blockM == 128) {
      const std::size_t m = s.batch * s.outD * s.outH * s.outW;
      const std::size_t mTiles = (m + 127) / 128;
      const std::size_t kSteps =
          (std::size_t(s.kD) * s.kH * s.kW * ciPadded + stepElems - 1) /
          stepElems;
      const std::size_t wide = mTiles * ((co + 127) / 128) * p.numConvGroups;
      const std::size_t narrow = mTiles * ((co + 63) / 64) * p.numConvGroups;
      std::size_t parts = 1;
      if (wide != 0 && wide * 2 <= gfx950::numCUs && kSteps >= 16)
        parts = std::max<std::size_t>(
            1, std::min<std::size_t>(gfx950::numCUs / wide, kSteps / 4));
      const std::size_t partial =
          parts * m * p.numConvGroups * ((co + 127) / 128 * 128) * 4;
      const double wideUs = std::min(
          estimateStreaming(wide, kSteps, wide > gfx950::numCUs ? 2 : 1, 128,
                            1, 0, stepKind),
          parts > 1 ? estimateStreaming(wide * parts,
                                        (kSteps + parts - 1) / parts, 1, 128,
                                        unsigned(parts), partial, stepKind)
                    : 1e30);
      const double wideWholeUs = estimateStreaming(
          wide, kSteps, wide > gfx950::numCUs ? 2 : 1, 128, 1, 0, stepKind);
      if (estimateStreaming(narrow, kSteps, 2, 64, 1, 0, stepKind) < wideUs) {
        g.blockN = 64, narrowWhole = true;
      } else if (wideUs < wideWholeUs && narrow * 2 <= gfx950::numCUs) {
        // K split wins: then over narrow tiles, in half as many parts of at
        // least 8 k-steps - the same number of workgroups, each with half the
        // weights to fetch per k-step and half the fp32 tile to write, and
        // half the partial tiles in all.  Measured for skinny products and
        // deep layers alike (wide -> narrow, us): 32 x 4096 x 4096 13.3 ->
        // 11.4, 256 x 4096 x 1024 17.5 -> 12.2, 512 x 4096 x 1024 18.1 ->
        // 14.2, N = 8 7 x 7 3 x 3 512 -> 512 15.2 -> 11.0, N = 1 9.9 -> 8.4;
        // level where the rule already chose few parts (N = 32 7 x 7 3 x 3
        // 512 -> 512 19.0 -> 18.6, 14 x 14 stride 2 18.2 -> 18.4).
        const std::size_t narrowParts = std::min<std::size_t>(
            gfx950::numCUs / narrow, kSteps / 8);
        if (narrowParts > 1)
          g.blockN = 64, narrowSplit = narrowParts;
      }
    }
    const bool anyHeight = pc.patch == 2 && g.blockM >= 1 && g.blockM <= 112;
    // (igemm_flex.hip)
    if (pc.flex > 0) {
      g.flex = uint32_t(pc.flex);
      if (!halfIn || pc.patch > 0 || !pc.blockM || !pc.blockN ||
          !mxk::igemmFlexTile(g.blockM, g.blockN, g.flex))
        throw poplar::invalid_option(
            "planConstraints gfx950 flex: that kernel takes half inputs and "
            "outputs in tiles of blockM 128, 192 or 256 and blockN 64 to 256 in "
            "steps of 32 (with flex 2 up to 288 of both together)");
    }
    // (tiles of 256 pixels: igemm_wide.hip)
    const bool wideTile = g.blockM == 256 && pc.patch < 1 && !g.flex;
    if ((g.blockM != 128 && g.blockM != 64 && !anyHeight && !wideTile &&
         !g.flex) ||
        (!wideTile && !g.flex && g.blockN != 64 && g.blockN != 128) ||
        (wideTile && ((g.blockN != 192 && g.blockN != 256) || floatIn)) ||
        g.blockK != stepElems)
      throw poplar::invalid_option(
          "planConstraints gfx950 tile not available: blockM must be 128 (64 "
          "with patch 1, 1 to 112 with patch 2), blockN 64 or 128 (blockM "
          "256, half and quarter: blockN 192 or 256), blockK 32 "
          "(float), 64 (half) or 128 (quarter)");
    const std::size_t k = std::size_t(s.kD) * s.kH * s.kW * ciPadded;
    plan.coPadded = (co + g.blockN - 1) / g.blockN * g.blockN;
    plan.kPadded = (k + g.blockK - 1) / g.blockK * g.blockK;
    plan.weightPackedElems = p.numConvGroups * plan.coPadded * plan.kPadded;
    // Too few output tiles to fill the chip but a long K (a weight update
    // pass, a skinny matrix product): cut K into parts, one workgroup each,
    // as many as bring the grid up to about one workgroup per CU while every
    // part keeps at least 4 k-steps; the fp32 partial tiles go through a
    // workspace (the role of PopLibs' in-channel split with ReduceAdd,
    // lib/poplin/ConvReduce.cpp:316-362).
    {
      const std::size_t m = s.batch * s.outD * s.outH * s.outW;
      const std::size_t tiles = ((m + g.blockM - 1) / g.blockM) *
                                (plan.coPadded / g.blockN) * p.numConvGroups;
      const std::size_t kSteps = plan.kPadded / g.blockK;
      std::size_t parts = 1;
      if (pc.splitK && g.flex)
        parts = pc.splitK;
      else if (g.blockM == 256 || g.flex)
        parts = 1;
      else if (pc.splitK)
        parts = pc.splitK;
      else if (narrowSplit)
        parts = narrowSplit;
      else if (!narrowWhole && tiles != 0 && tiles * 2 <= gfx950::numCUs &&
               kSteps >= 16)
        parts = std::min<std::size_t>(gfx950::numCUs / tiles, kSteps / 4);
      parts = std::max<std::size_t>(1, std::min(parts, kSteps));
      // ... where that is estimated to pay for the partial tiles' round trip
      // and the second kernel: N = 32, 14 x 14, 1 x 1, 1024 -> 256 channels
      // (98 tiles of 16 k-steps) 16.4 us in two parts, 8.9 us whole; 7 x 7,
      // 3 x 3, 512 -> 512 (52 tiles of 72 k-steps) 18.7 in four, 21.1 whole.
      if (!pc.splitK && !narrowSplit && parts > 1 &&
          estimateStreaming(tiles, kSteps, g.blockN == 64 ? 2 : 1, g.blockN, 1,
                            0, stepKind) <=
              estimateStreaming(tiles * parts, (kSteps + parts - 1) / parts,
                                1, g.blockN, unsigned(parts),
                                parts * m * p.numConvGroups * plan.coPadded *
                                    4, stepKind))
        parts = 1;
      const std::size_t chans = p.numConvGroups * co;
      // partial tiles of more than 1 GB are not worth it
      if (parts * m * chans * 4 > (1ull << 30))
        parts = 1;
      // (the sum of the parts is written pixel after pixel: not into a
      // padded output field)
      if (s.outputPadded())
        parts = 1;
      // (three dimensions over a dilated input run as phases only)
      if (s.hasDepth() && s.inputDilated())
        parts = 1;
      g.splitK = uint32_t(parts);
      plan.workspaceBytes = mxk::igemmWorkspaceBytes(g);
      if (ciPadded != ci) {
        plan.paddedInputChans = ciPadded;
        plan.paddedInputOffset = (plan.workspaceBytes + 255) / 256 * 256;
        plan.workspaceBytes = plan.paddedInputOffset +
                              s.batch * s.inD * s.inH * s.inW *
                                  p.numConvGroups * ciPadded *
                                  params.inputType.size();
      }
      // More workgroups than CUs: run the 128-wide tile with two LDS stages
      // instead of four, so that two workgroups share a CU and one's
      // start-up, barriers and epilogue are covered by the other's MFMAs.
      // With one workgroup per CU or fewer the deeper prefetch is worth
      // more.
      g.stages = pc.stages ? pc.stages
                           : (tiles * parts > gfx950::numCUs ? 2 : 4);
      if (g.stages != 2 && g.stages != 4)
        throw poplar::invalid_option(
            "planConstraints gfx950 stages must be 2 or 4");
    }
    // Zero-stuffed input, window moving by single pixels: one ordinary
    // convolution per phase instead of arithmetic on every tap - no MACs on
    // the stuffed zeros, and the fast tap-mask addressing.
    if (s.inputDilated() && g.splitK == 1 &&
        (s.inDilD == 1 || s.strideD == 1) &&
        (s.inDilH == 1 || s.strideH == 1) &&
        (s.inDilW == 1 || s.strideW == 1) &&
        std::size_t(s.inDilD) * s.inDilH * s.inDilW <= mxk::kIgemmMaxFused) {
      // One dimension of one phase.  The window of output o = q * inDil +
      // phase meets real input under kernel tap k when phase - pad + k * dil
      // is a multiple of inDil - taps first, first + step, ... - and reads
      // input q + (phase - pad + k * dil) / inDil there.
      struct Dim {
        uint32_t out = 0, first = 0, step = 1, count = 0;
        int32_t pad = 0;
        uint32_t dil = 1;
        bool dead = false; // no tap ever meets real input: all zeros
      };
      auto dimOf = [](uint32_t phase, uint32_t inDil, uint32_t out,
                      uint32_t k, int32_t pad, uint32_t dil) {
        Dim r;
        r.out = out > phase ? (out - phase + inDil - 1) / inDil : 0;
        int64_t firstOffset = 0;
        for (uint32_t t = 0; t != k; ++t) {
          const int64_t x = int64_t(phase) - pad + int64_t(t) * dil;
          if (x % int64_t(inDil) != 0)
            continue;
          if (r.count == 0)
            r.first = t, firstOffset = x / int64_t(inDil);
          else if (r.count == 1)
            r.step = t - r.first;
          ++r.count;
        }
        if (r.count == 0) {
          r.dead = true, r.count = 1;
          return r;
        }
        r.pad = int32_t(-firstOffset);
        r.dil = r.count > 1 ? r.step * dil / inDil : 1;
        return r;
      };
      std::size_t offset = 0;
      for (uint32_t pd = 0; pd != s.inDilD; ++pd)
      for (uint32_t ph = 0; ph != s.inDilH; ++ph)
        for (uint32_t pw = 0; pw != s.inDilW; ++pw) {
          // a dimension that is not dilated keeps its stride and geometry
          const Dim dd = s.inDilD == 1
                             ? Dim{s.outD, 0, 1, s.kD, s.padD, s.dilD, false}
                             : dimOf(pd, s.inDilD, s.outD, s.kD, s.padD,
                                     s.dilD);
          const Dim h = s.inDilH == 1
                            ? Dim{s.outH, 0, 1, s.kH, s.padH, s.dilH, false}
                            : dimOf(ph, s.inDilH, s.outH, s.kH, s.padH, s.dilH);
          const Dim w = s.inDilW == 1
                            ? Dim{s.outW, 0, 1, s.kW, s.padW, s.dilW, false}
                            : dimOf(pw, s.inDilW, s.outW, s.kW, s.padW, s.dilW);
          if (dd.out == 0 || h.out == 0 || w.out == 0)
            continue;
          mxconv_plan::IgemmPhase phase;
          mxk::IgemmDesc &q = phase.d;
          q = g;
          q.inDilH = q.inDilW = 1;
          q.outH = h.out, q.outW = w.out, q.kH = h.count, q.kW = w.count;
          q.padH = h.pad, q.padW = w.pad, q.dilH = h.dil, q.dilW = w.dil;
          q.outD = dd.out, q.kD = dd.count, q.padD = dd.pad, q.dilD = dd.dil;
          if (s.inDilD != 1)
            q.strideD = 1;
          if (dd.dead)
            q.loD = q.hiD = 0;
          q.outFullD = s.outD + s.outPadLoD + s.outPadHiD;
          q.outStepD = s.inDilD, q.outOffD = pd + s.outPadLoD;
          if (s.inDilH != 1)
            q.strideH = 1;
          if (s.inDilW != 1)
            q.strideW = 1;
          if (h.dead)
            q.loH = q.hiH = 0;
          if (w.dead)
            q.loW = q.hiW = 0;
          q.outFullH = s.outH + s.outPadLoH + s.outPadHiH;
          q.outFullW = s.outW + s.outPadLoW + s.outPadHiW;
          q.outStepH = s.inDilH, q.outStepW = s.inDilW;
          q.outOffH = ph + s.outPadLoH, q.outOffW = pw + s.outPadLoW;
          const bool dead = dd.dead || h.dead || w.dead;
          q.noTaps = dead ? 1 : 0;
          // (tap j of the phase is tap first + j * step of the applied
          // kernel, which is a selection of the stored one itself)
          phase.taps = {s.fullKW,
                        s.selFirstH + s.selStepH * h.first,
                        s.selStepH * h.step,
                        dead ? 0u : h.count,
                        s.selFirstW + s.selStepW * w.first,
                        s.selStepW * w.step,
                        dead ? 0u : w.count,
                        s.fullKH,
                        s.selFirstD + s.selStepD * dd.first,
                        s.selStepD * dd.step,
                        dead ? 0u : dd.count};
          const std::size_t kk =
              std::size_t(q.kD) * q.kH * q.kW * ciPadded;
          phase.kPadded = (kk + g.blockK - 1) / g.blockK * g.blockK;
          phase.packedOffset = offset;
          offset += p.numConvGroups * plan.coPadded * phase.kPadded;
          plan.igemmPhases.push_back(phase);
        }
      // (kernel of more than 32 taps per phase: the ranges take over inside
      // the kernel, as for any convolution)
      plan.weightPackedElems = offset;
      std::size_t phaseTiles = 0;
      for (const auto &ph : plan.igemmPhases)
        phaseTiles += (std::size_t(ph.d.batch) * ph.d.outD * ph.d.outH *
                           ph.d.outW +
                       g.blockM - 1) /
                      g.blockM * (plan.coPadded / g.blockN) * g.groups;
      const uint32_t stages =
          pc.stages ? pc.stages : (phaseTiles > gfx950::numCUs ? 2 : 4);
      for (auto &ph : plan.igemmPhases)
        ph.d.stages = stages;
      g.stages = stages;
    }
    const int inId = halfIn ? mxk::kHalf : floatIn ? mxk::kFloat
                                                   : mxk::kQuarter;
    const int outId =
        params.outputType == poplar::HALF ? mxk::kHalf : mxk::kFloat;
    // (a weight update pass on the layer's own tensors runs none of this)
    if (wideTile && !plan.denseWeightUpdate && !plan.depthwiseWeightUpdate) {
      bool takes = !plan.igemmPhases.empty() ||
                   mxk::igemmWideTakes(g, inId, outId);
      for (const auto &ph : plan.igemmPhases)
        takes = takes && mxk::igemmWideTakes(ph.d, inId, outId);
      if (!takes)
        throw poplar::invalid_option(
            "planConstraints gfx950 blockM 256: that kernel takes kernels of "
            "at most 32 taps on an input of which the images that 256 output "
            "pixels meet stay under 2^31 bytes (a zero-stuffed input where "
            "every phase has taps)");
    }
    if (g.flex) {
      bool takes = !plan.igemmPhases.empty() ||
                   mxk::igemmFlexTakes(g, inId, outId);
      for (const auto &ph : plan.igemmPhases)
        takes = takes && mxk::igemmFlexTakes(ph.d, inId, outId);
      if (!takes || plan.denseWeightUpdate || plan.depthwiseWeightUpdate)
        throw poplar::invalid_option(
            "planConstraints gfx950 flex: that kernel takes half inputs and "
            "outputs, kernels of at most 32 taps, packed weights under 2^31 "
            "bytes and an input of which the images that a tile's pixels meet "
            "do so too");
    }
    // A pointwise convolution with few input channels is bound by HBM, not
    // by the matrix cores: unless the big tile was asked for explicitly, the
    // streaming kernel of small workgroups takes it.
    mxk::PointwiseDesc &pw = plan.pointwise;
    pw.batch = g.batch, pw.pixels = s.outH * s.outW;
    pw.groups = g.groups, pw.inChansPerGroup = g.inChansPerGroup;
    pw.outChansPerGroup = g.outChansPerGroup;
    pw.chanTiles = pc.chanTiles;
    pw.elemBytes = uint32_t(params.inputType.size());
    const bool unitWindow =
        !s.hasDepth() && !s.outputPadded() && !s.kernelSelected &&
        !s.inputDilated() &&
        g.splitK == 1 && s.kH == 1 &&
        s.kW == 1 &&
        s.strideH == 1 && s.strideW == 1 &&
        s.padH == 0 && s.padW == 0 && s.loH == 0 && s.loW == 0 &&
        s.hiH == s.inH && s.hiW == s.inW && s.outH == s.inH &&
        s.outW == s.inW;
    // (The kernel runs 136 to 248 input channels as rows of 256, up to 44 %
    // of them padding it multiplies and makes room for: the big tile is
    // faster on small layers - N = 32, 28 x 28, 144 -> 32: 4.6 against 5.3 us,
    // 192 -> 32: 4.6 against 5.4, 7 x 7, 160 -> 960: 4.8 against 5.5 - and
    // slower on large ones: 56 x 56, 144 -> 24: 11.9 against 8.9.)
    // (fp8 rows count by their bytes: two channels for one of fp16)
    const std::size_t rowChans = ci * params.inputType.size() / 2;
    const bool paddedSmall = rowChans > 128 && rowChans < 256 &&
                             std::size_t(pw.batch) * pw.pixels < 65536 &&
                             pc.pointwise != 1;
    // (fp8 rows of 512 bytes or more: the kernel's MFMAs take 16 channels at
    // a time whatever the type, so deep fp8 layers are the matrix cores' -
    // N = 32, 28 x 28, 512 -> 128: 7.4 us against the big tile's 6.5,
    // N = 64, 14 x 14, 1024 -> 256: 8.5 against 7.8; with 256 channels and
    // fewer it wins, 14 x 14, 256 -> 1024: 10.0 against 12.2, 56 x 56,
    // 256 -> 64: 8.4 against 11.0, 112 x 112, 32 -> 64: 14.6 against 24.1)
    const bool deepQuarter =
        quarterIn && ci >= 512 && pc.pointwise != 1;
    // (A large output in rows of no whole 64-byte pieces, most of what is moved:
    // its pieces are written one by one, whole rows of tiles at a time by the
    // others.  Of 420 layers of such rows those of 150 MB and more took 1.04 to
    // 2.4 times as long here, fp8 81 x 61 x 61, 112 -> 400 167 us, 93 in tiles of
    // 128; smaller ones 0.6 to 1.5 times, 0.85 on average.  Two channel tiles to a
    // workgroup write 128 bytes at a time: of 93 layers of 0.15 to 1.7 GB and more
    // than 128 bytes of input to a pixel those with an odd number of tiles took
    // 1.24 times as long here on average, those with an even one of fp8 0.74 times
    // (128 x 56 x 56, 160 -> 368 74 us, 113 in tiles), of fp16 1.12 times up to 176
    // bytes and 0.95 beyond.)
    const std::size_t inPixel = ci * p.numConvGroups * params.inputType.size();
    const std::size_t outPixel = co * p.numConvGroups * params.outputType.size();
    const bool tilePairs =
        (co + 63) / 64 % 2 == 0 && params.outputType == poplar::HALF;
    const std::size_t mostIn = !tilePairs ? 256 : quarterIn ? 128 : 176;
    const bool largeOddRows =
        outPixel % 64 != 0 && inPixel <= mostIn && outPixel * 2 >= inPixel * 5 &&
        std::size_t(pw.batch) * pw.pixels * outPixel > mxk::kPointwiseOddRows &&
        pc.pointwise != 1;
    plan.pointwiseOn =
        unitWindow && ciPadded == ci && !paddedSmall && !deepQuarter &&
        !largeOddRows &&
        (pc.kernel != "igemm" || pc.pointwise == 1) && pc.pointwise != 0 &&
        pc.patch < 1 && !pc.blockM &&
        !pc.blockN && !pc.blockK &&
        mxk::pointwiseTakes(pw,
                            halfIn    ? mxk::kHalf
                            : floatIn ? mxk::kFloat
                                      : mxk::kQuarter,
                            params.outputType == poplar::HALF ? mxk::kHalf
                                                              : mxk::kFloat);
    if (plan.pointwiseOn)
      plan.weightPackedElems = mxk::pointwisePackedElems(pw);
    else if (pc.pointwise == 1)
      throw poplar::invalid_option(
          "planConstraints gfx950 pointwise: that kernel takes 1x1, unit "
          "stride, unpadded convolutions of half inputs with a multiple of 8 "
          "up to 512 input channels per group (quarter inputs: a multiple of "
          "16 up to 1024), with no other tile constraint");
    else if (pc.chanTiles)
      throw poplar::invalid_option(
          "planConstraints gfx950 chanTiles: the pointwise streaming kernel "
          "does not take this convolution with that many 64-channel tiles "
          "per workgroup (they divide the layer's; at most 4 with up to 64 "
          "input channels, 2 with up to 256, 1 beyond)");
    // Unit stride: the kernel that keeps the tile's input patch in LDS reads
    // every input element once instead of once per tap.
    // (A weight update pass's own convolution, whose channels are its images,
    // takes it for whole 128-byte slices of them only: the streaming kernel
    // writes its result in weight order.)
    if (!plan.pointwiseOn && plan.igemmPhases.empty() &&
        (!isWeightUpdatePass(options.pass) ||
         (!plan.paddedInputChans &&
          ciPadded * params.inputType.size() % 128 == 0)) &&
        (g.splitK == 1 || !pc.splitK || pc.patch == 2) && pc.patch != 0 &&
        !pc.blockN && !pc.blockK && !pc.stages) {
      const std::size_t m = std::size_t(s.batch) * s.outH * s.outW;
      const std::size_t nTiles128 = (co + 127) / 128 * p.numConvGroups;
      const std::size_t slices =
          (ciPadded * params.inputType.size() + 127) / 128;
      // Weigh the tilings by estimated time: the streaming kernel as planned
      // above against this kernel with tiles of 128 and 64 pixels (32-pixel
      // MFMA blocks) and with the layer cut into as many equal tiles of at
      // most 112 pixels as there are CUs (16-pixel blocks).
      struct Tiling {
        uint32_t patch, blockM, parts;
      };
      std::vector<Tiling> tilings;
      auto add = [&](const std::string &name, Tiling tiling,
                     std::size_t workgroups, std::size_t perCU,
                     std::size_t kSteps, double us, double rounds) {
        mxconv_plan::Candidate c;
        c.name = name, c.workgroups = workgroups, c.perCU = perCU;
        c.kSteps = kSteps, c.estimateUs = us, c.rounds = rounds;
        plan.candidates.push_back(c);
        tilings.push_back(tiling);
        return plan.candidates.size() - 1;
      };
      const std::size_t none = ~std::size_t(0);
      auto addPatch = [&](uint32_t mode, uint32_t bm,
                          uint32_t parts) -> std::size_t {
        mxk::IgemmDesc t = g;
        t.patch = mode, t.blockM = bm, t.splitK = parts;
        if (!mxk::igemmPatchTakes(t, inId, outId))
          return none;
        const std::size_t tiles = (m + bm - 1) / bm * nTiles128 * parts;
        const std::size_t steps =
            (slices + parts - 1) / parts * s.kH * s.kW;
        return add("resident patch " + std::to_string(bm) + " x 128" +
                       (mode == 2 ? ", 16-pixel blocks" : "") +
                       (parts > 1 ? ", K in " + std::to_string(parts) +
                                        " parts"
                                  : ""),
                   Tiling{mode, bm, parts}, tiles, 1, steps,
                   estimatePatch(tiles, steps, mode, bm, quarterIn,
                                 1e-6 * double(plan.outputBytes())) +
                       (parts > 1 ? patchSplitUs(mxk::igemmWorkspaceBytes(t))
                                  : 0.0),
                   roundsOf(tiles, 1));
      };
      // Equal tiles, one per CU, in whole 16-pixel MFMA blocks - a tile of 98
      // pixels costs its workgroup the seven blocks a tile of 112 does, and
      // 224 workgroups of 112 are through sooner than 256 of 98 (c2: 8.7
      // against 9.1 us); 112 pixels where that takes several rounds.
      auto equalTiles = [&](std::size_t parts) {
        const std::size_t across =
            gfx950::numCUs / std::max<std::size_t>(1, nTiles128 * parts);
        return across == 0
                   ? 112u
                   : uint32_t(std::min<std::size_t>(
                         112, ((m + across - 1) / across + 15) / 16 * 16));
      };
      const std::size_t streamTiles =
          (m + 127) / 128 * (plan.coPadded / g.blockN) * p.numConvGroups *
          g.splitK;
      const std::size_t streamSteps =
          (plan.kPadded / g.blockK + g.splitK - 1) / g.splitK;
      const std::size_t streamPerCU = g.blockN == 64 || g.stages == 2 ? 2 : 1;
      const std::size_t iStream =
          add("streaming 128 x " + std::to_string(g.blockN) + ", " +
                  std::to_string(g.blockN == 128 ? g.stages : 3) + " stages" +
                  (g.splitK > 1 ? ", K in " + std::to_string(g.splitK) +
                                      " parts"
                                : ""),
              Tiling{0, 128}, streamTiles, streamPerCU, streamSteps,
              estimateStreaming(streamTiles, streamSteps, streamPerCU,
                                g.blockN, g.splitK,
                                mxk::igemmWorkspaceBytes(g), stepKind),
              roundsOf(streamTiles, streamPerCU));
      std::size_t best = iStream;
      if (pc.patch >= 1) {
        // planConstraints: whenever the kernel can, with the tile asked for
        // (K whole unless its parts are named as well)
        const uint32_t parts = pc.patch == 2 && pc.splitK ? pc.splitK : 1;
        const uint32_t bm = pc.blockM         ? pc.blockM
                            : pc.patch == 2 ? equalTiles(parts)
                                            : 128u;
        const std::size_t i = addPatch(uint32_t(pc.patch), bm, parts);
        if (i != none)
          best = i;
      } else if (s.kH * s.kW > 1 && co > 64) {
        // (also against a streaming plan that splits K: the patch kernel's
        // equal tiles fill the chip without the second kernel - N = 32,
        // 14 x 14, 256 -> 256 channels 20.4 -> 12.4 us, N = 8, 28 x 28,
        // 128 -> 128 15.0 -> 7.7)
        std::vector<Tiling> weighed{
            {1, 128, 1}, {1, 64, 1}, {2, equalTiles(1), 1}};
        // ... and K cut along its slices, where the tiles leave CUs idle
        const std::size_t tiles112 = (m + 111) / 112 * nTiles128;
        if (!s.outputPadded() && !isWeightUpdatePass(options.pass))
          for (uint32_t parts = 2;
               parts <= slices && tiles112 * parts <= gfx950::numCUs; ++parts)
            weighed.push_back({2, equalTiles(parts), parts});
        for (Tiling t : weighed) {
          // (a forced tile height picks among the patch tilings only)
          if (pc.blockM && pc.blockM != t.blockM)
            continue;
          const std::size_t i = addPatch(t.patch, t.blockM, t.parts);
          if (i != none && plan.candidates[i].estimateUs <
                               plan.candidates[best].estimateUs)
            best = i;
        }
      }
      plan.candidates[best].chosen = true;
      if (best != iStream) {
        g.patch = tilings[best].patch;
        g.blockM = tilings[best].blockM;
        g.splitK = tilings[best].parts;
        g.blockN = 128;
        g.patchMaxRows = 0;
        g.patchMaxRows = mxk::igemmPatchMaxRows(g);
        plan.workspaceBytes = mxk::igemmWorkspaceBytes(g);
        if (plan.paddedInputChans) {
          const std::size_t copy =
              s.batch * s.inD * s.inH * s.inW * p.numConvGroups * ciPadded *
              params.inputType.size();
          plan.paddedInputOffset = (plan.workspaceBytes + 255) / 256 * 256;
          plan.workspaceBytes = plan.paddedInputOffset + copy;
        }
        plan.coPadded = (co + 127) / 128 * 128;
        plan.weightPackedElems = mxk::igemmPatchPackedElems(g, inId);
      }
    }
    // A problem that fills the chip: tiles of 256 pixels, where they are
    // estimated to be faster than what is chosen so far.
    if (!plan.pointwiseOn && plan.igemmPhases.empty() && !floatIn &&
        pc.kernel.empty() && pc.method == Method::ANY && !pc.blockM &&
        !pc.blockN && !pc.blockK && !pc.splitK && !pc.stages && pc.patch < 0 &&
        pc.pointwise < 0 && !pc.chanTiles && g.splitK == 1 &&
        !isWeightUpdatePass(options.pass)) {
      const std::size_t m = s.batch * s.outD * s.outH * s.outW;
      const std::size_t kSteps = plan.kPadded / g.blockK;
      double planned;
      if (g.patch) {
        planned = 1e30;
        for (const auto &c : plan.candidates)
          if (c.chosen)
            planned = c.estimateUs;
      } else {
        const std::size_t tiles =
            (m + 127) / 128 * (plan.coPadded / g.blockN) * p.numConvGroups;
        planned = std::max(
            estimateStreaming(tiles, kSteps,
                              g.blockN == 64 || g.stages == 2 ? 2 : 1,
                              g.blockN, 1, 0, kStep16),
            kLaunchUs + streamingPowerUs(tiles, kSteps, g.blockN,
                                         s.kD * s.kH * s.kW == 1));
      }
      // ... and by fillingUs: 15 x 57 x 57, 1 x 1, 192 -> 960 51.1 us in tiles
      // of 256 x 256, 36.4 in 128 x 128; 5248 x 192 x 2624 17.0 and 13.3.  83
      // random problems beside those of the fit that took wide tiles without
      // it were 4.8 % slower than in the best tile on average and up to 1.53
      // times; with it 2.5 % and 1.16.  The line: of 213 more around it, on three
      // sets of buffers in turn, the choice is 1.2 % behind the better tile; 1.7
      // with 1.1 in place of 0.97, 3.3 with 1.3, 4.7 in wide tiles all.
      const double mb =
          1e-6 * double(plan.outputBytes() + plan.weightBytes());
      const double narrowUs =
          g.patch ? 1e30
                  : fillingUs(128, g.blockN, g.stages,
                              (m + 127) / 128 * (plan.coPadded / g.blockN) *
                                  p.numConvGroups,
                              kSteps, mb);
      for (uint32_t bn : {192u, 256u}) {
        mxk::IgemmDesc t = g;
        t.patch = 0, t.blockM = 256, t.blockN = bn;
        const std::size_t tiles =
            (m + 255) / 256 * ((co + bn - 1) / bn) * p.numConvGroups;
        const double us = estimateWide(tiles, kSteps, bn);
        if (us >= planned ||
            fillingUs(256, bn, 2, tiles, kSteps, mb) >= 0.97 * narrowUs ||
            p.numConvGroups * ((co + bn - 1) / bn * bn) * plan.kPadded *
                    params.inputType.size() >=
                (1ull << 31) ||
            !mxk::igemmWideTakes(t, inId, outId))
          continue;
        planned = us;
        g = t;
        plan.coPadded = (co + bn - 1) / bn * bn;
        plan.weightPackedElems =
            p.numConvGroups * plan.coPadded * plan.kPadded;
        for (auto &c : plan.candidates)
          c.chosen = false;
        mxconv_plan::Candidate c;
        c.name = "streaming 256 x " + std::to_string(bn);
        c.workgroups = tiles, c.perCU = 1, c.kSteps = kSteps;
        c.estimateUs = us, c.rounds = roundsOf(tiles, 1), c.chosen = true;
        plan.candidates.push_back(c);
      }
    }
    // A problem too small for 128-pixel tiles to fill the chip: small tiles
    // with K split over the waves of a workgroup.
    {
      const std::size_t eb = params.inputType.size();
      auto asSmall = [&](uint32_t tile) {
        mxk::IgemmDesc t = g;
        t.small = tile, t.patch = 0, t.blockM = 128, t.splitK = 1;
        return t;
      };
      // The kernel's chosen so far.  (What its estimate leaves out at this end
      // of the range: the pointwise kernel takes 1.9 us more than launch and
      // bytes, phases run side by side.)
      auto plannedUs = [&] {
        if (plan.igemmPhases.empty()) {
          const mxconv_plan::DetailedEstimate e = plan.detailedEstimate();
          const double us = e.computeUs + e.reductionUs;
          return plan.pointwiseOn ? 0.9 * (us + 1.9) : 0.95 * us;
        }
        std::size_t tiles = 0, steps = 0;
        for (const auto &ph : plan.igemmPhases) {
          tiles += (std::size_t(ph.d.batch) * ph.d.outH * ph.d.outW +
                    g.blockM - 1) /
                   g.blockM * (plan.coPadded / g.blockN) * g.groups;
          steps = std::max(steps, ph.d.noTaps ? 0 : ph.kPadded / g.blockK);
        }
        return 0.95 * estimateStreaming(tiles, steps,
                                        g.blockN == 64 || g.stages == 2 ? 2 : 1,
                                        g.blockN, 1, 0, stepKindOf(floatIn, 0));
      };
      // ... on the scale of estimateManySmall
      auto plannedManyUs = [&] {
        const double pixels = double(s.batch) * s.outH * s.outW;
        const double mb = 1e-6 * double(plan.inputBytes() + plan.outputBytes() +
                                        plan.weightBytes());
        const std::size_t chanBytes = ciPadded * eb;
        if (plan.pointwiseOn) {
          const double macs = pixels * double(ci) * co * p.numConvGroups;
          return std::max(kCallUs, 3.0 + 0.127 * mb + 3.0e-9 * macs +
                                   0.95 * pixels * p.numConvGroups *
                                       double((co + 63) / 64) /
                                       (1024.0 * gfx950::numCUs) +
                                   (chanBytes <= 32 ? 0.127e-6 : 0.0) *
                                       double(plan.outputBytes()));
        }
        if (g.blockM == 256 || g.splitK > 1)
          return plan.detailedEstimate().totalUs() +
                 (g.splitK > 1 ? kCallOverKernelUs : 0.0);
        if (g.patch) {
          const double steps =
              double(s.kH * s.kW) * std::ceil(chanBytes / 128.0);
          const double perCU = std::ceil(pixels / g.blockM) *
                               double((co + 127) / 128 * p.numConvGroups) /
                               gfx950::numCUs;
          return std::max({kCallUs, 4.4 + 0.12 * steps,
                           1.8 + perCU * (3.16 + 0.266 * steps)});
        }
        const ManyTiles tiles{floatIn, g.blockN, g.stages};
        const bool ragged = chanBytes % 128 != 0;
        double alone = 0, turns = 0, dead = 0;
        auto add = [&](double m, double steps, bool noTaps) {
          const double perCU = std::ceil(m / 128.0) *
                               double(plan.coPadded / g.blockN) *
                               double(p.numConvGroups) / gfx950::numCUs;
          if (noTaps) {
            dead += perCU;
            return;
          }
          alone = std::max(alone, tiles.aloneUs(steps));
          turns += perCU * tiles.tileUs(steps, ragged);
        };
        if (plan.igemmPhases.empty())
          add(pixels, double(plan.kPadded / g.blockK), false);
        for (const auto &ph : plan.igemmPhases)
          add(double(ph.d.batch) * ph.d.outH * ph.d.outW,
              double(ph.kPadded / g.blockK), ph.d.noTaps);
        const double us = std::max(
            {kCallUs, alone, tiles.startUs() + turns, 2.5 + 0.085 * mb});
        if (dead > 0) // (outputs that no tap meets)
          return us + 3.5 + dead * (g.blockN == 64 ? 0.6 : 1.25);
        return plan.igemmPhases.empty() ? us : 1.1 * us;
      };
      uint32_t tile = 0;
      if (pc.smallTile > 0) {
        tile = uint32_t(pc.smallTile);
        if (!mxk::igemmSmallTakes(asSmall(tile), inId, outId))
          throw poplar::invalid_option(
              "planConstraints gfx950 smallTile: that kernel takes "
              "convolutions of up to two field dimensions");
      } else if (pc.smallTile != 0 && pc.kernel.empty() &&
                 pc.method == Method::ANY && !pc.blockM && !pc.blockN &&
                 !pc.blockK && !pc.splitK && !pc.stages && pc.patch < 0 &&
                 pc.pointwise < 0 && !pc.chanTiles &&
                 !isWeightUpdatePass(options.pass) &&
                 double(s.batch) * s.outH * s.outW * co * p.numConvGroups *
                         double(k) <=
                     3e9) {
        // The planner's choice: the tile with the lowest estimate, where that
        // is clearly below the kernel's chosen above.  Where many tiles take
        // turns on a CU it is weighed again, by estimates that hold there, and
        // changed for what is clearly faster.  4672 random layers of that kind
        // took 8.7 % more than the best of the five before, up to 2.6 times
        // (N = 31, 87 x 87, 3 x 3, 4 groups of 4 -> 14: 50.5 us, 19.1 without
        // small tiles), and 3.2 % after.
        double best = plannedUs();
        for (uint32_t t = 1; t <= mxk::kIgemmSmallTiles; ++t) {
          const mxk::IgemmDesc d = asSmall(t);
          if (!mxk::igemmSmallTakes(d, inId, outId))
            continue;
          const double us = estimateSmall(d, inId);
          if (us < best)
            best = us, tile = t;
        }
        if (manySmallTiles(asSmall(1), inId)) {
          auto manyUs = [&](uint32_t t) {
            const mxk::IgemmDesc d = asSmall(t);
            if (t == 0)
              return plannedManyUs();
            if (!mxk::igemmSmallTakes(d, inId, outId))
              return 1e30;
            // (large outputs behind a padded copy of the input: 25 to 30 us
            // more for 90 MB in all tiles but the smallest)
            return estimateManySmall(d, inId) +
                   (plan.paddedInputChans && t > 1 &&
                            plan.outputBytes() > (64u << 20)
                        ? 0.25e-6 * double(plan.outputBytes())
                        : 0.0);
          };
          double bestMany = 0.93 * manyUs(tile);
          for (uint32_t t = 0; t <= mxk::kIgemmSmallTiles; ++t)
            if (manyUs(t) < bestMany)
              bestMany = manyUs(t), tile = t;
        }
      }
      if (tile) {
        g = asSmall(tile);
        plan.reason = "few output tiles: small ones, K shared by the waves of "
                      "a workgroup";
        plan.pointwiseOn = false;
        plan.candidates.clear();
        plan.igemmPhases.clear();
        plan.workspaceBytes = 0;
        if (plan.paddedInputChans) {
          plan.paddedInputOffset = 0;
          plan.workspaceBytes = s.batch * s.inH * s.inW * p.numConvGroups *
                                ciPadded * eb;
        }
        plan.weightPackedElems = mxk::igemmSmallPackedElems(g, inId);
      }
    }
    // A tile's height and width closer to the layer's (fp16).
    const bool flexFree =
        halfIn && params.outputType == poplar::HALF && !g.small &&
        pc.flex < 0 && pc.kernel.empty() && pc.method == Method::ANY &&
        !pc.blockM && !pc.blockN && !pc.blockK && !pc.splitK && !pc.stages &&
        pc.patch < 0 && pc.pointwise < 0 && pc.smallTile < 0 &&
        !pc.chanTiles && g.splitK == 1 && !isWeightUpdatePass(options.pass);
    if (flexFree && !plan.igemmPhases.empty() && g.blockN == 128) {
      // The phases of a zero-stuffed input, all with taps, in two rounds or more
      // of tiles of 128 x 128 that their channels fill badly: tiles of 160
      // channels where those cover them in 0.7 of the columns (N = 42, 35 x 35,
      // 3 x 3 stride 2, 136 -> 80 backwards 14.4 -> 10.7 us; 17 such layers 1.39
      // times as fast), of 96 where those do in three quarters (N = 25, 57 x 57,
      // 72 -> 200 20.5 -> 19.4; 55 1.16, the slowest two 0.93).  Single taps,
      // whose other phases write zeros, and fewer tiles gain nothing or lose (N =
      // 38, 27 x 27, 192 -> 56 7.4 -> 8.6).
      std::size_t tiles = 0;
      bool taps = true;
      for (const auto &ph : plan.igemmPhases) {
        tiles += (std::size_t(ph.d.batch) * ph.d.outD * ph.d.outH * ph.d.outW +
                  127) /
                 128 * ((co + 127) / 128) * p.numConvGroups;
        taps = taps && !ph.d.noTaps;
      }
      const std::size_t columns = (co + 127) / 128 * 128;
      const uint32_t bn = (co + 159) / 160 * 160 * 10 <= columns * 7  ? 160
                          : (co + 95) / 96 * 96 * 4 <= columns * 3 ? 96
                                                                    : 0;
      const uint32_t bm = bn == 160 ? 128 : 192;
      bool takes = taps && bn && tiles >= 2 * gfx950::numCUs;
      auto tileOf = [&](mxk::IgemmDesc d) {
        d.blockM = bm, d.blockN = bn, d.flex = 2;
        return d;
      };
      for (const auto &ph : plan.igemmPhases)
        takes = takes && mxk::igemmFlexTakes(tileOf(ph.d), inId, outId);
      if (takes) {
        g = tileOf(g);
        plan.coPadded = (co + bn - 1) / bn * bn;
        std::size_t offset = 0;
        for (auto &ph : plan.igemmPhases) {
          ph.d = tileOf(ph.d);
          ph.packedOffset = offset;
          offset += p.numConvGroups * plan.coPadded * ph.kPadded;
        }
        plan.weightPackedElems = offset;
      }
    } else if (flexFree && plan.igemmPhases.empty() &&
               // (the resident patch and the pointwise kernel fetch a group's
               // channels, a piece of every pixel, once, not once per tap and
               // tile: 190 x 15 x 15, 5 x 5, 4 groups of 720 -> 80 532 us, 799 in
               // tiles of 256 x 96)
               (p.numConvGroups == 1 || (!g.patch && !plan.pointwiseOn)) &&
               // (large pointwise layers of 392 to 512 input channels: their time
               // is their tensors' way, which igemmFlexKernel's estimate, of
               // tensors in the cache, makes too little of.  111 layers of 50 to
               // 200 MB, 136 to 800 channels out, were 0.93 times as fast with
               // three calls' tensors in turn and 0.98 with one's, N = 101, 49 x
               // 14, 408 -> 432 44.4 us and 56.9; 38 larger ones 1.32 and 0.93, 101
               // of 264 to 384 channels in 1.08 and 1.14)
               !(plan.pointwiseOn && k > 384 && co <= 800 &&
                 plan.inputBytes() + plan.outputBytes() > 50000000 &&
                 plan.inputBytes() + plan.outputBytes() < 200000000) &&
               // (below, a call costs its launch, whatever the tile)
               2.0 * double(s.batch) * s.outD * s.outH * s.outW * double(co) *
                       double(k) * p.numConvGroups >=
                   3e8) {
      const std::size_t m = s.batch * s.outD * s.outH * s.outW;
      const std::size_t kSteps = (k + 63) / 64;
      const double inMB = 1e-6 * double(plan.inputBytes());
      const double outMB = 1e-6 * double(plan.outputBytes());
      const double weightsMB = 1e-6 * double(plan.weightBytes());
      const bool ragged = ciPadded % 64 != 0;
      const std::size_t taps = std::size_t(s.kD) * s.kH * s.kW;
      auto tilesOf = [&](std::size_t bm, std::size_t bn) {
        return (m + bm - 1) / bm * ((co + bn - 1) / bn) * p.numConvGroups;
      };
      double planned =
          plan.pointwiseOn
              ? pointwiseBesideFlex(double(m) * p.numConvGroups, double(co),
                                    double(m) * double(co) *
                                        double((k + 127) / 128 * 128) *
                                        p.numConvGroups,
                                    outMB, inMB, weightsMB)
              : estimateBesideFlex(
                    g.patch, g.blockN, g.stages,
                    tilesOf(g.blockM, g.patch ? 128 : g.blockN),
                    g.patch ? (ciPadded + 63) / 64 * taps : kSteps, ragged,
                    outMB, inMB + weightsMB);
      planned *= flexShare(plan.pointwiseOn, g.patch, g.blockN, g.stages);
      mxk::IgemmDesc chosenTile = g;
      // (Tiles of 256 x 192 and 256 x 256 were chosen for their size: this
      // kernel's of the same shape are faster for each of 56 such layers of the
      // fit, 4096 x 4096 x 4096 118 -> 105 us.  Others have to be 8 % below: 2320 x
      // 10111 x 12070 500 us in 256 x 256 tiles of either, 568 in 192 x 192.)
      if (!plan.pointwiseOn && !g.patch && g.blockM == 256) {
        chosenTile.flex = 1;
        planned = 0.92 * estimateFlex(256, g.blockN, false,
                                      tilesOf(256, g.blockN), kSteps, ragged,
                                      outMB, inMB + weightsMB);
        if (!mxk::igemmFlexTakes(chosenTile, inId, outId))
          chosenTile = g, planned = 0.0;
      }
      for (uint32_t bm : {128u, 192u, 256u})
        for (uint32_t bn = 64; bn <= 256; bn += 32)
          for (uint32_t flex : {1u, 2u}) {
            if (!mxk::igemmFlexTile(bm, bn, flex) || (bn > 64 && co <= 64))
              continue;
            // (two workgroups to a CU fetch windows of an input beyond the L2s
            // twice as far apart: seven such layers of 48 to 242 MB 0.96 times as
            // fast as in tiles of 128 x 64, N = 99, 61 x 61, 5 x 5, 328 -> 40 626 us
            // and 834, one to a CU 550; up to 45 MB eight 1.09)
            if (flex == 2 && bn == 64 && taps > 1 && plan.inputBytes() > 45000000)
              continue;
            mxk::IgemmDesc t = g;
            t.patch = 0, t.blockM = bm, t.blockN = bn, t.flex = flex;
            const double us =
                estimateFlex(bm, bn, flex == 2, tilesOf(bm, bn), kSteps, ragged,
                             outMB, inMB + weightsMB);
            if (us >= planned || !mxk::igemmFlexTakes(t, inId, outId))
              continue;
            planned = us, chosenTile = t;
          }
      if (chosenTile.flex) {
        g = chosenTile;
        plan.pointwiseOn = false;
        plan.coPadded = (co + g.blockN - 1) / g.blockN * g.blockN;
        plan.kPadded = (k + 63) / 64 * 64;
        plan.weightPackedElems =
            p.numConvGroups * plan.coPadded * plan.kPadded;
        for (auto &c : plan.candidates)
          c.chosen = false;
        mxconv_plan::Candidate c;
        c.name = "flexible " + std::to_string(g.blockM) + " x " +
                 std::to_string(g.blockN);
        c.workgroups = tilesOf(g.blockM, g.blockN), c.perCU = g.flex;
        c.kSteps = kSteps, c.estimateUs = plan.flexEstimateUs();
        c.rounds = roundsOf(c.workgroups, c.perCU), c.chosen = true;
        plan.candidates.push_back(c);
      }
    }
    // A long sum over few outputs (fp16): large tiles with K in parts, which
    // fetch half as much for a product as tiles of 128 x 64 with K whole.  133 x
    // 4872 x 5488 35.5 -> 20.7 us, 450 x 7416 x 1400 31.8 -> 23.4, N = 8, 31 x 31, 5
    // x 5 stride 2, 376 -> 392 34.7 -> 28.8.  Taken below 0.92 of the estimate for
    // tiles of 128 x 64 with K whole (106 such layers of the fit 1.08 times as fast
    // on average, two slower by more than 3 %), 0.88 with K in parts already (117,
    // 1.02), 0.95 for 128 x 128 in parts (15, 1.10).  Shorter sums do not pay for
    // the second kernel (K of 1 500 to 2 000 0.7 to 0.9 times as fast), nor do 64
    // channels and fewer, whose windows are most of what is fetched (7 x 36 x 36,
    // 5 x 5, 552 -> 40 33.7 -> 44.6).  Of 260 to 800 such tiles, planned in tiles of
    // 128 x 128 that leave the last round of workgroups part empty, 10 % below the
    // estimate for those: 388 x 6240 x 5568 50.9 -> 39.2 us, 10 x 53 x 53, 5 x 5 stride
    // 2, 352 -> 320 57.8 -> 49.0.  There windows with fewer than 192 channels lose (7
    // x 54 x 54, 5 x 5, 704 -> 128 88.9 -> 109), and tiles of 128 x 256 are as often
    // slower as faster than estimated (340 x 7072 x 6816 48.1 -> 54.2).
    if (halfIn && params.outputType == poplar::HALF && !g.small && !g.patch &&
        (g.flex || g.blockM == 128) && !plan.pointwiseOn &&
        plan.igemmPhases.empty() && !s.outputPadded() && pc.flex < 0 &&
        pc.kernel.empty() && pc.method == Method::ANY && !pc.blockM &&
        !pc.blockN && !pc.blockK && !pc.splitK && !pc.stages && pc.patch < 0 &&
        pc.pointwise < 0 && pc.smallTile < 0 && !pc.chanTiles &&
        !isWeightUpdatePass(options.pass) && p.numConvGroups == 1 &&
        co % 4 == 0 && co > 64 && k >= 2000) {
      const std::size_t m = s.batch * s.outD * s.outH * s.outW;
      const std::size_t kSteps = (k + 63) / 64;
      const double outMB = 1e-6 * double(plan.outputBytes());
      const double inMB = 1e-6 * double(plan.inputBytes() + plan.weightBytes());
      const bool ragged = ciPadded % 64 != 0;
      auto tilesOf = [&](std::size_t bm, std::size_t bn) {
        return (m + bm - 1) / bm * ((co + bn - 1) / bn);
      };
      const std::size_t tiles = tilesOf(g.blockM, g.blockN);
      const std::size_t planSteps = (kSteps + g.splitK - 1) / g.splitK;
      double planned =
          g.flex ? 0.9 * estimateFlex(g.blockM, g.blockN, g.flex == 2, tiles,
                                      kSteps, ragged, outMB, inMB)
          : g.splitK == 1 && g.blockN == 128
              ? 0.9 * estimateBesideFlex(0, 128, g.stages, tiles, kSteps, ragged,
                                         outMB, inMB)
                 : (g.splitK == 1       ? 0.92
                    : g.blockN == 64 ? 0.88
                                        : 0.95) *
                       estimateBesideFlexParts(g.blockN, g.splitK,
                                               tiles * g.splitK, planSteps,
                                               ragged, outMB, inMB);
      const std::size_t copy =
          plan.paddedInputChans
              ? s.batch * s.inD * s.inH * s.inW * ciPadded * 2
              : 0;
      // (callers that bring no workspace have 32 MB of it)
      const std::size_t most =
          std::max<std::size_t>(plan.workspaceBytes, std::size_t(32) << 20);
      mxk::IgemmDesc chosenTile = g;
      chosenTile.flex = 0;
      const std::size_t narrow = tilesOf(128, 64);
      // (windows of up to 128 channels on many pixels fetch more than they
      // multiply once the L2s no longer hold their input: of 56 layers of 8 200 to
      // 16 300 pixels whose input is larger than the bounds below 37 were more than
      // 3 % slower in parts, 0.95 times as fast on average, N = 9, 45 x 30, 3 x 3, 616
      // -> 120 33.5 us and 41.9; of 65 with fewer pixels or a smaller input two,
      // 1.13)
      const bool wideWindows =
          s.kD * s.kH * s.kW > 1 && co <= 128 && m > 8200 &&
          plan.inputBytes() > (g.splitK > 1 ? 7500000u : 10500000u);
      if (!wideWindows &&
          (narrow <= 260 ? g.flex || g.splitK > 1 || g.blockN == 64
                         : narrow <= 800 && co >= 192) &&
          2.0 * double(m) * double(co) * double(k) >= 4e8)
        for (uint32_t bm : {128u, 192u, 256u})
          for (uint32_t bn = 64; bn <= 256; bn += 32)
            for (std::size_t slots :
                 {std::size_t(gfx950::numCUs), std::size_t(gfx950::numCUs / 2)}) {
              const std::size_t own = tilesOf(bm, bn);
              const std::size_t parts = std::min(slots / own, kSteps / 3);
              if (parts < 2 || !mxk::igemmFlexTile(bm, bn, 1) ||
                  (narrow > 260 && bm == 128 && bn == 256))
                continue;
              mxk::IgemmDesc t = g;
              t.blockM = bm, t.blockN = bn, t.flex = 1;
              t.splitK = uint32_t(parts);
              const double us = estimateFlexParts(
                  bm, bn, own * parts, (kSteps + parts - 1) / parts, parts,
                  ragged, 2.0 * outMB * double(parts));
              if (us >= planned ||
                  mxk::igemmWorkspaceBytes(t) + copy + 256 > most ||
                  !mxk::igemmFlexTakes(t, inId, outId))
                continue;
              planned = us, chosenTile = t;
            }
      // Up to 128 pixels, where the weights' bytes count, beside tiles of igemmKernel:
      // 3 % below the estimates that know of them.  Of 855 products and layers that
      // the estimates above chose parts for, 217 stay as they were, among them 78 of
      // the 82 that were more than 3 % slower in parts (12 x 2384 x 31152 30.1 ->
      // 37.7 us, 99 x 4096 x 23768 53.0 -> 65.0); all are 1.155 times as fast as
      // without parts, 1.145 with all of them in parts.  Beside these tiles with K
      // whole, from K of 5 000 on: 41 such products 1.16 times as fast, ten of
      // shorter sums 0.97.
      if (chosenTile.flex && m <= 128) {
        const double partialMB = 2.0 * outMB;
        const double weightsMB = 1e-6 * double(plan.weightBytes());
        if (g.flex
                ? k < 5000
                : estimateFlexPartsOfFewRows(
                      chosenTile.blockM, chosenTile.blockN,
                      (kSteps + chosenTile.splitK - 1) / chosenTile.splitK,
                      chosenTile.splitK, partialMB * chosenTile.splitK,
                      weightsMB) >=
                      0.97 * estimateBesideFlexPartsOfFewRows(
                                 g.blockN, g.splitK, tiles * g.splitK,
                                 planSteps, m, ragged, partialMB * g.splitK,
                                 weightsMB))
          chosenTile.flex = 0;
      }
      if (chosenTile.flex) {
        g = chosenTile;
        plan.coPadded = (co + g.blockN - 1) / g.blockN * g.blockN;
        plan.kPadded = kSteps * 64;
        plan.weightPackedElems = plan.coPadded * plan.kPadded;
        plan.workspaceBytes = mxk::igemmWorkspaceBytes(g);
        if (plan.paddedInputChans) {
          plan.paddedInputOffset = (plan.workspaceBytes + 255) / 256 * 256;
          plan.workspaceBytes = plan.paddedInputOffset + copy;
        }
        for (auto &c : plan.candidates)
          c.chosen = false;
        mxconv_plan::Candidate c;
        c.name = "flexible " + std::to_string(g.blockM) + " x " +
                 std::to_string(g.blockN) + ", K in " +
                 std::to_string(g.splitK) + " parts";
        c.workgroups = tilesOf(g.blockM, g.blockN) * g.splitK, c.perCU = 1;
        c.kSteps = (kSteps + g.splitK - 1) / g.splitK;
        c.estimateUs = plan.flexEstimateUs();
        c.rounds = 1.0, c.chosen = true;
        plan.candidates.push_back(c);
      }
    }
    if (!g.patch && !g.flex && g.blockM != 128 && g.blockM != 256)
      throw poplar::invalid_option(
          "planConstraints gfx950 blockM 64 goes with the resident-patch "
          "kernel only");
  } else if (chosen == Kernel::DEPTHWISE) {
    mxk::DepthwiseDesc &d = plan.depthwise;
    d.batch = uint32_t(s.batch);
    d.channels = uint32_t(p.numConvGroups);
    d.inH = s.inH, d.inW = s.inW, d.outH = s.outH, d.outW = s.outW;
    d.kH = s.kH, d.kW = s.kW, d.padH = s.padH, d.padW = s.padW;
    d.strideH = s.strideH, d.strideW = s.strideW;
    d.dilH = s.dilH, d.dilW = s.dilW;
    d.loH = s.loH, d.hiH = s.hiH, d.loW = s.loW, d.hiW = s.hiW;
    d.tileH = dwTile.first, d.tileW = dwTile.second;
    d.inDilH = s.inDilH, d.inDilW = s.inDilW;
    d.elemBytes = uint32_t(params.inputType.size());
    const int dwType = halfIn ? mxk::kHalf
                       : floatIn ? mxk::kFloat
                                 : mxk::kQuarter;
    // 5 x 5 and 7 x 7 taps: strips of columns, wherever no other kernel is
    // named.  Against the kernels below, at their choice, 90 random layers were
    // 1.1 to 7 times as fast; small, large, strided and narrow ones alike, so
    // there is no line to draw.
    const bool columns =
        !plan.depthwiseWeightUpdate && pc.columns != 0 &&
        !(pc.tileH || pc.tileW) && pc.rowRing != 1 &&
        mxk::depthwiseColumnsTakes(d, dwType,
                                   params.outputType == poplar::HALF
                                       ? mxk::kHalf
                                       : mxk::kFloat) &&
        (d.kH != 3 || pc.strips);
    if (pc.strips && !plan.depthwiseWeightUpdate &&
        (!columns || d.kH != 3 || pc.columns > 0))
      throw poplar::invalid_option(
          "planConstraints gfx950 strips: fp16 inputs and 3x3 taps at stride 1 "
          "or 2, without columns, a tile or rowRing named");
    if (columns)
      mxk::chooseDepthwiseColumns(d, pc.strips        ? uint32_t(pc.strips)
                                     : pc.columns > 0 ? uint32_t(pc.columns)
                                                      : 0);
    else if (pc.columns > 0 && !plan.depthwiseWeightUpdate)
      throw poplar::invalid_option(
          "planConstraints gfx950 columns: that kernel takes fp16 inputs, 5x5 "
          "or 7x7 taps at stride 1 or 2, without a tile or rowRing named");
    else
      chooseDepthwiseTileOrRing(d, pc, s.inputDilated(), dwType);
    // 3 x 3 taps that would go to the ring, whose workgroups walk a band each and
    // wait for its first rows: strips of columns where they are estimated at 5 %
    // less, 10 % below 24 MB of tensors, up to 96 MB (43 x 26 x 26, 336 channels 14.4
    // -> 9.2 us).  With three calls' tensors in turn the 337 such layers of 467 with
    // a lower estimate are 1.13 times as fast as in rings, the slowest 0.97; of the
    // 130 left in rings 71 would be more than 3 % slower in strips, with up to 24 MB
    // down to 0.92 (13 x 19 x 19, 912) and with more than 96 - which the cache of 256
    // MB in front of HBM does not hold three times - 0.94 on average (28 x 46 x 46,
    // 424 23.9 -> 29.0).  Strips want their input in that cache: behind a kernel that
    // has just written it they are 1.08 and 1.03 times as fast at stride 1 and 2,
    // from HBM 0.95 and 1.00.
    const double tensorBytes =
        2.0 * double(d.batch) * double(d.channels) *
        (double(d.inH) * d.inW + double(d.outH) * d.outW);
    if (!columns && d.kH == 3 && d.kW == 3 && d.dense3x3 == 2 &&
        !plan.depthwiseWeightUpdate && pc.columns < 0 && pc.rowRing < 0 &&
        params.outputType == poplar::HALF && tensorBytes <= 96e6 &&
        mxk::depthwiseColumnsTakes(d, dwType, mxk::kHalf)) {
      mxk::DepthwiseDesc c = d;
      mxk::chooseDepthwiseColumns(c, 0);
      if (mxk::depthwiseColumnsEstimateUs(c) <
          (tensorBytes < 24e6 ? 0.9 : 0.95) * mxk::depthwiseRowsEstimateUs(d)) {
        d = c;
        d.dense3x3 = 0;
      }
    }
    plan.weightPackedElems = plan.weightElems; // [kH*kW][C]
  } else {
    plan.weightPackedElems = plan.weightElems; // [G][K][Ci][Co]
  }
  if (convGroupsPerGroup > 1 && chosen == Kernel::IGEMM)
    plan.convGroupsPerGroup = convGroupsPerGroup;
  return plan;
}

} // namespace

} // namespace poplin

std::string mxconv_plan::constraintsJson() const {
  std::ostringstream os;
  os << "{";
  if (wuGroupsPerGroup > 1 ||
      (madeForWeightUpdate && canonical.numConvGroups > 1))
    os << "\"convGroupsPerGroup\": " << wuGroupsPerGroup << ", ";
  else if (kernel == Kernel::IGEMM && canonical.numConvGroups > 1)
    os << "\"convGroupsPerGroup\": " << convGroupsPerGroup << ", ";
  os << "\"gfx950\": {";
  switch (kernel) {
  case Kernel::GENERIC:
    os << "\"kernel\": \"generic\"";
    break;
  case Kernel::DEPTHWISE:
    os << "\"kernel\": \"depthwise\", \"rowRing\": "
       << (depthwise.dense3x3 == 2 ? 1 : 0);
    // (an explicit tile names the LDS-tiled kernel)
    if (depthwise.columns)
      os << (depthwise.kH == 3 ? ", \"strips\": " : ", \"columns\": ")
         << depthwise.columns;
    else if (!depthwise.dense3x3 && depthwise.inDilH == 1 && depthwise.inDilW == 1)
      os << ", \"tileH\": " << depthwise.tileH << ", \"tileW\": "
         << depthwise.tileW;
    break;
  case Kernel::IGEMM:
    os << "\"kernel\": \"igemm\"";
    if (thinInputOn) {
      os << ", \"thinInput\": 1";
    } else if (pointwiseOn) {
      os << ", \"pointwise\": 1, \"chanTiles\": "
         << mxk::pointwiseLaunchShape(pointwise, gfx950::numCUs).chansPerWorkgroup / 64;
    } else if (igemm.small) {
      os << ", \"smallTile\": " << igemm.small;
    } else if (igemm.patch) {
      if (igemm.splitK > 1)
        os << ", \"splitK\": " << igemm.splitK;
      os << ", \"pointwise\": 0, \"patch\": " << igemm.patch
         << ", \"blockM\": " << igemm.blockM;
    } else {
      os << ", \"pointwise\": 0, \"patch\": 0, \"blockM\": "
         << igemm.blockM << ", \"blockN\": " << igemm.blockN;
      if (igemm.flex)
        os << ", \"flex\": " << igemm.flex;
      os
         << ", \"blockK\": " << igemm.blockK << ", \"splitK\": "
         << igemm.splitK << ", \"stages\": " << igemm.stages;
    }
    break;
  }
  if (madeForWeightUpdate) {
    os << ", \"weightDeltas\": "
       << (weightUpdateProduct                           ? 2
           : denseWeightUpdate || depthwiseWeightUpdate ? 1
                                                        : 0);
    if (denseWeightUpdate)
      os << ", \"deltaWindow\": " << (denseForward.windowCo ? 1 : 0);
    if (depthwiseWeightUpdate && kernel != Kernel::DEPTHWISE)
      os << ", \"rowRing\": " << (depthwiseForward.dense3x3 == 2 ? 1 : 0);
    if (depthwiseWeightUpdate)
      os << ", \"columns\": " << depthwiseForward.columns;
  }
  os << "}}";
  return os.str();
}

double mxconv_plan::flexEstimateUs() const {
  const mxk::IgemmDesc &g = igemm;
  const std::size_t m = std::size_t(g.batch) * g.outD * g.outH * g.outW;
  const std::size_t workgroups =
      (m + g.blockM - 1) / g.blockM *
      ((g.outChansPerGroup + g.blockN - 1) / g.blockN) * g.groups * g.splitK;
  const std::size_t steps = (kPadded / g.blockK + g.splitK - 1) / g.splitK;
  const bool ragged = g.inChansPerGroup % 64 != 0;
  const double outMB = 1e-6 * double(outputBytes());
  const double weightsMB = 1e-6 * double(weightBytes());
  // (a part's sums are fp32)
  const double partialMB = 2.0 * outMB * double(g.splitK);
  if (g.splitK == 1)
    return poplin::estimateFlex(g.blockM, g.blockN, g.flex == 2, workgroups,
                                steps, ragged, outMB,
                                1e-6 * double(inputBytes()) + weightsMB);
  return m <= 128 ? poplin::estimateFlexPartsOfFewRows(
                        g.blockM, g.blockN, steps, g.splitK, partialMB,
                        weightsMB)
                  : poplin::estimateFlexParts(g.blockM, g.blockN, workgroups,
                                              steps, g.splitK, ragged,
                                              partialMB);
}

mxconv_plan::DetailedEstimate mxconv_plan::detailedEstimate() const {
  // Kernels that stream their tensors once (1x1 with few channels, depthwise,
  // fills) run at about 6.4 TB/s behind the launch: 64 MB in 11.6 us and
  // 96 MB in 17.9 us measured.
  constexpr double kStreamBytesPerUs = 6.4e6;
  auto streamed = [&](std::size_t bytes) {
    return poplin::kLaunchUs + double(bytes) / kStreamBytesPerUs;
  };
  auto spread = [](DetailedEstimate &e, std::size_t workgroups,
                   std::size_t perCU) {
    const std::size_t slots = std::size_t(gfx950::numCUs) * perCU;
    e.parallelSplit = std::max<std::size_t>(1, std::min(workgroups, slots));
    e.serialSplit =
        std::max<std::size_t>(1, (workgroups + slots - 1) / slots);
  };
  DetailedEstimate e;
  if (zeroConv) {
    e.computeUs = streamed(outputBytes());
    return e;
  }
  // A weight update pass that runs on the layer's own tensors: what those
  // kernels were measured at.  Matrix-core kernel + ordered sum, two
  // launches, about 350 TFLOP/s of the dense count while the loop waits for
  // its loads (N = 32, 28 x 28, 128 -> 128, 3 x 3: 24.5 us, of which the sum
  // of the chunks' 16.8 MB of fp32 tiles 5.2); depthwise rows + the sum of
  // the workgroups' tiles (4.5 us) behind one pass over both tensors (N = 32,
  // 112 x 112, 96 channels, stride 2: 20.4 us).
  if (weightUpdateProduct) {
    // the product as planned, behind the deltas' transpose and the packing
    // of the activations (each read once and written once)
    DetailedEstimate e = weightUpdateProduct->detailedEstimate();
    if (e.known) {
      e.rearrangementBytes += weightUpdateProduct->inputBytes() +
                              weightUpdateProduct->weightPackedBytes();
      e.rearrangementUs +=
          streamed(2 * weightUpdateProduct->inputBytes()) +
          streamed(2 * weightUpdateProduct->weightPackedBytes());
    }
    return e;
  }
  if (denseWeightUpdate) {
    const auto &f = denseForward;
    const double flops = 2.0 * f.batch * f.outH * f.outW * f.groups * f.ci *
                         f.co * f.kH * f.kW;
    const double all = 2 * poplin::kLaunchUs + flops / 3.5e8;
    if (f.resultCi != f.ci || f.resultCo != f.co) {
      // (a read and a write of the tensors that are copied)
      const std::size_t m = std::size_t(f.batch) * f.groups;
      if (f.resultCi != f.ci)
        e.rearrangementBytes += m * f.inH * f.inW * f.ci * 2;
      if (f.resultCo != f.co)
        e.rearrangementBytes += m * f.outH * f.outW * f.co * 2;
      e.rearrangementUs += streamed(2 * e.rearrangementBytes);
    }
    if (f.windowCo) {
      e.reductionBytes = mxk::wuWindowWorkspaceBytes(f);
      e.reductionUs =
          e.reductionBytes
              ? std::min(windowUs / 2, 2.7 + streamed(e.reductionBytes))
              : 0.0;
      e.computeUs =
          std::max(0.0, windowUs - e.reductionUs - e.rearrangementUs);
      spread(e, mxk::wuWindowWorkgroups(f), 1);
      return e;
    }
    e.reductionBytes = mxk::wuTapWorkspaceBytes(f);
    e.reductionUs = std::min(all / 2, streamed(e.reductionBytes));
    e.computeUs = all - e.reductionUs;
    const std::size_t m = std::size_t(f.batch) * f.outH * f.outW;
    spread(e,
           std::size_t(f.groups) * f.kH * f.kW * ((f.ci + 127) / 128) *
               ((f.co + 127) / 128) * ((m + f.chunkPixels - 1) / f.chunkPixels),
           1);
    return e;
  }
  if (depthwiseWeightUpdate) {
    const auto &f = depthwiseForward;
    const std::size_t bytes =
        (std::size_t(f.batch) * f.inH * f.inW + std::size_t(f.batch) * f.outH *
                                                     f.outW) *
        f.channels * 2;
    e.computeUs = streamed(bytes);
    e.reductionUs = 4.5;
    if (f.dense3x3 == 2) {
      e.reductionBytes = mxk::depthwiseRowsDeltaWorkspaceBytes(f);
      spread(e, mxk::depthwiseRowsDeltaLaunchShape(f).workgroups, 1);
    } else if (f.columns) {
      e.computeUs = mxk::depthwiseColumnDeltasEstimateUs(f) - e.reductionUs;
      e.reductionBytes = mxk::depthwiseWeightDeltaWorkspaceBytes(f);
    }
    return e;
  }
  switch (kernel) {
  case Kernel::GENERIC:
    e.known = false;
    return e;
  case Kernel::DEPTHWISE:
    e.computeUs = streamed(inputBytes() + outputBytes() + weightPackedBytes());
    if (depthwise.columns)
      e.computeUs = mxk::depthwiseColumnsEstimateUs(depthwise);
    else if (depthwise.dense3x3 == 2)
      spread(e, mxk::depthwiseRowsLaunchShape(depthwise).workgroups, 1);
    break;
  case Kernel::IGEMM: {
    if (thinInputOn) {
      // Launch, weights and the first tile's rows (3.5 us), then the block
      // loop - matrix pipe and vector ALU take turns on a SIMD: 1.3 PFLOP/s
      // of the k-steps' padded work - and the tensors' bytes beside it, which
      // overlap it only in part.  Against measurements (N = 32, 224 x 224):
      // 7 x 7 stride 2 3 -> 64 17.9 for 19-21 us, 3 x 3 3 -> 64 37.5 for 35,
      // 3 x 3 3 -> 32 21.1 for 21.1, stride 2 8.7 for 9.5.
      const mxk::ThinInputLaunch l =
          mxk::thinInputLaunchShape(thinInput, gfx950::numCUs);
      const double flops = 2.0 * thinInput.batch * thinInput.outH *
                           ((thinInput.outW + 15) / 16 * 16) *
                           thinInput.outChans * 32.0 *
                           mxk::thinInputKSteps(thinInput);
      e.computeUs =
          3.5 + flops / 1.3e9 +
          double(inputBytes() + outputBytes() + weightPackedBytes()) / 9.0e6;
      spread(e, l.workgroups, 1);
      break;
    }
    if (igemm.small) {
      const int inId = params.inputType == poplar::FLOAT  ? mxk::kFloat
                       : params.inputType == poplar::HALF ? mxk::kHalf
                                                          : mxk::kQuarter;
      e.computeUs = std::max(
          poplin::manySmallTiles(igemm, inId)
              ? poplin::estimateManySmall(igemm, inId) -
                    poplin::kCallOverKernelUs
              : poplin::estimateSmall(igemm, inId),
          streamed(inputBytes() + outputBytes() + weightPackedBytes()));
      spread(e, mxk::igemmSmallTileCount(igemm), 1);
      break;
    }
    if (pointwiseOn) {
      e.computeUs =
          streamed(inputBytes() + outputBytes() + weightPackedBytes());
      // With many input channels a 1x1 layer is as much the matrix cores' as
      // the memory's: N = 32, 28 x 28, 512 -> 512 runs at 710 TFLOP/s
      // (18.5 us where its bytes alone would stream in 10).
      const double flops = 2.0 * pointwise.batch * pointwise.pixels *
                           pointwise.groups * pointwise.inChansPerGroup *
                           pointwise.outChansPerGroup;
      e.computeUs = std::max(e.computeUs, poplin::kLaunchUs + flops / 7.0e8);
      spread(e, mxk::pointwiseLaunchShape(pointwise, gfx950::numCUs).workgroups,
             1);
      break;
    }
    // (K split: the fp32 partial tiles' way out and in again and the second
    // kernel, see splitPenaltyUs)
    const std::size_t partialBytes = mxk::igemmWorkspaceBytes(igemm);
    const double kSplitUs = igemm.splitK <= 1 ? 0.0
                            : igemm.patch || igemm.flex
                                ? poplin::patchSplitUs(partialBytes)
                                : poplin::splitPenaltyUs(partialBytes);
    e.reductionUs = kSplitUs;
    e.reductionBytes = kSplitUs > 0 ? partialBytes : 0;
    bool weighed = false;
    for (const auto &c : candidates)
      if (c.chosen) {
        e.computeUs = c.estimateUs - kSplitUs, weighed = true;
        spread(e, c.workgroups, c.perCU);
      }
    if (weighed)
      break;
    const auto &g = igemm;
    const std::size_t m = std::size_t(g.batch) * g.outD * g.outH * g.outW;
    const std::size_t tiles =
        (m + g.blockM - 1) / g.blockM *
        ((g.outChansPerGroup + g.blockN - 1) / g.blockN) * g.groups * g.splitK;
    const std::size_t steps =
        (kPadded / g.blockK + g.splitK - 1) / g.splitK;
    const std::size_t perCU = g.blockN == 64 || g.stages == 2 ? 2 : 1;
    double us =
        g.flex ? flexEstimateUs()
        : g.blockM == 256
            ? poplin::estimateWide(tiles, steps, g.blockN)
            : poplin::estimateStreaming(tiles, steps, perCU, g.blockN,
                                        g.splitK,
                                        mxk::igemmWorkspaceBytes(igemm),
                                        poplin::stepKindOf(
                                            params.inputType == poplar::FLOAT,
                                            std::size_t(g.kD) * g.kH * g.kW));
    // No kernel is faster than its tensors stream.
    us = std::max(us, streamed(inputBytes() + outputBytes() +
                               weightPackedBytes()));
    e.computeUs = us - kSplitUs;
    spread(e, tiles, perCU);
    break;
  }
  }
  if (paddedInputChans) { // the zero-filling copy of the input
    e.rearrangementUs += streamed(2 * inputBytes());
    e.rearrangementBytes += workspaceBytes - paddedInputOffset;
  }
  if (outputPadded) // the fill of the output before the kernel
    e.rearrangementUs += streamed(outputBytes());
  return e;
}

double mxconv_plan::estimatedMicroseconds() const {
  const DetailedEstimate e = detailedEstimate();
  return e.known ? e.totalUs() : -1.0;
}

std::string mxconv_plan::describe() const {
  std::ostringstream os;
  os << "  Plan (gfx950: " << gfx950::numCUs << " CUs, "
     << gfx950::ldsBytesPerCU / 1024 << " KB LDS/CU, wave"
     << gfx950::wavefrontSize << "):\n";
  os << "        kernel                     ";
  switch (kernel) {
  case Kernel::GENERIC:
    os << "generic direct (vector ALU, any parameters)";
    break;
  case Kernel::IGEMM:
    os << "implicit GEMM (MFMA, "
       << (params.inputType == poplar::QUARTER ? "fp8"
           : params.inputType == poplar::FLOAT ? "fp32"
                                               : "fp16")
       << " operands, fp32 accumulate)"
       << (pointwiseOn ? ", pointwise streaming variant" : "")
       << (thinInputOn ? ", kernel rows as k-steps" : "")
       << (!igemm.patch ? ""
           : igemm.inChansPerGroup * params.inputType.size() % 128 == 0
               ? ", input patch resident in LDS"
               : ", input patch in LDS, its last channel slice a partial one")
       << (igemm.small ? ", small tiles" : "");
    break;
  case Kernel::DEPTHWISE:
    os << (mxk::depthwiseDirectInBlocks(depthwise)
               ? "depthwise direct (vector ALU, one thread per 2x2 block of "
                 "outputs, dilated input)"
           : depthwise.inDilH != 1 || depthwise.inDilW != 1
               ? "depthwise direct (vector ALU, one thread per output "
                 "vector, dilated input)"
           : depthwise.columns
               ? "depthwise direct (vector ALU, strips of columns in registers)"
           : depthwise.dense3x3 == 2
               ? "depthwise direct (vector ALU, input rows streamed through "
                 "an LDS ring by persistent workgroups)"
           : depthwise.dense3x3
               ? "depthwise direct (vector ALU, dense row loads, small "
                 "workgroups)"
               : "depthwise direct (vector ALU, LDS halo tiles)");
    break;
  }
  os << "\n        reason                     " << reason << "\n";
  os << "        zeroConv                   " << (zeroConv ? "true" : "false")
     << "\n";
  os << "        partialsType               float\n";
  if (wuGroupsPerGroup > 1)
    os << "        conv groups per group      " << wuGroupsPerGroup
       << " (the weight update pass of the layer with that many of its "
       << canonical.numConvGroups * wuGroupsPerGroup
       << " groups taken as one; the diagonal blocks of the fused layer's "
          "deltas are handed back)\n";
  if (kernel == Kernel::IGEMM && thinInputOn) {
    const auto &t = thinInput;
    const mxk::ThinInputLaunch l =
        mxk::thinInputLaunchShape(t, gfx950::numCUs);
    const unsigned steps = mxk::thinInputKSteps(t);
    const unsigned perRow = (t.kW * t.inChans + 7) / 8;
    os << "        gemm M x N x K             "
       << std::size_t(t.batch) * t.outH * t.outW << " x " << t.outChans
       << " x " << steps * 32 << " (a kernel row's " << t.kW << " x "
       << t.inChans << " = " << t.kW * t.inChans
       << " neighbouring elements as " << perRow
       << " chunk(s) of 8; the " << t.kH * perRow << " chunks of " << t.kH
       << " kernel rows in " << steps << " k-step(s) of four)\n";
    os << "        block M x N x K            16 x " << t.outChans
       << " x 32 per wave; tiles of " << l.tileRows
       << " output rows of one image, their input rows in " << l.ldsBytes
       << " bytes of LDS\n";
    os << "        workgroups                 " << l.workgroups
       << " persistent (4 waves) taking " << l.tiles << " tiles in turn on "
       << gfx950::numCUs << " CUs\n";
    os << "        packed weights             [" << t.outChans / 16
       << " blocks of 16][" << steps << " k-steps][64 lanes][8]\n";
  } else if (kernel == Kernel::IGEMM) {
    const auto &g = igemm;
    const std::size_t m = std::size_t(g.batch) * g.outD * g.outH * g.outW;
    const std::size_t k =
        std::size_t(g.kD) * g.kH * g.kW * g.inChansPerGroup;
    const std::size_t tiles =
        (m + g.blockM - 1) / g.blockM *
        ((g.outChansPerGroup + g.blockN - 1) / g.blockN) * g.groups;
    os << "        gemm M x N x K             " << m << " x "
       << g.outChansPerGroup << " x " << k << " (x " << g.groups
       << " groups)\n";
    if (convGroupsPerGroup > 1)
      os << "        conv groups per group      " << convGroupsPerGroup
         << " (" << canonical.numConvGroups << " groups of "
         << canonical.inputChannelsPerConvGroup << " -> "
         << canonical.outputChannelsPerConvGroup << " channels run as "
         << g.groups << " of " << g.inChansPerGroup << " -> "
         << g.outChansPerGroup << ", weights block-diagonal)\n";
    if (g.small) {
      const int inId = params.inputType == poplar::FLOAT  ? mxk::kFloat
                       : params.inputType == poplar::HALF ? mxk::kHalf
                                                          : mxk::kQuarter;
      const std::size_t chans = mxk::igemmSmallTileChans(g.small);
      os << "        block M x N x K            "
         << mxk::igemmSmallTilePixels(g.small) << " x " << chans << " x "
         << 64 / params.inputType.size() << "\n";
      os << "        workgroups                 "
         << mxk::igemmSmallTileCount(g) << " on " << gfx950::numCUs
         << " CUs, K shared by the " << mxk::igemmSmallWaves(g, inId)
         << " waves of each\n";
      os << "        packed weights             [G=" << g.groups << "]["
         << (g.outChansPerGroup + chans - 1) / chans * chans / 16 << " blocks of 16]["
         << (k * params.inputType.size() + 63) / 64
         << " k-steps][64 lanes][16 bytes]\n";
      if (paddedInputChans)
        os << "        input channels padded      "
           << params.inputChannelsPerConvGroup << " -> " << paddedInputChans
           << " per group (zero-filled copy in the workspace, every "
              "launch)\n";
    } else if (pointwiseOn) {
      const std::size_t nTiles = (g.outChansPerGroup + 63) / 64;
      const mxk::PointwiseLaunch l =
          mxk::pointwiseLaunchShape(pointwise, gfx950::numCUs);
      os << "        block M x N x K            " << l.tilePixels
         << " x " << l.chansPerWorkgroup << " x " << k << "\n";
      os << "        workgroups                 " << l.workgroups << " on "
         << gfx950::numCUs << " CUs, each taking " << l.tilesPerWorkgroup
         << " tiles in turn through a ring of " << l.ring
         << " LDS buffers filled by " << l.loaderWaves << " loader waves\n";
      os << "        packed weights             [G=" << g.groups << "]["
         << nTiles * 2 << " blocks of 32][" << k / 16
         << " slices of 16][64 lanes][8]\n";
    } else {
      os << "        block M x N x K            " << g.blockM << " x "
         << g.blockN << " x " << g.blockK << "\n";
      os << "        workgroups                 " << tiles * g.splitK
         << " on " << gfx950::numCUs << " CUs ("
         << std::min<std::size_t>(tiles * g.splitK, gfx950::numCUs)
         << " busy, "
         << (tiles * g.splitK + gfx950::numCUs - 1) / gfx950::numCUs
         << " round(s) of tiles)\n";
      if (g.patch)
        os << "        data path                  input rows of the tile "
              "resident in LDS, weights straight to registers; 8 waves, one "
              "workgroup per CU; MFMA blocks of "
           << (g.patch == 2
                   ? "16 pixels, k-steps taken in turn by the two waves of a "
                     "SIMD\n"
                   : "32 pixels, each k-step halved between the two waves of "
                     "a SIMD\n");
      else if (g.flex)
        os << "        data path                  8 waves, each fetching its "
              "share and multiplying "
           << g.blockM / 4 << " x " << g.blockN / 2
           << (g.flex == 2 ? "; two workgroups per CU\n"
                           : "; one workgroup per CU\n");
      else if (g.blockM == 256)
        os << "        data path                  8 waves, each fetching its "
              "share and multiplying 64 x "
           << g.blockN / 2 << "; 2 LDS stages, one workgroup per CU\n";
      else if (g.blockN == 128)
        os << "        LDS stages                 " << g.stages
           << (g.stages == 2 ? " (two workgroups per CU)\n"
                             : " (one workgroup per CU)\n");
      if (g.splitK > 1)
        os << "        K split into parts         " << g.splitK
           << " (fp32 partial tiles, summed by a second kernel)\n";
      if (mxk::igemmTapAddressing(g) == mxk::kRangeTaps)
        os << "        tap addressing             ranges of valid kernel rows "
              "and columns (more than 32 taps)\n";
      else if (!igemmPhases.empty())
        os << "        dilated input              " << igemmPhases.size()
           << " phases, one convolution of the undilated input each, in "
              "one launch\n";
      else if (mxk::igemmTapAddressing(g) == mxk::kDilatedTaps)
        os << "        tap addressing             arithmetic (dilated "
              "input)\n";
      if (g.patch)
        os << "        packed weights             [G=" << g.groups << "]["
           << coPadded / 32 << " blocks of 32]["
           << (std::size_t(g.inChansPerGroup) * params.inputType.size() + 127) /
                  128 * g.kH * g.kW
           << " k-steps]"
           << (g.patch == 2 ? "[4 operands]" : "[2 halves][2]")
           << "[64 lanes][16 bytes]\n";
      else
        os << "        packed weights             [G=" << g.groups << "]["
           << coPadded << "][" << kPadded << "]\n";
      if (!candidates.empty()) {
        os << "        tilings weighed            workgroups  per CU  rounds  "
              "k-steps  estimate\n";
        for (const auto &c : candidates) {
          char line[160];
          std::snprintf(line, sizeof line,
                        "          %c %-34s %8zu  %6zu  %6.2f  %7zu  %7.1f us\n",
                        c.chosen ? '*' : ' ', c.name.c_str(), c.workgroups,
                        c.perCU, c.rounds, c.kSteps, c.estimateUs);
          os << line;
        }
      }
      if (paddedInputChans)
        os << "        input channels padded      "
           << params.inputChannelsPerConvGroup << " -> " << paddedInputChans
           << " per group (zero-filled copy in the workspace, every "
              "launch)\n";
    }
  } else if (kernel == Kernel::DEPTHWISE) {
    const auto &d = depthwise;
    os << "        channels                   " << d.channels << "\n";
    if (d.columns)
      os << "        output columns per lane    " << d.columns
         << ", walked down in bands of " << d.columnRows << " rows\n";
    else if (!d.dense3x3)
      os << "        output tile H x W          " << d.tileH << " x "
         << d.tileW
         << (d.stripPixels == 7
                 ? ", a strip of 7 neighbouring pixels per thread"
                 : d.stripPixels == 4
                       ? ", a strip of 4 neighbouring pixels per thread"
                       : "")
         << "\n";
    if (d.dense3x3 == 2) {
      const mxk::DepthwiseRowsLaunch l = mxk::depthwiseRowsLaunchShape(d);
      os << "        workgroups                 " << l.workgroups << " on "
         << d.cus << " CUs: per image " << l.strips << " strips of "
         << l.colsOut << " output columns x " << l.bands << " bands of "
         << l.rowsOut << " output rows; ring of " << l.ringRows
         << " input rows in LDS filled by " << l.loaderWaves
         << " loader waves, read by " << l.computeWaves << " compute waves\n";
    }
    os << "        packed weights             [" << d.kH * d.kW << "]["
       << d.channels << "]\n";
  } else {
    os << "        packed weights             [G][K][Ci][Co]\n";
  }
  if (depthwiseWeightUpdate) {
    os << "        as a weight update pass    depthwise weight-delta kernel "
          "on the layer's own tensors";
    if (depthwiseForward.dense3x3 == 2) {
      const mxk::DepthwiseRowsLaunch l =
          mxk::depthwiseRowsDeltaLaunchShape(depthwiseForward);
      os << ", rows of both streamed through LDS rings by " << l.workgroups
         << " persistent workgroups (" << l.strips << " strips x " << l.bands
         << " bands of " << l.rowsOut << " rows per image)";
    }
    if (depthwiseForward.columns)
      os << ", strips of " << depthwiseForward.columns
         << " columns walked down in registers, bands of "
         << depthwiseForward.columnRows << " rows";
    os << "\n";
  }
  if (denseWeightUpdate && denseForward.windowCo) {
    const auto &f = denseForward;
    // (groups that leave most of a 128 x 128 tile empty: what the kernel of
    // such tiles is not for)
    const bool narrow = f.groups > 1 && std::size_t(f.ci) * f.co * 4 <=
                                            std::size_t((f.ci + 127) / 128) *
                                                ((f.co + 127) / 128) * 16384;
    os << "        as a weight update pass    "
       << (narrow             ? "kernel of narrow groups"
           : f.elemBytes == 4 ? "fp32 matrix-core kernel"
                              : "matrix-core weight-delta kernel")
       << " on the layer's own tensors (pixels gathered in registers): tiles "
          "of "
       << f.windowCo << " output x " << f.windowCi
       << " input channels and a kernel row, chunks of " << f.windowSteps
       << " k-steps of 32 columns = " << mxk::wuWindowWorkgroups(f)
       << " workgroups"
       << (mxk::wuWindowWorkspaceBytes(f) ? ", fp32 partial sums added in order"
                                          : ", the result written at once");
    if (f.resultCi != f.ci)
      os << "; input channels padded " << f.resultCi << " -> " << f.ci;
    if (f.resultCo != f.co)
      os << "; output channels padded " << f.resultCo << " -> " << f.co;
    os << "\n";
  } else if (denseWeightUpdate) {
    const auto &f = denseForward;
    const std::size_t m = std::size_t(f.batch) * f.outH * f.outW;
    const std::size_t chunks = (m + f.chunkPixels - 1) / f.chunkPixels;
    const std::size_t tiles = std::size_t(f.groups) * f.kH * f.kW *
                              ((f.ci + 127) / 128) * ((f.co + 127) / 128);
    os << "        as a weight update pass    matrix-core weight-delta kernel "
          "on the layer's own tensors (transposing LDS reads): "
       << tiles << " tap x channel tiles x " << chunks << " chunks of "
       << f.chunkPixels << " pixels = " << tiles * chunks
       << " workgroups, fp32 partial tiles summed in order";
    if (f.resultCi != f.ci)
      os << "; input channels padded " << f.resultCi << " -> " << f.ci;
    if (f.resultCo != f.co)
      os << "; output channels padded " << f.resultCo << " -> " << f.co;
    os << "\n";
  }
  if (weightUpdateProduct) {
    const auto &q = weightUpdateProduct->params;
    std::string tiling;
    for (const auto &c : weightUpdateProduct->candidates)
      if (c.chosen)
        tiling = c.name;
    os << "        as a weight update pass    one matrix product, "
          "transpose(deltas) x activations: "
       << q.batchSize << " x " << q.inputChannelsPerConvGroup << " x "
       << q.outputChannelsPerConvGroup
       << " (output channels x batch x input channels), its result in "
          "weight order as it is"
       << (tiling.empty() ? "" : "; " + tiling) << "\n";
  }
  os << "        workspaceBytes             " << workspaceBytes << "\n";
  const bool columns = kernel == Kernel::DEPTHWISE && depthwise.columns;
  if (columns || (kernel == Kernel::IGEMM &&
                  (igemm.small || (igemm.patch && igemm.splitK > 1)))) {
    // the plan without the small tiles, without a resident patch and its
    // parts of K or without strips of columns, which they stand in for
    poplin::ConvOptions o = options;
    o.planConstraints = poplin::PlanConstraints{};
    if (columns)
      o.planConstraints.columns = 0;
    else
      o.planConstraints.smallTile = 0;
    if (!columns && !igemm.small)
      o.planConstraints.patch = 0;
    o.planConstraints.convGroupsPerGroup = convGroupsPerGroup;
    const mxconv_plan other = poplin::makePlan(params, o);
    char line[96] = "  Left aside for it:\n";
    if (!columns) // (the other depthwise estimates count bytes alone)
      std::snprintf(line, sizeof line,
                    "  Left aside for it (estimates: %.1f us, above %.1f us):\n",
                    other.estimatedMicroseconds(), estimatedMicroseconds());
    // (without the heading, which names the chip again)
    const std::string text = other.describe();
    os << line << text.substr(text.find('\n') + 1);
  }
  return os.str();
}
