// The runtime-radix transforms fused with the image-domain work on either side
// (hws_fft_fused.hip at the power-of-two sizes): the forward rows pass computed
// from the model image for every layer, and the backward columns pass with the
// w-projection.
#include "hws_fft_generic.h"

#include <algorithm>

namespace hws {

namespace {

// The first-stage cells of this thread in a blocked runtime-radix transform
// whose first radix is R: visit(slot, pos, f) for each (the slots of
// blockedRtStage's first stage).
template <int R, int L, class Visit>
__device__ __forceinline__ void firstStageCells(int n, int tid, int nthr, const Visit& visit) {
  constexpr int kBatches = kMaxValues / R;
  constexpr int LS = L == 4 ? 2 : L == 2 ? 1 : 0;
  asm volatile("" : "+v"(tid));
  const int B = n / R;
  const int total = B * L;
#pragma unroll
  for (int q = 0; q < kBatches; ++q) {
    const int t = tid + q * nthr;
    if (t < total) {
      const int f = t & (L - 1), b = t >> LS;
#pragma unroll
      for (int r = 0; r < R; ++r) visit(q * R + r, b + r * B, f);
    }
  }
}

// Forward rows pass computed from the model for every layer of the batch at
// the sizes the runtime-radix kernels serve (fftRowsModelLayersKernel at the
// power-of-two sizes): a workgroup owns L rows of one image, reads their
// model values and computes their n' once into registers (the cells of its
// first stage), and then, layer after layer, forms each cell's w-phased
// input (modelTerm, as modelCell forms it), transforms the rows and writes
// the tile columns the columns pass reads (colNeed: one bit per (layer, tile
// column)). grid (H / L, layer groups): group blockIdx.y takes perGroup
// consecutive layers. Mixed precision only: the 1024 threads of the long rows
// leave 128 registers, and with the reference precision's FP64 sine and cosine
// 106 to 240 values spill inside the layer loop.
template <bool CPLX, int L>
__global__ void __launch_bounds__(1024)
fftRowsModelLayersGenericKernel(float2* __restrict__ data, int W, int H, int nbatch,
                                int perGroup, unsigned long long radices, const float2* __restrict__ tw,
                                ModelSource ms, const uint32_t* __restrict__ colNeed,
                                int tshift) {
  extern __shared__ float2 lds[];
  const int tid = threadIdx.x, nthr = blockDim.x;
  const int rblk = sharedSegmentBlock<L>(int(blockIdx.x), int(gridDim.x));
  const int r0 = rblk * L;
  const size_t HW = size_t(W) * H;
  float2* rowBase = data + size_t(r0 >> 2) * 4 * W + (r0 & 3);
  const int tilesX = (W + (1 << tshift) - 1) >> tshift;
  float re[kMaxValues], imv[CPLX ? kMaxValues : 1];
  double np[kMaxValues];
  auto cell = [&](int slot, int x, int f) {
    const int y = r0 + f;
    int yDest = y + H / 2;
    if (yDest >= H) yDest -= H;
    int xDest = (W - x) + W / 2;
    if (xDest >= W) xDest -= W;
    const double m = pixelM(yDest, H, ms.dm, ms.mShift);
    const double l = pixelL(xDest, W, ms.dl, ms.lShift);
    np[slot] = nPrimeSeries(l, m);
    const size_t src = size_t(yDest) * W + xDest;
    re[slot] = ms.re[src];
    if (CPLX) imv[slot] = -ms.im[src];
  };
  switch (radices & 15ull) {
    case 1: firstStageCells<16, L>(W, tid, nthr, cell); break;
    case 8: firstStageCells<8, L>(W, tid, nthr, cell); break;
    case 4: firstStageCells<4, L>(W, tid, nthr, cell); break;
    case 2: firstStageCells<2, L>(W, tid, nthr, cell); break;
    case 3: firstStageCells<3, L>(W, tid, nthr, cell); break;
    case 5: firstStageCells<5, L>(W, tid, nthr, cell); break;
    case 7: firstStageCells<7, L>(W, tid, nthr, cell); break;
    default: break;
  }
  const int bEnd = min(nbatch, (int(blockIdx.y) + 1) * perGroup);
#pragma unroll 1
  for (int b = int(blockIdx.y) * perGroup; b < bEnd; ++b) {
    const int layer = ms.layer0 + b;
    const double w = layerToW(ms.map, layer);
    float2* base = rowBase + size_t(b) * HW;
    const size_t cbit = size_t(layer) * tilesX;
    auto load = [&](int slot, int, int) -> float2 {
      return modelTerm<false>(re[slot], CPLX ? imv[slot] : 0.0f, CPLX, w, np[slot]);
    };
    auto store = [&](int, int x, int f, float2 v) {
      const size_t bit = cbit + size_t(x >> tshift);
      if ((colNeed[bit >> 5] >> (bit & 31)) & 1u) streamStore(&base[size_t(x) * 4 + f], v);
    };
    blockedRtFft<-1, L>(lds, W, radices, tw, tid, nthr, load, store);
    __syncthreads();  // the last stage's LDS reads precede the next layer's writes
  }
}

// Backward columns pass fused with the projection at the runtime-radix
// sizes (fftColsProjectKernel at the power-of-two sizes): a workgroup owns
// one column of one image and transforms it layer after layer, in the pass's
// layer order; each transformed cell is rotated by its layer's w term and
// added (Kahan) to its pixel's sums, which stay in registers with the
// pixel's n' (the cells of the last stage's slots). Cells of tile rows
// without samples read as zero. Every term is computed and added as
// projectKernel computes and adds it. grid (W, images of the kind);
// dynamic LDS: the transform buffer, then the row bits of the pass's layers.
// Real images keep to 128 registers (82 values spill in the mixed precision, 78 in
// the reference one: 52 and 60 bytes of scratch a lane) and take the closest
// multiple of 64 threads, so that two workgroups share a CU at the large sizes:
// with 142 registers and a power of two of threads one did, and 6144^2 x 96 layers
// took 28.1 ms against 21.8; in the reference precision the invert of one image at
// 3072^2 x 48 layers took 3.96 ms and takes 2.23. Complex images hold twice the sums
// (206 registers; 128 would spill them).
template <bool REF, bool CPLX>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(CPLX ? 2 : 4)))
fftColsProjectGenericKernel(ColsProjectArgs a, const float2* __restrict__ layers,
                            unsigned long long radices, const float2* __restrict__ tw,
                            float* __restrict__ sum, float* __restrict__ comp,
                            float* __restrict__ isum, float* __restrict__ icomp) {
  extern __shared__ float2 lds[];
  const int tid = threadIdx.x, nthr = blockDim.x;
  const int W = a.W, H = a.H;
  const size_t HW = size_t(W) * H;
  const int img = a.img[blockIdx.y];
  const bool fresh = a.fresh != 0;
  // the four columns of a 128-byte segment run on one XCD, one after the other
  const int nb = int(gridDim.x);
  int x0 = int(blockIdx.x);
  if ((nb & 7) == 0) x0 = (x0 & 7) * (nb >> 3) + (x0 >> 3);
  uint32_t* bits =
      reinterpret_cast<uint32_t*>(reinterpret_cast<unsigned char*>(lds) + blockedGenericLds(1, H));
  const int nl = a.nLayersInPass;
  {
    const size_t nbits = size_t(nl) * a.tilesY;
    const size_t bit0 = size_t(a.passStart) * a.tilesY;
    const size_t w0 = bit0 >> 5;
    const int sh = int(bit0 & 31);
    for (size_t wd = size_t(tid); wd < (nbits + 31) / 32; wd += size_t(nthr)) {
      uint32_t v = a.rowLive[w0 + wd] >> sh;
      if (sh != 0 && w0 + wd + 1 < a.rowLiveWords) v |= a.rowLive[w0 + wd + 1] << (32 - sh);
      bits[wd] = v;
    }
  }
  // this thread's output pixels (the last stage's slots): n' and the sums
  float s[kMaxValues], c[kMaxValues], is[CPLX ? kMaxValues : 1], ic[CPLX ? kMaxValues : 1];
  double np[kMaxValues];
  auto pixel = [&](int y) {
    int ySrc = (H - y) + H / 2;
    if (ySrc >= H) ySrc -= H;
    int xSrc = x0 + W / 2;
    if (xSrc >= W) xSrc -= W;
    return size_t(img) * HW + size_t(ySrc) * W + xSrc;
  };
  auto init = [&](int slot, int y, int) {
    int ySrc = (H - y) + H / 2;
    if (ySrc >= H) ySrc -= H;
    int xSrc = x0 + W / 2;
    if (xSrc >= W) xSrc -= W;
    const double m = pixelM(ySrc, H, a.dm, a.mShift);
    const double l = pixelL(xSrc, W, a.dl, a.lShift);
    double v = nPrime(l, m);
    if (REF) v = double(float(v));
    np[slot] = v;
    const size_t o = pixel(y);
    s[slot] = fresh ? 0.0f : sum[o];
    c[slot] = fresh ? 0.0f : comp[o];
    if (CPLX) {
      is[slot] = fresh ? 0.0f : isum[o];
      ic[slot] = fresh ? 0.0f : icomp[o];
    }
  };
  auto finish = [&](int slot, int y, int) {
    const size_t o = pixel(y);
    sum[o] = s[slot];
    comp[o] = c[slot];
    if (CPLX) {
      isum[o] = is[slot];
      icomp[o] = ic[slot];
    } else if (fresh && isum != nullptr) {
      // a fresh pass also zeroes the imaginary accumulators of real images
      isum[o] = 0.0f;
      icomp[o] = 0.0f;
    }
  };
  // the last stage's radix: the highest nonzero 4-bit code
  int lastCode = 0;
  for (unsigned long long r = radices; r != 0ull; r >>= 4) lastCode = int(r & 15ull);
  auto overLastSlots = [&](const auto& visit) {
    switch (lastCode) {
      case 1: firstStageCells<16, 1>(H, tid, nthr, visit); break;
      case 8: firstStageCells<8, 1>(H, tid, nthr, visit); break;
      case 4: firstStageCells<4, 1>(H, tid, nthr, visit); break;
      case 2: firstStageCells<2, 1>(H, tid, nthr, visit); break;
      case 3: firstStageCells<3, 1>(H, tid, nthr, visit); break;
      case 5: firstStageCells<5, 1>(H, tid, nthr, visit); break;
      case 7: firstStageCells<7, 1>(H, tid, nthr, visit); break;
      default: break;
    }
  };
  overLastSlots(init);
  __syncthreads();  // the row bits
  const float2* col = layers + size_t(img) * a.nLayersPass * HW + size_t(x0) * 4;
#pragma unroll 1
  for (int li = 0; li < nl; ++li) {
    const float2* lay = col + size_t(li) * HW;
    const double w = layerToW(a.map, a.passStart + li);
    auto load = [&](int, int y, int) -> float2 {
      const int bit = li * a.tilesY + (y >> a.tshift);
      if (!((bits[bit >> 5] >> (bit & 31)) & 1u)) return make_float2(0.0f, 0.0f);
      return lay[size_t(y >> 2) * W * 4 + (y & 3)];
    };
    auto project = [&](int slot, int, int, float2 v) {
      const float2 t = projectTerm<REF>(v, w, np[slot]);
      kahanAdd(s[slot], c[slot], t.x);
      if (CPLX) kahanAdd(is[slot], ic[slot], t.y);
    };
    blockedRtFft<+1, 1>(lds, H, radices, tw, tid, nthr, load, project);
    __syncthreads();  // the last stage's LDS reads precede the next layer's writes
  }
  overLastSlots(finish);
}

}  // namespace

void launchModelLayersGeneric(int threads, int lines, dim3 grid, size_t lds, hipStream_t st,
                              float2* data, int W, int H, int nbatch, unsigned long long rad,
                              const float2* tw, const ModelSource& ms, const uint32_t* colNeed,
                              int tshift) {
  const bool cplx = ms.cplx != 0;
  // At least kModelGroups workgroups, in layer groups of at least two (a group
  // computes its rows' n' anew): 1500 x 1260 has 315 four-row workgroups, which
  // left some CUs with two and others with one (24 layers: 420 us an image in
  // one group, 280 in four).
  constexpr int kModelGroups = 1024;
  const int rowBlocks = int(grid.x);
  const int groups = std::min((nbatch + 1) / 2, (kModelGroups + rowBlocks - 1) / rowBlocks);
  const int per = (nbatch + groups - 1) / groups;
  grid.y = unsigned((nbatch + per - 1) / per);
#define HWS_MODEL_GENERIC(C, LL)                                                                \
  hipLaunchKernelGGL((fftRowsModelLayersGenericKernel<C, LL>), grid, dim3(threads), lds,  \
                     st, data, W, H, nbatch, per, rad, tw, ms, colNeed, tshift)
  if (lines == 4) {
    if (cplx) HWS_MODEL_GENERIC(true, 4);
    else HWS_MODEL_GENERIC(false, 4);
  } else if (lines == 2) {
    if (cplx) HWS_MODEL_GENERIC(true, 2);
    else HWS_MODEL_GENERIC(false, 2);
  } else {
    if (cplx) HWS_MODEL_GENERIC(true, 1);
    else HWS_MODEL_GENERIC(false, 1);
  }
#undef HWS_MODEL_GENERIC
}

namespace {
// The runtime-radix fused kernel: one column per workgroup of at most 512
// threads; its LDS is the transform buffer and the row bits.
size_t colsProjectGenericLds(int H, int nLayersInPass, int tilesY) {
  const size_t words = (size_t(nLayersInPass) * tilesY + 31) / 32;
  return blockedGenericLds(1, H) + words * sizeof(uint32_t);
}
}  // namespace

bool colsProjectGenericSupported(const hws_gridder* g, int nLayersInPass, size_t maxLds) {
  const int t = threadsFor(g->colPlan, 1, true);
  // (the kinds are launched one after the other: the smaller counts)
  int images = kMaxImages;
  for (const KindPlan& kp : g->plan.kinds)
    if (kp.active) images = std::min(images, kp.nImg);
  return fusedColumns(long(g->W) * images, (t + 63) / 64) && t != 0 && t <= 512 &&
         colsProjectGenericLds(g->H, nLayersInPass, g->plan.tilesY) <= maxLds;
}

void launchColsProjectGeneric(hws_gridder* g, const ColsProjectArgs& a, bool cplx,
                              const float2* layers, float* sum, float* comp, float* isum,
                              float* icomp) {
  const bool ref = g->cfg.precision == HWS_PRECISION_REFERENCE;
  const dim3 grid(unsigned(a.W), unsigned(a.nImg));
  const int threads = threadsFor(g->colPlan, 1, true);
  const size_t lds = colsProjectGenericLds(a.H, a.nLayersInPass, a.tilesY);
  const unsigned long long rad = packRadices(g->colPlan);
  const float2* tw = g->colPlan.twBackward;
#define HWS_COLS_PROJECT_GENERIC(R, C)                                                          \
  hipLaunchKernelGGL((fftColsProjectGenericKernel<R, C>), grid, dim3(threads), lds, g->stream,   \
                   a, layers, rad, tw, sum, comp, isum, icomp)
  if (ref && cplx) HWS_COLS_PROJECT_GENERIC(true, true);
  else if (ref) HWS_COLS_PROJECT_GENERIC(true, false);
  else if (cplx) HWS_COLS_PROJECT_GENERIC(false, true);
  else HWS_COLS_PROJECT_GENERIC(false, false);
#undef HWS_COLS_PROJECT_GENERIC
}

}  // namespace hws
