// The power-of-two layer transforms (256 to 4096) fused with the image-domain
// work on either side: the backward columns pass with the w-projection, and
// the forward rows pass computed from the model image for every layer.
#include "hws_fft_device.h"

#include <algorithm>

namespace hws {

namespace {

// Two waves per SIMD (256 registers a lane). Left to itself the compiler
// takes up to 512 at the sizes whose workgroups allow it (below 4096) to hold
// the layer-independent twiddles, and the one wave left per SIMD waits out
// every LDS access and barrier: at 2048^2 with 32 layers the fused columns of
// two real images took 1108 us and take 682, the model rows 547 and 486 us an
// image (reference precision: 1410 -> 818 and 690 -> 550). The twiddles that no
// longer fit spill: 14 to 58 values of the fused columns from 512 up (20 at 2048
// for real images in the mixed precision, 56 for complex ones). Three waves (168
// registers) spill the sums too.
#define HWS_TWO_WAVES __attribute__((amdgpu_waves_per_eu(2, 2)))

// Backward columns pass (after fftRowsBlockedSparseKernel) fused with
// projectOnImageAndCorrect (gridding/wstackinggridder.cpp:874-907) for every
// layer of the pass: a workgroup owns two columns of one image and transforms
// them layer after layer, in the pass's layer order; each transformed cell is
// rotated by its layer's w term and added (Kahan) to its pixel's sums, which
// stay in registers. So the transformed layers are never written, and the
// accumulators are read (unless the pass is the first) and written once per
// pass. Cells of tile rows without samples read as zero, as in
// fftColsBlockedRowSparseKernel. The next layer's inputs are loaded while the
// current layer is transformed. Every term is computed and added as
// projectKernel computes and adds it, so the sums are the same bits.
// grid (W / 2, images of the kind); dynamic LDS: the transform buffer and
// the row bits of the pass's layers.
template <int N, bool REF, bool CPLX>
__global__ void __launch_bounds__(kProjectColumns * N / 16) HWS_TWO_WAVES
fftColsProjectKernel(ColsProjectArgs a, const float2* __restrict__ layers,
                     const float2* __restrict__ tw, float* __restrict__ sum,
                     float* __restrict__ comp, float* __restrict__ isum,
                     float* __restrict__ icomp) {
  constexpr int NF = kProjectColumns;
  constexpr int T = NF * N / 16;
  constexpr int B0 = N / 16;  // the first stage is radix 16: one butterfly per thread
  constexpr int RL = LastStage<N>::R, NSL = LastStage<N>::NS, PERL = 16 / RL;
  extern __shared__ float2 fusedLds[];
  float2* lds = fusedLds;
  // n' of this thread's 16 output cells: [k][thread] (registers would not
  // hold them beside the transform, the prefetch and the sums)
  double* npl = reinterpret_cast<double*>(fusedLds + NF * N + (NF * N) / 64);
  uint32_t* bits = reinterpret_cast<uint32_t*>(npl + 16 * T);
  const int tid = int(threadIdx.x);
  const int W = a.W;
  const size_t HW = size_t(W) * N;
  const int img = a.img[blockIdx.y];
  const bool fresh = a.fresh != 0;
  // column pairs sharing 128-byte segments run on one XCD, one after the other
  const int nb = int(gridDim.x);
  int cp = int(blockIdx.x);
  if ((nb & 7) == 0) cp = (cp & 7) * (nb >> 3) + (cp >> 3);
  const int x0 = cp * NF;
  // the row bits of the pass's layers: bit li * tilesY + ty
  const int nl = a.nLayersInPass;
  const size_t nbits = size_t(nl) * a.tilesY;
  const size_t bit0 = size_t(a.passStart) * a.tilesY;
  const size_t w0 = bit0 >> 5;
  const int sh = int(bit0 & 31);
  for (size_t wd = size_t(tid); wd < (nbits + 31) / 32; wd += T) {
    uint32_t v = a.rowLive[w0 + wd] >> sh;
    if (sh != 0 && w0 + wd + 1 < a.rowLiveWords) v |= a.rowLive[w0 + wd + 1] << (32 - sh);
    bits[wd] = v;
  }
  // this thread's output pixels: n' and the accumulators
  float s[16], c[16], is[CPLX ? 16 : 1], ic[CPLX ? 16 : 1];
#pragma unroll
  for (int q = 0; q < PERL; ++q) {
    const int bt = tid + q * T;
    const int f = bt % NF, b = bt / NF;
    const int base = (b / NSL) * NSL * RL + b % NSL;
#pragma unroll
    for (int r = 0; r < RL; ++r) {
      const int k = q * RL + r;
      const int y = base + r * NSL, x = x0 + f;
      int ySrc = (N - y) + N / 2;
      if (ySrc >= N) ySrc -= N;
      int xSrc = x + W / 2;
      if (xSrc >= W) xSrc -= W;
      const double m = pixelM(ySrc, N, a.dm, a.mShift);
      const double l = pixelL(xSrc, W, a.dl, a.lShift);
      double np = nPrime(l, m);
      if (REF) np = double(float(np));
      npl[k * T + tid] = np;
      const size_t o = size_t(img) * HW + size_t(ySrc) * W + xSrc;
      // (read also in a fresh pass, where the values are not used: no
      // branch around the loads)
      s[k] = fresh ? 0.0f : sum[o];
      c[k] = fresh ? 0.0f : comp[o];
      if (CPLX) {
        is[k] = fresh ? 0.0f : isum[o];
        ic[k] = fresh ? 0.0f : icomp[o];
      }
    }
  }
  __syncthreads();  // the row bits
  const int f0 = tid % NF, b0 = tid / NF;
  const float2* col = layers + size_t(img) * a.nLayersPass * HW + size_t(x0) * 4;
  float2 in[16], out[16];
  // cells of tile rows without samples were never written: their loads
  // take an offset out of the buffer's range and return zero (no branch
  // around the loads, and 32-bit offsets against a per-layer resource)
  const int colBytes = int((HW - size_t(x0) * 4) * sizeof(float2));
  auto load = [&](int li, float2* dst) {
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float2*>(col + size_t(li) * HW), 0, colBytes, kRawBufferFlags);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int pos = b0 + r * B0;
      const int bit = li * a.tilesY + (pos >> a.tshift);
      const uint32_t off = ((bits[bit >> 5] >> (bit & 31)) & 1u)
                               ? uint32_t(blockedAddr<false>(pos, f0, W) * sizeof(float2))
                               : kOffsetOutOfRange;
      const auto v = __builtin_amdgcn_raw_buffer_load_b64(rs, off, 0, 0);
      // (the elements by value: a bit cast of a vector element would read
      // element 0 for both with this compiler)
      const unsigned lo = v[0], hi = v[1];
      dst[r] = make_float2(__uint_as_float(lo), __uint_as_float(hi));
    }
  };
  load(0, in);
#pragma unroll 1
  for (int li = 0; li < nl; ++li) {
    // the next layer's inputs are loaded once the first stage has read this one's
    regFft<+1, N, NF>(lds, tw, tid, in, out, [&] {
      if (li + 1 < nl) load(li + 1, in);
    });
    const double w = layerToW(a.map, a.passStart + li);
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const float2 t = projectTerm<REF>(out[k], w, npl[k * T + tid]);
      kahanAdd(s[k], c[k], t.x);
      if (CPLX) kahanAdd(is[k], ic[k], t.y);
      // one cell's term at a time: interleaving the sixteen would hold
      // their temporaries at once
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  const bool zeroImag = !CPLX && fresh && isum != nullptr;
#pragma unroll
  for (int q = 0; q < PERL; ++q) {
    const int bt = tid + q * T;
    const int f = bt % NF, b = bt / NF;
    const int base = (b / NSL) * NSL * RL + b % NSL;
#pragma unroll
    for (int r = 0; r < RL; ++r) {
      const int k = q * RL + r;
      const int y = base + r * NSL, x = x0 + f;
      int ySrc = (N - y) + N / 2;
      if (ySrc >= N) ySrc -= N;
      int xSrc = x + W / 2;
      if (xSrc >= W) xSrc -= W;
      const size_t o = size_t(img) * HW + size_t(ySrc) * W + xSrc;
      sum[o] = s[k];
      comp[o] = c[k];
      if (CPLX) {
        isum[o] = is[k];
        icomp[o] = ic[k];
      } else if (zeroImag) {
        // a fresh pass also zeroes the imaginary accumulators of real images
        isum[o] = 0.0f;
        icomp[o] = 0.0f;
      }
    }
  }
}

// Rows per workgroup of the model rows pass: the four of a row block, so that
// every store fills its 32-byte group and the lanes of a wave whole lines.
// With two rows, whose partner rows another workgroup stored some time later,
// most of the output reached memory in half groups (4096^2 x 64 layers x four
// images: 14.3 ms against 11.6; 1024^2 x 32 layers: 156 us against 84).
constexpr int kModelRows = 4;

// Whether the model rows pass keeps to 128 registers and four waves per SIMD
// by forming the thread index and the twiddle address anew for each layer;
// else two waves hold what the compiler hoists out of the layer loop. 1024
// threads (4096) leave no choice; below, measured: real mixed images 320 us
// against 359 (2048^2 x 32 layers) and 84 against 93 (1024^2), but complex ones
// 427 against 373, the reference precision 515 against 496 (both spill), and
// 512^2 x 16 layers, which does not fill the chip, 24 against 18.
template <int N, bool REF, bool CPLX>
constexpr bool kModelLean = N > 2048 || (N >= 1024 && !REF && !CPLX);

// Forward rows pass computed from the model for every layer of the batch
// (copyImageToLayerAndInverseCorrect, gridding/wstackinggridder.cpp:934-969,
// then the row transforms): a workgroup owns four rows of one image, reads
// their model values and computes their n' once, and then, layer after
// layer, forms each cell's w-phased input (modelTerm, as modelCell forms it),
// transforms the rows and writes the tile columns the columns pass reads
// (colNeed: one bit per (layer, tile column); the columns pass skips the
// others). The cells' model values and n' stay in registers across the
// layers, so a layer costs the phase, the transform and the stores.
// grid (H / 4, layer groups): group blockIdx.y takes perGroup consecutive
// layers; each XCD takes a contiguous range of row blocks.
template <int N, bool REF, bool CPLX>
__global__ void __launch_bounds__(kModelRows * N / 16)
    __attribute__((amdgpu_waves_per_eu(kModelLean<N, REF, CPLX> ? 4 : 2)))
fftRowsModelLayersKernel(float2* __restrict__ data, int H, int nbatch, int perGroup,
                         const float2* __restrict__ tw, ModelSource ms,
                         const uint32_t* __restrict__ colNeed, int tshift) {
  constexpr int NF = kModelRows;
  constexpr int T = NF * N / 16;
  constexpr int B0 = N / 16;
  constexpr int RL = LastStage<N>::R, NSL = LastStage<N>::NS, PERL = 16 / RL;
  __shared__ float2 lds[NF * N + (NF * N) / 64];
  const int tid = int(threadIdx.x);
  const int W = N;
  const size_t HW = size_t(W) * H;
  const int nb = int(gridDim.x);
  int rp = int(blockIdx.x);
  if ((nb & 7) == 0) rp = (rp & 7) * (nb >> 3) + (rp >> 3);
  const int y0 = rp * NF;
  const int tilesX = W >> tshift;
  // this thread's first-stage cells: x = b0 + r N / 16 of row y0 + f0
  const int f0 = tid % NF, b0 = tid / NF;
  float re[16], imv[CPLX ? 16 : 1];
  double np[16];
  {
    const int y = y0 + f0;
    int yDest = y + H / 2;
    if (yDest >= H) yDest -= H;
    const double m = pixelM(yDest, H, ms.dm, ms.mShift);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int x = b0 + r * B0;
      int xDest = (W - x) + W / 2;
      if (xDest >= W) xDest -= W;
      const double l = pixelL(xDest, W, ms.dl, ms.lShift);
      np[r] = nPrimeSeries(l, m);
      if (REF) np[r] = double(float(np[r]));
      const size_t src = size_t(yDest) * W + xDest;
      re[r] = ms.re[src];
      if (CPLX) imv[r] = -ms.im[src];
    }
  }
  // the rows' cells in the blocked layout: row y0 + f of a layer at
  // rowBase + layer offset + x * 4 + f
  const size_t rowBase = size_t(y0 >> 2) * 4 * W + size_t(y0 & 3);
  float2 in[16], out[16];
  const int bEnd = min(nbatch, (int(blockIdx.y) + 1) * perGroup);
#pragma unroll 1
  for (int b = int(blockIdx.y) * perGroup; b < bEnd; ++b) {
    const int layer = ms.layer0 + b;
    const double w = layerToW(ms.map, layer);
#pragma unroll
    for (int r = 0; r < 16; ++r)
      in[r] = modelTerm<REF>(re[r], CPLX ? imv[r] : 0.0f, CPLX, w, np[r]);
    int tl = tid;
    const float2* twl = tw;
    if constexpr (kModelLean<N, REF, CPLX>) asm volatile("" : "+v"(tl), "+s"(twl));
    regFft<-1, N, NF>(lds, twl, tl, in, out, [] {});
    float2* g = data + size_t(b) * HW + rowBase;
    const size_t cbit = size_t(layer) * tilesX;
#pragma unroll
    for (int q = 0; q < PERL; ++q) {
      const int bt = tl + q * T;
      const int f = bt % NF, bb = bt / NF;
      const int base = (bb / NSL) * NSL * RL + bb % NSL;
#pragma unroll
      for (int r = 0; r < RL; ++r) {
        const int x = base + r * NSL;
        const size_t bit = cbit + size_t(x >> tshift);
        if ((colNeed[bit >> 5] >> (bit & 31)) & 1u)
          streamStore(&g[size_t(x) * 4 + f], out[q * RL + r]);
      }
    }
  }
}
}  // namespace

size_t colsProjectLds(int H, int nLayersInPass, int tilesY) {
  const size_t words = (size_t(nLayersInPass) * tilesY + 31) / 32;
  const size_t n = size_t(kProjectColumns) * H;
  // transform buffer, n' of every output cell, row bits
  return (n + n / 64) * sizeof(float2) + n * sizeof(double) + words * sizeof(uint32_t);
}

bool launchColsProjectPow2(hws_gridder* g, const ColsProjectArgs& a, bool cplx,
                           const float2* layers, float* sum, float* comp, float* isum,
                           float* icomp) {
  const bool ref = g->cfg.precision == HWS_PRECISION_REFERENCE;
  const dim3 grid(unsigned(a.W / kProjectColumns), unsigned(a.nImg));
  const size_t lds = colsProjectLds(a.H, a.nLayersInPass, a.tilesY);
  const float2* tw = g->colPlan.twBackward;
  bool ok = false;
  switch (a.H) {
#define HWS_COLS_PROJECT(NN)                                                                    \
  case NN:                                                                                      \
    if (ref && cplx)                                                                            \
      hipLaunchKernelGGL((fftColsProjectKernel<NN, true, true>), grid,                          \
                         dim3(kProjectColumns * NN / 16), lds, g->stream, a, layers, tw, sum,   \
                         comp, isum, icomp);                                                    \
    else if (ref)                                                                               \
      hipLaunchKernelGGL((fftColsProjectKernel<NN, true, false>), grid,                         \
                         dim3(kProjectColumns * NN / 16), lds, g->stream, a, layers, tw, sum,   \
                         comp, isum, icomp);                                                    \
    else if (cplx)                                                                              \
      hipLaunchKernelGGL((fftColsProjectKernel<NN, false, true>), grid,                         \
                         dim3(kProjectColumns * NN / 16), lds, g->stream, a, layers, tw, sum,   \
                         comp, isum, icomp);                                                    \
    else                                                                                        \
      hipLaunchKernelGGL((fftColsProjectKernel<NN, false, false>), grid,                        \
                         dim3(kProjectColumns * NN / 16), lds, g->stream, a, layers, tw, sum,   \
                         comp, isum, icomp);                                                    \
    ok = true;                                                                                  \
    break;
    HWS_COLS_PROJECT(256)
    HWS_COLS_PROJECT(512)
    HWS_COLS_PROJECT(1024)
    HWS_COLS_PROJECT(2048)
    HWS_COLS_PROJECT(4096)
#undef HWS_COLS_PROJECT
    default: break;
  }
  return ok;
}

// Waves that the model rows pass is spread over: two rounds of the two waves a
// SIMD holds.
constexpr size_t kModelWaves = 4096;

// Every layer of a group per workgroup, the model and n' read and computed
// once.
bool launchModelLayersPow2(hws_gridder* g, float2* data, int nbatch, const float2* tw,
                           const ModelSource& model, const FftSparse& sparse) {
  const int W = g->W, H = g->H;
  const bool ref = model.precision == HWS_PRECISION_REFERENCE;
  const bool cplx = model.cplx != 0;
  // Small images do not fill the chip with one workgroup per row block
  // (1024^2: one wave per SIMD), so the layers are dealt to as many groups of
  // workgroups as bring kModelWaves waves, in groups of at least two layers (a
  // group computes its rows' n' anew, about the time of one layer).
  const size_t waves = size_t(H / kModelRows) * size_t((kModelRows * W / 16 + 63) / 64);
  const int groups = int(std::min<size_t>(size_t(nbatch + 1) / 2,
                                          std::max<size_t>(1, kModelWaves / waves)));
  const int per = (nbatch + groups - 1) / groups;
  const dim3 mgrid(H / kModelRows, (nbatch + per - 1) / per);
  bool ok = false;
  switch (W) {
#define HWS_MODEL_LAYERS(NN)                                                                   \
  case NN:                                                                                     \
    if (ref && cplx)                                                                           \
      hipLaunchKernelGGL((fftRowsModelLayersKernel<NN, true, true>), mgrid,                    \
                         dim3(kModelRows * NN / 16), 0, g->stream, data, H, nbatch, per,   \
                         tw, model, sparse.colNeed, sparse.tshift);                       \
    else if (ref)                                                                              \
      hipLaunchKernelGGL((fftRowsModelLayersKernel<NN, true, false>), mgrid,                   \
                         dim3(kModelRows * NN / 16), 0, g->stream, data, H, nbatch, per,   \
                         tw, model, sparse.colNeed, sparse.tshift);                       \
    else if (cplx)                                                                             \
      hipLaunchKernelGGL((fftRowsModelLayersKernel<NN, false, true>), mgrid,                   \
                         dim3(kModelRows * NN / 16), 0, g->stream, data, H, nbatch, per,   \
                         tw, model, sparse.colNeed, sparse.tshift);                       \
    else                                                                                       \
      hipLaunchKernelGGL((fftRowsModelLayersKernel<NN, false, false>), mgrid,                  \
                         dim3(kModelRows * NN / 16), 0, g->stream, data, H, nbatch, per,   \
                         tw, model, sparse.colNeed, sparse.tshift);                       \
    ok = true;                                                                                 \
    break;
    HWS_MODEL_LAYERS(256)
    HWS_MODEL_LAYERS(512)
    HWS_MODEL_LAYERS(1024)
    HWS_MODEL_LAYERS(2048)
    HWS_MODEL_LAYERS(4096)
#undef HWS_MODEL_LAYERS
    default: break;
  }
  return ok;
}

}  // namespace hws
