// The blocked layout's layer transforms at sizes without a compile-time
// kernel: mixed-radix Stockham stages with runtime radices and their sparse
// modes (their fusions are in hws_fft_generic_fused.hip).
#include "hws_fft_generic.h"

namespace hws {

namespace {

template <int SIGN, int MODE, bool REF, int L>
__global__ void __launch_bounds__(1024)
fftRowsBlockedGenericKernel(float2* __restrict__ data, int W, int H,
                            unsigned long long radices, const float2* __restrict__ tw,
                            GenericSparseArgs sp, ModelSource ms) {
  extern __shared__ float2 lds[];
  const int tid = threadIdx.x, nthr = blockDim.x;
  const int rblk = sharedSegmentBlock<L>(int(blockIdx.x), int(gridDim.x));
  const int r0 = rblk * L;                // rows of this workgroup: 4, 2 or 1 of a row block
  const int f0 = r0 & 3;                  // their position in the four-row block
  const int layer = sp.layer0 + int(blockIdx.y);
  const int ty = r0 >> sp.tshift;
  const size_t rowBase = (size_t(layer) * sp.tilesY + ty) * sp.tilesX;
  if (MODE == 1) {
    int any = 0;
    for (int t = tid; t < sp.tilesX; t += nthr) any |= bitAt(sp.bits, rowBase + t);
    if (!__syncthreads_or(any)) return;
  }
  float2* base = data + size_t(blockIdx.y) * size_t(W) * size_t(H) + size_t(r0 >> 2) * 4 * W + f0;
  const double w = MODE == 2 ? layerToW(ms.map, ms.layer0 + int(blockIdx.y)) : 0.0;
  auto load = [&](int, int x, int f) -> float2 {
    if (MODE == 2) return modelCell<REF>(ms, w, x, r0 + f, W, H);
    if (MODE == 1 && !bitAt(sp.bits, rowBase + (x >> sp.tshift))) return make_float2(0.0f, 0.0f);
    return base[size_t(x) * 4 + f];
  };
  auto store = [&](int, int x, int f, float2 v) { base[size_t(x) * 4 + f] = v; };
  blockedRtFft<SIGN, L>(lds, W, radices, tw, tid, nthr, load, store);
}

template <int SIGN, int MODE, int L>
__global__ void __launch_bounds__(1024)
fftColsBlockedGenericKernel(float2* __restrict__ data, int W, int H, int nColBlocks,
                            unsigned long long radices, const float2* __restrict__ tw,
                            GenericSparseArgs sp) {
  extern __shared__ float2 lds[];
  const int tid = threadIdx.x, nthr = blockDim.x;
  int blk = blockIdx.x;
  // (the sparse forward mode keeps the natural order: its live column blocks
  // lie near the uv origin, at both ends of the row)
  if (MODE != 2 && (nColBlocks & 7) == 0)
    blk = (blk & 7) * (nColBlocks >> 3) + (blk >> 3);
  else if (MODE == 2)
    blk = sharedSegmentBlock<L>(blk, nColBlocks);
  const int layer = sp.layer0 + int(blockIdx.y);
  const int c0 = blk * L;  // columns of this workgroup: 4, 2 or 1
  const int tx = c0 >> sp.tshift;
  // MODE 1: bit (layer, tile row); MODE 2: bit (layer, tile row, this tile column)
  auto live = [&](int y) -> bool {
    const int ty = y >> sp.tshift;
    if (MODE == 1) return bitAt(sp.bits, size_t(layer) * sp.tilesY + ty);
    return bitAt(sp.bits, (size_t(layer) * sp.tilesY + ty) * sp.tilesX + tx);
  };
  if (MODE == 2) {
    int any = 0;
    for (int t = tid; t < sp.tilesY; t += nthr) any |= live(t << sp.tshift);
    if (!__syncthreads_or(any)) return;
  }
  float2* base = data + size_t(blockIdx.y) * size_t(W) * size_t(H) + size_t(c0) * 4;
  // element (y, column c0 + f): row block y >> 2, row y & 3 in it
  auto addr = [&](int y, int f) { return size_t(y >> 2) * W * 4 + size_t(f) * 4 + (y & 3); };
  auto load = [&](int, int y, int f) -> float2 {
    if (MODE == 1 && !live(y)) return make_float2(0.0f, 0.0f);
    return base[addr(y, f)];
  };
  auto store = [&](int, int y, int f, float2 v) {
    if (MODE == 2 && !live(y)) return;
    base[addr(y, f)] = v;
  };
  blockedRtFft<SIGN, L>(lds, H, radices, tw, tid, nthr, load, store);
}

template <int SIGN, int MODE, bool REF>
void launchRowsGeneric(int threads, int lines, dim3 grid, size_t lds, hipStream_t st,
                       float2* data, int W, int H, unsigned long long rad, const float2* tw,
                       GenericSparseArgs sp, ModelSource ms) {
  if (lines == 4)
    hipLaunchKernelGGL((fftRowsBlockedGenericKernel<SIGN, MODE, REF, 4>), grid, dim3(threads),
                       lds, st, data, W, H, rad, tw, sp, ms);
  else if (lines == 2)
    hipLaunchKernelGGL((fftRowsBlockedGenericKernel<SIGN, MODE, REF, 2>), grid, dim3(threads),
                       lds, st, data, W, H, rad, tw, sp, ms);
  else
    hipLaunchKernelGGL((fftRowsBlockedGenericKernel<SIGN, MODE, REF, 1>), grid, dim3(threads),
                       lds, st, data, W, H, rad, tw, sp, ms);
}

template <int SIGN, int MODE>
void launchColsGeneric(int threads, int lines, dim3 grid, size_t lds, hipStream_t st,
                       float2* data, int W, int H, int nColBlocks, unsigned long long rad,
                       const float2* tw, GenericSparseArgs sp) {
  if (lines == 4)
    hipLaunchKernelGGL((fftColsBlockedGenericKernel<SIGN, MODE, 4>), grid, dim3(threads), lds,
                       st, data, W, H, nColBlocks, rad, tw, sp);
  else if (lines == 2)
    hipLaunchKernelGGL((fftColsBlockedGenericKernel<SIGN, MODE, 2>), grid, dim3(threads), lds,
                       st, data, W, H, nColBlocks, rad, tw, sp);
  else
    hipLaunchKernelGGL((fftColsBlockedGenericKernel<SIGN, MODE, 1>), grid, dim3(threads), lds,
                       st, data, W, H, nColBlocks, rad, tw, sp);
}

// LDS a runtime-radix workgroup may take (the device's 160 KiB per workgroup,
// less room for the kernels' static arrays).
constexpr size_t kGenericLdsBytes = size_t(152) * 1024;

// log2 of the lines (rows or columns) a runtime-radix workgroup of the
// blocked layout transforms: the four of a row block where two such
// workgroups fit the LDS of a CU and the plan the threads, else two, else
// one; -1 if one does not fit.
int genericLinesShift(const FftPlan& plan, int force) {
  auto fits = [&](int lines) {
    return blockedGenericLds(lines, plan.n) <= kGenericLdsBytes &&
           threadsFor(plan, lines) != 0;
  };
  if (force && fits(force)) return force == 4 ? 2 : force == 2 ? 1 : 0;
  // (four lines only while two workgroups fit a CU: at 3072, four lines in
  // one workgroup per CU took 26.6 / 19.5 ms per step for the backward /
  // forward transforms, two lines in three 25.1 / 18.5; one line, whose
  // workgroups read a quarter of each segment, 27.9 / 28.8)
  if (fits(4) && blockedGenericLds(4, plan.n) <= kGenericLdsBytes / 2) return 2;
  if (fits(2)) return 1;
  return fits(1) ? 0 : -1;
}
}  // namespace

bool blockedGenericLineFits(int n) { return blockedGenericLds(1, n) <= kGenericLdsBytes; }

bool blockedGenericFits(const hws_gridder* g) {
  return genericLinesShift(g->rowPlan, 0) >= 0 && genericLinesShift(g->colPlan, 0) >= 0;
}

// The 2-D transforms of fft2d with runtime radices (sparse modes as for the
// compile-time kernels).
hws_status fft2dGeneric(hws_gridder* g, float2* data, int nbatch, int sign,
                        const FftSparse* sparse, const ModelSource* model) {
  const int W = g->W, H = g->H;
  const float2* twRow = sign > 0 ? g->rowPlan.twBackward : g->rowPlan.twForward;
  const float2* twCol = sign > 0 ? g->colPlan.twBackward : g->colPlan.twForward;
  // four rows (columns) per workgroup where they fit the LDS, else two, else one
  const int rbShift = genericLinesShift(g->rowPlan, g->fftLines);
  const int cbShift = genericLinesShift(g->colPlan, g->fftLines);
  if (rbShift < 0 || cbShift < 0)
    return setLastError(g, HWS_ERR_UNSUPPORTED, "transform does not fit one workgroup");
  const int tr = threadsFor(g->rowPlan, 1 << rbShift), tc = threadsFor(g->colPlan, 1 << cbShift);
  const int rl = 1 << rbShift, cl = 1 << cbShift;
  const size_t ldsR = blockedGenericLds(rl, W), ldsC = blockedGenericLds(cl, H);
  const unsigned long long radR = packRadices(g->rowPlan), radC = packRadices(g->colPlan);
  const int nColBlocks = W >> cbShift;
  GenericSparseArgs rs{}, cs{};
  ModelSource msrc{};
  if (sparse) {
    rs.layer0 = cs.layer0 = sparse->layer0;
    rs.tilesY = cs.tilesY = sparse->tilesY;
    rs.tshift = cs.tshift = sparse->tshift;
    rs.tilesX = cs.tilesX = g->plan.tilesX;
    if (sign > 0) {
      rs.bits = sparse->occ;
      cs.bits = sparse->rowLive;
    } else {
      cs.bits = sparse->occ;  // the need bits
    }
  }
  if (model) msrc = *model;
  const dim3 gr(H >> rbShift, nbatch), gc(nColBlocks, nbatch);
  hipStream_t st = g->stream;
  if (sign > 0) {
    if (sparse) {
      launchRowsGeneric<+1, 1, false>(tr, rl, gr, ldsR, st, data, W, H, radR, twRow, rs, msrc);
      // (rowsOnly: the columns pass runs fused with the projection)
      if (!sparse->rowsOnly)
        launchColsGeneric<+1, 1>(tc, cl, gc, ldsC, st, data, W, H, nColBlocks, radC, twCol, cs);
    } else {
      launchRowsGeneric<+1, 0, false>(tr, rl, gr, ldsR, st, data, W, H, radR, twRow, rs, msrc);
      launchColsGeneric<+1, 0>(tc, cl, gc, ldsC, st, data, W, H, nColBlocks, radC, twCol, cs);
    }
  } else {
    // (the mixed precision: the reference precision's terms leave no registers
    // for the cells it keeps)
    if (model && sparse && sparse->colNeed && fusedModelRows(W, H) &&
        model->precision != HWS_PRECISION_REFERENCE)
      launchModelLayersGeneric(tr, rl, dim3(H >> rbShift), ldsR, st, data, W, H, nbatch, radR,
                               twRow, msrc, sparse->colNeed, sparse->tshift);
    else if (model && model->precision == HWS_PRECISION_REFERENCE)
      launchRowsGeneric<-1, 2, true>(tr, rl, gr, ldsR, st, data, W, H, radR, twRow, rs, msrc);
    else if (model)
      launchRowsGeneric<-1, 2, false>(tr, rl, gr, ldsR, st, data, W, H, radR, twRow, rs, msrc);
    else
      launchRowsGeneric<-1, 0, false>(tr, rl, gr, ldsR, st, data, W, H, radR, twRow, rs, msrc);
    if (sparse)
      launchColsGeneric<-1, 2>(tc, cl, gc, ldsC, st, data, W, H, nColBlocks, radC, twCol, cs);
    else
      launchColsGeneric<-1, 0>(tc, cl, gc, ldsC, st, data, W, H, nColBlocks, radC, twCol, cs);
  }
  return checkHip(g, hipGetLastError(), "fft blocked generic launch");
}

}  // namespace hws
