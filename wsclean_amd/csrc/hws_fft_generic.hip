// The blocked layout's layer transforms at sizes without a compile-time
// kernel: mixed-radix Stockham stages with runtime radices, their sparse modes
// and their fusions with the projection and the model image.
#include "hws_fft_device.h"

namespace hws {

namespace {

// Blocked layout at sizes without a compile-time kernel (any 7-smooth size
// with W and H multiples of 4): one workgroup per 4 rows (row pass) or 4
// columns (column pass), read and written as whole 128-byte segments of the
// blocked layout (two rows or columns, 64-byte segments, where four do not
// fit the LDS), by the mixed-radix stages: the first reads memory, the middle
// ones exchange through the lines interleaved in LDS, the last writes memory.
// The sparse modes mirror the compile-time kernels:
//   rows MODE 1 (backward): only tiles with samples are read (bits: the
//     occupancy of (layer, tile), sp.occ); a row block without any is
//     skipped (not written); MODE 2 (forward): the input is computed from the
//     model image (ms);
//   columns MODE 1 (backward): tile rows without samples (sp.rowLive) read as
//     zero; MODE 2 (forward): only the tiles degridding reads (sp.occ = the
//     need bits) are written, and a column block without any is skipped.
struct GenericSparseArgs {
  const uint32_t* bits;
  int layer0, tilesX, tilesY, tshift;
};

__device__ __forceinline__ bool bitAt(const uint32_t* bits, size_t b) {
  return (bits[b >> 5] >> (b & 31)) & 1u;
}

// LDS position of value i of the interleaved lines of a blocked runtime-radix
// workgroup (element e of line f is value e * L + f): one pad value after
// every 16, so that the first stage's writes (stride R * L values across the
// lanes) fall in distinct banks.
__device__ __forceinline__ int ipad(int i) { return i + (i >> 4); }

// LDS bytes of L interleaved lines of length n.
__host__ __device__ constexpr size_t blockedGenericLds(int L, int n) {
  return (size_t(L) * n + (size_t(L) * n >> 4) + 1) * sizeof(float2);
}

// One Stockham stage of radix R over the L interleaved lines of length n
// (butterfly t: line f = t % L, index b = t / L, so the lanes of a wave read
// and write the L lines of consecutive positions together). Butterfly b reads
// x[b + r*B] (B = n/R), applies twiddle w^(jm*r) with jm = b % ns, and writes
// y[(b/ns)*ns*R + jm + r*ns]. The first stage (ns == 1) reads its inputs with
// load(slot, pos, f) instead of from LDS (slot = q * R + r, this thread's
// q-th butterfly's r-th input, below kMaxValues) and needs no barrier before
// its writes; the last one writes its outputs with store(slot, pos, f, v)
// instead of to LDS.
template <int SIGN, int R, int L, bool FIRST, bool LAST, class Load, class Store>
__device__ __forceinline__ void blockedRtStage(float2* lds, int n, int ns,
                                               const float2* __restrict__ tw, int tid, int nthr,
                                               const Load& load, const Store& store) {
  constexpr int kBatches = kMaxValues / R;
  constexpr int LS = L == 4 ? 2 : L == 2 ? 1 : 0;
  static_assert(L == 1 || L == 2 || L == 4, "lines");
  // (an opaque tid keeps the compiler from hoisting the batch indices of
  // every radix out of the stage loop, which keeps them all live)
  asm volatile("" : "+v"(tid));
  const int B = n / R;
  const int total = B * L;
  const int twStep = n / (ns * R);
  const UniformDiv byNs = uniformDiv(ns);
  float2 v[kBatches][R];
#pragma unroll
  for (int q = 0; q < kBatches; ++q) {
    const int t = tid + q * nthr;
    if (t < total) {
      const int f = t & (L - 1), b = t >> LS;
      const int jm = FIRST ? 0 : b - divBy(b, byNs) * ns;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int pos = b + r * B;
        float2 x;
        if (FIRST) {
          x = load(q * R + r, pos, f);
        } else {
          x = lds[ipad(pos * L + f)];
          if (r != 0 && jm != 0) x = cmul(x, tw[jm * r * twStep]);
        }
        v[q][r] = x;
      }
    }
  }
  if (!FIRST) __syncthreads();  // every read of this stage precedes its writes
#pragma unroll
  for (int q = 0; q < kBatches; ++q) {
    const int t = tid + q * nthr;
    if (t < total) {
      const int f = t & (L - 1), b = t >> LS;
      Butterfly<SIGN, R>::run(v[q]);
      const int bq = FIRST ? b : divBy(b, byNs);
      const int idxD = bq * ns * R + (b - bq * ns);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int pos = idxD + r * ns;
        if (LAST)
          store(q * R + r, pos, f, v[q][r]);
        else
          lds[ipad(pos * L + f)] = v[q][r];
      }
    }
  }
  if (!LAST) __syncthreads();
}

template <int SIGN, int L, bool FIRST, bool LAST, class Load, class Store>
__device__ __forceinline__ void blockedRtStageR(int R, float2* lds, int n, int ns,
                                                const float2* __restrict__ tw, int tid, int nthr,
                                                const Load& load, const Store& store) {
  switch (R) {
#define HWS_RT_STAGE(RR)                                                                    \
  case RR:                                                                                  \
    blockedRtStage<SIGN, RR, L, FIRST, LAST>(lds, n, ns, tw, tid, nthr, load, store);       \
    break;
    HWS_RT_STAGE(16)
    HWS_RT_STAGE(8)
    HWS_RT_STAGE(4)
    HWS_RT_STAGE(2)
    HWS_RT_STAGE(3)
    HWS_RT_STAGE(5)
    HWS_RT_STAGE(7)
#undef HWS_RT_STAGE
    default: break;
  }
}

// The whole transform of the L lines: the first stage from load, the middle
// stages through LDS, the last stage to store (radices packed 4 bits per
// stage, 16 packed as 1).
template <int SIGN, int L, class Load, class Store>
__device__ __forceinline__ void blockedRtFft(float2* lds, int n, unsigned long long radices,
                                             const float2* __restrict__ tw, int tid, int nthr,
                                             const Load& load, const Store& store) {
  auto radixOf = [](unsigned long long rad) {
    const int code = int(rad & 15ull);
    return code == 1 ? 16 : code;
  };
  int R = radixOf(radices);
  radices >>= 4;
  auto toLds = [](int, int, int, float2) {};
  auto fromLds = [](int, int, int) { return make_float2(0.0f, 0.0f); };
  if (radices == 0ull) {  // a single stage: memory to memory
    blockedRtStageR<SIGN, L, true, true>(R, lds, n, 1, tw, tid, nthr, load, store);
    return;
  }
  blockedRtStageR<SIGN, L, true, false>(R, lds, n, 1, tw, tid, nthr, load, toLds);
  int ns = R;
  for (;;) {
    R = radixOf(radices);
    radices >>= 4;
    if (radices == 0ull) break;
    blockedRtStageR<SIGN, L, false, false>(R, lds, n, ns, tw, tid, nthr, fromLds, toLds);
    ns *= R;
  }
  blockedRtStageR<SIGN, L, false, true>(R, lds, n, ns, tw, tid, nthr, fromLds, store);
}

// Fewer than four lines per workgroup: the workgroups of a four-line block
// read and write parts of the same 32-byte (rows) or 128-byte (columns)
// segments. The hardware sends workgroup b to XCD b % 8, so within every
// 8 * P workgroups (P = 4 / L parts per block) b, b + 8, ... are given the
// parts of one block: they run on the same XCD at about the same time and
// share its L2.
template <int L>
__device__ __forceinline__ int sharedSegmentBlock(int b, int nBlocks) {
  constexpr int P = 4 / L, G = 8 * P;
  if (P == 1 || nBlocks % G != 0) return b;
  return (b / G) * G + (b & 7) * P + ((b >> 3) & (P - 1));
}

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
// column)). grid (H / L).
template <bool REF, bool CPLX, int L>
__global__ void __launch_bounds__(1024)
fftRowsModelLayersGenericKernel(float2* __restrict__ data, int W, int H, int nbatch,
                                unsigned long long radices, const float2* __restrict__ tw,
                                ModelSource ms, const uint32_t* __restrict__ colNeed,
                                int tshift) {
  extern __shared__ float2 lds[];
  const int tid = threadIdx.x, nthr = blockDim.x;
  const int rblk = sharedSegmentBlock<L>(int(blockIdx.x), int(gridDim.x));
  const int r0 = rblk * L;
  const size_t HW = size_t(W) * H;
  float2* rowBase = data + size_t(r0 >> 2) * 4 * W + (r0 & 3);
  const int tilesX = W >> tshift;
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
    double v = nPrimeSeries(l, m);
    if (REF) v = double(float(v));
    np[slot] = v;
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
#pragma unroll 1
  for (int b = 0; b < nbatch; ++b) {
    const int layer = ms.layer0 + b;
    const double w = layerToW(ms.map, layer);
    float2* base = rowBase + size_t(b) * HW;
    const size_t cbit = size_t(layer) * tilesX;
    auto load = [&](int slot, int, int) -> float2 {
      return modelTerm<REF>(re[slot], CPLX ? imv[slot] : 0.0f, CPLX, w, np[slot]);
    };
    auto store = [&](int, int x, int f, float2 v) {
      const size_t bit = cbit + size_t(x >> tshift);
      if ((colNeed[bit >> 5] >> (bit & 31)) & 1u) streamStore(&base[size_t(x) * 4 + f], v);
    };
    blockedRtFft<-1, L>(lds, W, radices, tw, tid, nthr, load, store);
    __syncthreads();  // the last stage's LDS reads precede the next layer's writes
  }
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

// Backward columns pass fused with the projection at the runtime-radix
// sizes (fftColsProjectKernel at the power-of-two sizes): a workgroup owns
// one column of one image and transforms it layer after layer, in the pass's
// layer order; each transformed cell is rotated by its layer's w term and
// added (Kahan) to its pixel's sums, which stay in registers with the
// pixel's n' (the cells of the last stage's slots). Cells of tile rows
// without samples read as zero. Every term is computed and added as
// projectKernel computes and adds it. grid (W / 1, images of the kind);
// dynamic LDS: the transform buffer, then the row bits of the pass's layers.
template <bool REF, bool CPLX>
__global__ void __launch_bounds__(512)
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

void launchModelLayersGeneric(int threads, int lines, dim3 grid, size_t lds, hipStream_t st,
                              float2* data, int W, int H, int nbatch, unsigned long long rad,
                              const float2* tw, const ModelSource& ms, const uint32_t* colNeed,
                              int tshift) {
  const bool cplx = ms.cplx != 0;
#define HWS_MODEL_GENERIC(C, LL)                                                                \
  hipLaunchKernelGGL((fftRowsModelLayersGenericKernel<false, C, LL>), grid, dim3(threads), lds,  \
                     st, data, W, H, nbatch, rad, tw, ms, colNeed, tshift)
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

namespace {
// The runtime-radix fused kernel: one column per workgroup of at most 512
// threads; its LDS is the transform buffer and the row bits.
size_t colsProjectGenericLds(int H, int nLayersInPass, int tilesY) {
  const size_t words = (size_t(nLayersInPass) * tilesY + 31) / 32;
  return blockedGenericLds(1, H) + words * sizeof(uint32_t);
}
}  // namespace

bool colsProjectGenericSupported(const hws_gridder* g, int nLayersInPass, size_t maxLds) {
  const int t = threadsFor(g->colPlan, 1);
  return t != 0 && t <= 512 &&
         colsProjectGenericLds(g->H, nLayersInPass, g->H / g->plan.tileSize) <= maxLds;
}

void launchColsProjectGeneric(hws_gridder* g, const ColsProjectArgs& a, bool cplx,
                              const float2* layers, float* sum, float* comp, float* isum,
                              float* icomp) {
  const bool ref = g->cfg.precision == HWS_PRECISION_REFERENCE;
  const dim3 grid(unsigned(a.W), unsigned(a.nImg));
  const int threads = threadsFor(g->colPlan, 1);
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
    rs.tilesX = cs.tilesX = W >> sparse->tshift;
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
    // (the mixed precision: the reference precision's FP64 sincos leaves no
    // registers for the cells it keeps)
    if (model && sparse && sparse->colNeed && model->precision != HWS_PRECISION_REFERENCE)
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
