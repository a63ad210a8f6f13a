// LDS-staged mixed-radix Stockham FFT for the per-layer 2-D transforms
// (the reference runs fftw[f]_plan_dft_2d per layer,
// gridding/wstackinggridder.cpp:200-239, 282-321).
//
// A 2-D transform of a batch of H x W layers is two launches:
//   rows:    one workgroup per (row block, layer); a row of W complex values
//            is loaded with coalesced float2 loads, transformed through the
//            Stockham stages in LDS, and written back in place;
//   columns: one workgroup per (column block of Bc columns, layer); the Bc
//            columns are gathered into LDS as [Bc][H+1] (padded to spread
//            banks), transformed, and scattered back. Column blocks that
//            share 128-byte lines are mapped onto the same XCD so that they
//            share its L2.
// Each Stockham stage reads its R inputs into registers, synchronises, and
// writes its R outputs in natural (autosorted) order, so one LDS buffer per
// transform suffices. Radices 8, 4, 2, 3, 5, 7.
#include "hws_fft_device.h"

#include <algorithm>
#include <cmath>

namespace hws {

namespace {

// One Stockham stage of radix R over nfft transforms of length n stored at
// buf + f * pitch (element e at lp(e)). Butterfly b of transform f reads
// x[b + r*B] (B = n/R), applies twiddle w^(jm*r) with jm = b % ns, and writes
// y[(b/ns)*ns*R + jm + r*ns].
template <int SIGN, int R>
__device__ __forceinline__ void stockhamStage(float2* buf, int n, int pitch,
                                              int nfft, int ns,
                                              const float2* __restrict__ tw,
                                              int tid, int nthr) {
  constexpr int kBatches = kMaxValues / R;
  // The batch indices below depend only on (tid, n, R, nthr), so the compiler
  // would hoist those of every radix out of the stage loop of fftLds and keep
  // them all live (208 VGPRs, spills at 1024 threads); an opaque tid makes
  // each stage compute its own.
  asm volatile("" : "+v"(tid));
  const int B = n / R;
  const int total = B * nfft;
  const int twStep = n / (ns * R);
  const UniformDiv byB = uniformDiv(B), byNs = uniformDiv(ns);
  float2 v[kBatches][R];
#pragma unroll
  for (int q = 0; q < kBatches; ++q) {
    const int t = tid + q * nthr;
    if (t < total) {
      const int f = divBy(t, byB), b = t - f * B;
      const int jm = b - divBy(b, byNs) * ns;
      const float2* x = buf + f * pitch;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        float2 val = x[lp(b + r * B)];
        if (r != 0 && jm != 0) val = cmul(val, tw[jm * r * twStep]);
        v[q][r] = val;
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < kBatches; ++q) {
    const int t = tid + q * nthr;
    if (t < total) {
      const int f = divBy(t, byB), b = t - f * B;
      Butterfly<SIGN, R>::run(v[q]);
      const int bq = divBy(b, byNs), jm = b - bq * ns;
      const int idxD = bq * ns * R + jm;
      float2* y = buf + f * pitch;
#pragma unroll
      for (int r = 0; r < R; ++r) y[lp(idxD + r * ns)] = v[q][r];
    }
  }
  __syncthreads();
}

// Stage radices are packed 4 bits per stage (stage 0 lowest) so that the
// per-stage dispatch reads a scalar rather than an indexed argument array.
// Lines are stored padded (element e of line f at buf[f * pitch + lp(e)],
// pitch >= ldsPitch(n)).
template <int SIGN>
__device__ __forceinline__ void fftLds(float2* buf, int pitch, int nfft, int n,
                       unsigned long long radices, const float2* tw, int tid,
                       int nthr) {
  int ns = 1;
  while (radices != 0ull) {
    const int code = int(radices & 15ull);
    const int R = code == 1 ? 16 : code;  // (radix 16 is packed as 1)
    radices >>= 4;
    switch (R) {
      case 16: stockhamStage<SIGN, 16>(buf, n, pitch, nfft, ns, tw, tid, nthr); break;
      case 8: stockhamStage<SIGN, 8>(buf, n, pitch, nfft, ns, tw, tid, nthr); break;
      case 4: stockhamStage<SIGN, 4>(buf, n, pitch, nfft, ns, tw, tid, nthr); break;
      case 2: stockhamStage<SIGN, 2>(buf, n, pitch, nfft, ns, tw, tid, nthr); break;
      case 3: stockhamStage<SIGN, 3>(buf, n, pitch, nfft, ns, tw, tid, nthr); break;
      case 5: stockhamStage<SIGN, 5>(buf, n, pitch, nfft, ns, tw, tid, nthr); break;
      case 7: stockhamStage<SIGN, 7>(buf, n, pitch, nfft, ns, tw, tid, nthr); break;
      default: break;
    }
    ns *= R;
  }
}

// ---- power-of-two lengths: every index is a compile-time shift or mask.
// Stage radices are 8 while the remaining length allows, then 4, then 2.
template <int SIGN, int R, int N, int NS, int NT, int NFFT>
__device__ __forceinline__ void pow2Stage(float2* buf, int pitch, int nfft,
                                          const float2* __restrict__ tw, int tid) {
  constexpr int B = N / R;
  constexpr int TOTAL = B * NFFT;
  constexpr int BATCHES = (TOTAL + NT - 1) / NT;
  constexpr int TWSTEP = N / (NS * R);
  float2 v[BATCHES][R];
#pragma unroll
  for (int q = 0; q < BATCHES; ++q) {
    const int t = tid + q * NT;
    const int f = t / B, b = t % B;
    if (f < nfft) {
      const int jm = b % NS;
      const float2* x = buf + f * pitch;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        float2 val = x[b + r * B];
        if (NS > 1 && r != 0) val = cmul(val, tw[jm * r * TWSTEP]);
        v[q][r] = val;
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < BATCHES; ++q) {
    const int t = tid + q * NT;
    const int f = t / B, b = t % B;
    if (f < nfft) {
      Butterfly<SIGN, R>::run(v[q]);
      const int jm = b % NS;
      float2* y = buf + f * pitch + (b / NS) * NS * R + jm;
#pragma unroll
      for (int r = 0; r < R; ++r) y[r * NS] = v[q][r];
    }
  }
  __syncthreads();
}

template <int SIGN, int N, int NT, int NFFT, int NS = 1>
__device__ __forceinline__ void pow2Fft(float2* buf, int pitch, int nfft,
                                        const float2* __restrict__ tw, int tid) {
  if constexpr (NS < N) {
    constexpr int REM = N / NS;
    constexpr int R = (REM % 8 == 0) ? 8 : (REM % 4 == 0) ? 4 : 2;
    pow2Stage<SIGN, R, N, NS, NT, NFFT>(buf, pitch, nfft, tw, tid);
    pow2Fft<SIGN, N, NT, NFFT, NS * R>(buf, pitch, nfft, tw, tid);
  }
}

// grid (H / 4, nbatch): block = row block yb of layer blockIdx.y
template <int SIGN, int N>
__global__ void __launch_bounds__(N / 4)
fftRowsBlockedKernel(float2* __restrict__ data, int H, const float2* __restrict__ tw) {
  __shared__ float2 lds[4 * N + (4 * N) / 64];
  float2* g = data + size_t(blockIdx.y) * size_t(N) * size_t(H) + size_t(blockIdx.x) * 4 * N;
  blockedFft<SIGN, N, true>(lds, g, N, tw, threadIdx.x);
}

// Rows pass of a forward transform whose layers are computed from the model
// image on the fly (the layer memory is written by this pass only): grid
// (H / 4, nbatch), batch entry b = layer ms.layer0 + b.
template <int SIGN, int N, bool REF>
__global__ void __launch_bounds__(N / 4)
fftRowsFromModelKernel(float2* __restrict__ data, int H, int nbatch,
                       const float2* __restrict__ tw, ModelSource ms) {
  __shared__ float2 lds[4 * N + (4 * N) / 64];
#pragma unroll 1
  for (int li = 0; li < modelLayers<REF>(); ++li) {
    const int bi = int(blockIdx.y) * modelLayers<REF>() + li;
    if (bi >= nbatch) break;  // workgroup-uniform
    // the empty asm gives the model pointers, pixel scale, twiddle table and
    // thread index new values each iteration: nothing derived from them is
    // held across the layers (the registers of one layer's transform are
    // all the workgroup size allows)
    ModelSource msl = ms;
    const float2* twl = tw;
    int tid = int(threadIdx.x);
    asm volatile("" : "+s"(msl.re), "+s"(msl.im), "+s"(msl.dl), "+s"(twl), "+v"(tid));
    float2* g = data + size_t(bi) * size_t(N) * size_t(H) + size_t(blockIdx.x) * 4 * N;
    const double w = layerToW(ms.map, ms.layer0 + bi);
    blockedFft<SIGN, N, true, 1, REF ? 2 : 1>(lds, g, N, twl, tid, nullptr, 0, true, &msl, w,
                                              int(blockIdx.x) * 4, H);
  }
}

// The same over layers whose uv tiles without samples were never written:
// occ holds one bit per (layer, tile row, tile) bin of the layer set
// (bin = (layer * tilesY + ty) * tilesX + tx), layer0 is the layer of batch
// entry 0, the tile edge is 1 << tshift (>= 4, so the four rows of a row
// block share one tile row).
template <int SIGN, int N>
__global__ void __launch_bounds__(N / 4)
fftRowsBlockedSparseKernel(float2* __restrict__ data, int H, const float2* __restrict__ tw,
                           const uint32_t* __restrict__ occ, int layer0, int tilesY,
                           int tshift) {
  __shared__ float2 lds[4 * N + (4 * N) / 64];
  __shared__ unsigned char live[N / 4];
  const int tilesX = N >> tshift;
  const int ty = (int(blockIdx.x) * 4) >> tshift;
  const size_t base = (size_t(layer0 + int(blockIdx.y)) * tilesY + ty) * tilesX;
  int any = 0;
  for (int t = threadIdx.x; t < tilesX; t += blockDim.x) {
    const size_t b = base + t;
    live[t] = (occ[b >> 5] >> (b & 31)) & 1u;
    any |= live[t];
  }
  float2* g = data + size_t(blockIdx.y) * size_t(N) * size_t(H) + size_t(blockIdx.x) * 4 * N;
  // no tile of the row block holds samples: its transform is zero, which the
  // columns pass knows from the same bits (it is not written)
  if (!__syncthreads_or(any)) return;
  blockedFft<SIGN, N, true>(lds, g, N, tw, threadIdx.x, live, tshift, true);
}

// Columns pass of a backward transform after fftRowsBlockedSparseKernel:
// rows of a tile row without samples were not written and read as zero.
// rowLive holds one bit per (layer, tile row) (bit = layer * tilesY + ty).
template <int SIGN, int N>
__global__ void __launch_bounds__(N / 4)
fftColsBlockedRowSparseKernel(float2* __restrict__ data, int W, const float2* __restrict__ tw,
                              const uint32_t* __restrict__ rowLive, int layer0, int tilesY,
                              int tshift) {
  __shared__ float2 lds[4 * N + (4 * N) / 64];
  __shared__ unsigned char live[N / 4];
  const int nb = gridDim.x;
  int cb = blockIdx.x;
  if ((nb & 7) == 0) cb = (cb & 7) * (nb >> 3) + (cb >> 3);
  const size_t base = size_t(layer0 + int(blockIdx.y)) * tilesY;
  for (int t = threadIdx.x; t < tilesY; t += blockDim.x) {
    const size_t b = base + t;
    live[t] = (rowLive[b >> 5] >> (b & 31)) & 1u;
  }
  __syncthreads();
  float2* g = data + size_t(blockIdx.y) * size_t(W) * size_t(N) + size_t(cb) * 16;
  blockedFft<SIGN, N, false>(lds, g, W, tw, threadIdx.x, live, tshift, true);
}

// Columns pass of a forward transform whose output is read only in some uv
// tiles (the degridding subgrids): need holds one bit per (layer, tile) bin
// as occ does for fftRowsBlockedSparseKernel; other tiles are not written.
template <int SIGN, int N>
__global__ void __launch_bounds__(N / 4)
fftColsBlockedSparseKernel(float2* __restrict__ data, int W, const float2* __restrict__ tw,
                           const uint32_t* __restrict__ need, int layer0, int tilesY,
                           int tshift) {
  __shared__ float2 lds[4 * N + (4 * N) / 64];
  __shared__ unsigned char live[N / 4];
  // column blocks in their natural order, so consecutive workgroups (dealt
  // round-robin to the XCDs) spread over all XCDs: the column blocks with
  // needed tiles lie near the uv origin, at both ends of the row, and a
  // contiguous range per XCD would leave most XCDs without work
  const int cb = blockIdx.x;
  const int tilesX = W >> tshift;
  const int tx = (cb * 4) >> tshift;
  const size_t layerBase = size_t(layer0 + int(blockIdx.y)) * tilesY;
  int any = 0;
  for (int t = threadIdx.x; t < tilesY; t += blockDim.x) {
    const size_t b = (layerBase + t) * tilesX + tx;
    live[t] = (need[b >> 5] >> (b & 31)) & 1u;
    any |= live[t];
  }
  // no tile of the column block is read afterwards: nothing to do
  if (!__syncthreads_or(any)) return;
  float2* g = data + size_t(blockIdx.y) * size_t(W) * size_t(N) + size_t(cb) * 16;
  blockedFft<SIGN, N, false>(lds, g, W, tw, threadIdx.x, live, tshift, false);
}

// grid (W / 4, nbatch): block = columns 4*cb .. 4*cb+3 of layer blockIdx.y;
// column blocks sharing an XCD are contiguous
template <int SIGN, int N>
__global__ void __launch_bounds__(N / 4)
fftColsBlockedKernel(float2* __restrict__ data, int W, const float2* __restrict__ tw) {
  __shared__ float2 lds[4 * N + (4 * N) / 64];
  const int nb = gridDim.x;
  int cb = blockIdx.x;
  if ((nb & 7) == 0) cb = (cb & 7) * (nb >> 3) + (cb >> 3);
  float2* g = data + size_t(blockIdx.y) * size_t(W) * size_t(N) + size_t(cb) * 16;
  blockedFft<SIGN, N, false>(lds, g, W, tw, threadIdx.x);
}

// rows of length N, NFFT rows per block (the last block may hold fewer)
template <int SIGN, int N, int NT, int NFFT>
__global__ void __launch_bounds__(NT)
fftRowsPow2Kernel(float2* __restrict__ data, int H, const float2* __restrict__ tw) {
  __shared__ float2 lds[NFFT * N];
  const int tid = threadIdx.x;
  const int row0 = blockIdx.x * NFFT;
  const int nrows = min(NFFT, H - row0);
  float2* base = data + size_t(blockIdx.y) * size_t(N) * size_t(H) + size_t(row0) * N;
  const int total = nrows * N;
  for (int i = tid; i < total; i += NT) lds[i] = base[i];
  __syncthreads();
  pow2Fft<SIGN, N, NT, NFFT>(lds, N, nrows, tw, tid);
  for (int i = tid; i < total; i += NT) base[i] = lds[i];
}

// columns of length N (= H), NFFT columns per block, LDS [NFFT][N + 1]
template <int SIGN, int N, int NT, int NFFT>
__global__ void __launch_bounds__(NT)
fftColsPow2Kernel(float2* __restrict__ data, int W, int nColBlocks,
                  const float2* __restrict__ tw) {
  __shared__ float2 lds[NFFT * (N + 1)];
  const int tid = threadIdx.x;
  int blk = blockIdx.x;
  if ((nColBlocks & 7) == 0) blk = (blk & 7) * (nColBlocks >> 3) + (blk >> 3);
  const int c0 = blk * NFFT;
  const int ncols = min(NFFT, W - c0);
  float2* base = data + size_t(blockIdx.y) * size_t(W) * size_t(N) + c0;
  const int total = ncols * N;
  for (int i = tid; i < total; i += NT) {
    const int y = i / ncols, c = i - y * ncols;
    lds[c * (N + 1) + y] = base[size_t(y) * W + c];
  }
  __syncthreads();
  pow2Fft<SIGN, N, NT, NFFT>(lds, N + 1, ncols, tw, tid);
  for (int i = tid; i < total; i += NT) {
    const int y = i / ncols, c = i - y * ncols;
    base[size_t(y) * W + c] = lds[c * (N + 1) + y];
  }
}

// rows: grid (ceil(H / rowsPerBlock), nbatch); each block transforms
// rowsPerBlock consecutive rows of one layer.
template <int SIGN, int NT>
__global__ void __launch_bounds__(NT)
fftRowsKernel(float2* __restrict__ data, int W, int H, int rowsPerBlock,
              unsigned long long radices, const float2* __restrict__ tw) {
  extern __shared__ float2 lds[];
  const int tid = threadIdx.x, nthr = blockDim.x;
  const int row0 = blockIdx.x * rowsPerBlock;
  const int nrows = min(rowsPerBlock, H - row0);
  float2* base = data + size_t(blockIdx.y) * size_t(W) * size_t(H) +
                 size_t(row0) * size_t(W);
  const int pitch = ldsPitch(W);
  for (int r = 0; r < nrows; ++r)
    for (int x = tid; x < W; x += nthr) lds[r * pitch + lp(x)] = base[size_t(r) * W + x];
  __syncthreads();
  fftLds<SIGN>(lds, pitch, nrows, W, radices, tw, tid, nthr);
  for (int r = 0; r < nrows; ++r)
    for (int x = tid; x < W; x += nthr) base[size_t(r) * W + x] = lds[r * pitch + lp(x)];
}

// columns: grid (nColBlocks, nbatch); block handles columns
// [c0, c0 + bc) of one layer; LDS holds [bc][ldsPitch(H)].
template <int SIGN, int NT>
__global__ void __launch_bounds__(NT)
fftColsKernel(float2* __restrict__ data, int W, int H, int bc, int nColBlocks,
              unsigned long long radices, const float2* __restrict__ tw) {
  extern __shared__ float2 lds[];
  const int tid = threadIdx.x, nthr = blockDim.x;
  // XCD-aware remap: hardware dispatches block b to XCD b % 8; give each XCD
  // a contiguous range of column blocks so neighbours share its L2.
  int blk = blockIdx.x;
  if ((nColBlocks & 7) == 0) blk = (blk & 7) * (nColBlocks >> 3) + (blk >> 3);
  const int c0 = blk * bc;
  const int ncols = min(bc, W - c0);
  const int pitch = ldsPitch(H);
  float2* base = data + size_t(blockIdx.y) * size_t(W) * size_t(H) + c0;
  const int total = ncols * H;
  for (int i = tid; i < total; i += nthr) {
    const int y = i / ncols, c = i - y * ncols;
    lds[c * pitch + lp(y)] = base[size_t(y) * W + c];
  }
  __syncthreads();
  fftLds<SIGN>(lds, pitch, ncols, H, radices, tw, tid, nthr);
  for (int i = tid; i < total; i += nthr) {
    const int y = i / ncols, c = i - y * ncols;
    base[size_t(y) * W + c] = lds[c * pitch + lp(y)];
  }
}

// The plain (row-major) runtime-radix kernels are compiled for three launch
// bounds; a launch takes the smallest that holds its threads.
template <int SIGN>
void launchRowsPlain(int threads, dim3 grid, size_t lds, hipStream_t st, float2* data, int W,
                     int H, int rows, unsigned long long rad, const float2* tw) {
  if (threads <= 256)
    hipLaunchKernelGGL((fftRowsKernel<SIGN, 256>), grid, dim3(threads), lds, st, data, W, H, rows,
                       rad, tw);
  else if (threads <= 512)
    hipLaunchKernelGGL((fftRowsKernel<SIGN, 512>), grid, dim3(threads), lds, st, data, W, H, rows,
                       rad, tw);
  else
    hipLaunchKernelGGL((fftRowsKernel<SIGN, 1024>), grid, dim3(threads), lds, st, data, W, H,
                       rows, rad, tw);
}

template <int SIGN>
void launchColsPlain(int threads, dim3 grid, size_t lds, hipStream_t st, float2* data, int W,
                     int H, int bc, int nColBlocks, unsigned long long rad, const float2* tw) {
  if (threads <= 256)
    hipLaunchKernelGGL((fftColsKernel<SIGN, 256>), grid, dim3(threads), lds, st, data, W, H, bc,
                       nColBlocks, rad, tw);
  else if (threads <= 512)
    hipLaunchKernelGGL((fftColsKernel<SIGN, 512>), grid, dim3(threads), lds, st, data, W, H, bc,
                       nColBlocks, rad, tw);
  else
    hipLaunchKernelGGL((fftColsKernel<SIGN, 1024>), grid, dim3(threads), lds, st, data, W, H, bc,
                       nColBlocks, rad, tw);
}
}  // namespace

unsigned long long packRadices(const FftPlan& plan) {
  unsigned long long r = 0;
  for (int i = plan.nstages - 1; i >= 0; --i)
    r = (r << 4) | unsigned(plan.radix[i] == 16 ? 1 : plan.radix[i]);
  return r;
}

// Threads such that every stage's butterflies fit in kMaxValues / R batches
// per thread: the smallest power of two (whose idle lanes cost less than the
// fewer waves of a closer count: 1500 x 1260 columns 284 us an image against
// 317), or with `close` the smallest multiple of 64; 0 if more than 1024 would
// be needed.
int threadsFor(const FftPlan& plan, int nfft, bool close) {
  const int elements = nfft * plan.n;
  for (int t = 64; t <= 1024; t = close ? t + 64 : t * 2) {
    bool ok = true;
    for (int s = 0; s < plan.nstages; ++s) {
      const int R = plan.radix[s];
      if (t * (kMaxValues / R) < elements / R) ok = false;
    }
    if (ok) return std::max(t, 64);
  }
  return 0;
}
hws_status makeFftPlan(hws_gridder* g, int n, FftPlan& plan) {
  plan.n = n;
  plan.nstages = 0;
  int m = n;
  // radix 16 first, then 8 / 4 / 2, then the odd factors (fewer stages, each
  // a round trip through LDS)
  while (m % 16 == 0 && plan.nstages < kMaxFftStages) { plan.radix[plan.nstages++] = 16; m /= 16; }
  while (m % 8 == 0 && plan.nstages < kMaxFftStages) { plan.radix[plan.nstages++] = 8; m /= 8; }
  while (m % 4 == 0 && plan.nstages < kMaxFftStages) { plan.radix[plan.nstages++] = 4; m /= 4; }
  while (m % 2 == 0 && plan.nstages < kMaxFftStages) { plan.radix[plan.nstages++] = 2; m /= 2; }
  for (int r : {3, 5, 7})
    while (m % r == 0 && plan.nstages < kMaxFftStages) { plan.radix[plan.nstages++] = r; m /= r; }
  if (m != 1)
    return setLastError(g, HWS_ERR_UNSUPPORTED,
                        "image dimension " + std::to_string(n) +
                            " is not a product of 2, 3, 5 and 7");
  if (n > 16384 || plan.nstages > 16)
    return setLastError(g, HWS_ERR_UNSUPPORTED,
                        "image dimension above 16384 is not supported");
  std::vector<float2> tb(n), tf(n);
  const long double pi = 3.141592653589793238462643383279502884L;
  for (int k = 0; k < n; ++k) {
    const long double a = 2.0L * pi * (long double)k / (long double)n;
    const float c = (float)cosl(a), s = (float)sinl(a);
    tb[k] = make_float2(c, s);
    tf[k] = make_float2(c, -s);
  }
  hws_status st;
  if ((st = checkHip(g, hipMalloc(&plan.twBackward, n * sizeof(float2)), "hipMalloc twiddles")) != HWS_OK) return st;
  if ((st = checkHip(g, hipMalloc(&plan.twForward, n * sizeof(float2)), "hipMalloc twiddles")) != HWS_OK) return st;
  if ((st = checkHip(g, hipMemcpy(plan.twBackward, tb.data(), n * sizeof(float2), hipMemcpyHostToDevice), "twiddle upload")) != HWS_OK) return st;
  return checkHip(g, hipMemcpy(plan.twForward, tf.data(), n * sizeof(float2), hipMemcpyHostToDevice), "twiddle upload");
}

void freeFftPlan(FftPlan& plan) {
  if (plan.twBackward) (void)hipFree(plan.twBackward);
  if (plan.twForward) (void)hipFree(plan.twForward);
  plan.twBackward = plan.twForward = nullptr;
}

namespace {

// Power-of-two launch shapes: rows take max(1, 4096/N) rows per block,
// columns max(1, 8192/N) columns (at most 16); 16 values per thread.
template <int SIGN, int N>
void launchPow2(float2* data, int W, int H, int nbatch, const float2* twRow,
                const float2* twCol, bool rows, hipStream_t stream) {
  if (rows) {
    constexpr int NFFT = (4096 / N) > 0 ? (4096 / N) : 1;
    constexpr int E = NFFT * N;
    constexpr int NT = (E / 16) < 64 ? 64 : (E / 16) > 1024 ? 1024 : (E / 16);
    const int nfft = std::min(NFFT, H);
    (void)nfft;
    dim3 grid((H + NFFT - 1) / NFFT, nbatch);
    hipLaunchKernelGGL((fftRowsPow2Kernel<SIGN, N, NT, NFFT>), grid, dim3(NT), 0, stream, data, H, twRow);
  } else {
    constexpr int NFFT0 = (8192 / N) > 0 ? (8192 / N) : 1;
    constexpr int NFFT = NFFT0 > 16 ? 16 : NFFT0;
    constexpr int E = NFFT * N;
    constexpr int NT = (E / 16) < 64 ? 64 : (E / 16) > 1024 ? 1024 : (E / 16);
    const int nColBlocks = (W + NFFT - 1) / NFFT;
    dim3 grid(nColBlocks, nbatch);
    hipLaunchKernelGGL((fftColsPow2Kernel<SIGN, N, NT, NFFT>), grid, dim3(NT), 0, stream, data, W, nColBlocks, twCol);
  }
}

template <int SIGN>
bool dispatchPow2(int n, float2* data, int W, int H, int nbatch, const float2* twRow,
                  const float2* twCol, bool rows, hipStream_t stream) {
  switch (n) {
    case 64: launchPow2<SIGN, 64>(data, W, H, nbatch, twRow, twCol, rows, stream); return true;
    case 128: launchPow2<SIGN, 128>(data, W, H, nbatch, twRow, twCol, rows, stream); return true;
    case 256: launchPow2<SIGN, 256>(data, W, H, nbatch, twRow, twCol, rows, stream); return true;
    case 512: launchPow2<SIGN, 512>(data, W, H, nbatch, twRow, twCol, rows, stream); return true;
    case 1024: launchPow2<SIGN, 1024>(data, W, H, nbatch, twRow, twCol, rows, stream); return true;
    case 2048: launchPow2<SIGN, 2048>(data, W, H, nbatch, twRow, twCol, rows, stream); return true;
    case 4096: launchPow2<SIGN, 4096>(data, W, H, nbatch, twRow, twCol, rows, stream); return true;
    case 8192: launchPow2<SIGN, 8192>(data, W, H, nbatch, twRow, twCol, rows, stream); return true;
    default: return false;
  }
}

}  // namespace

namespace {
template <int SIGN>
bool launchBlocked(int n, bool rows, float2* data, int W, int H, int nbatch,
                   const float2* tw, hipStream_t stream) {
#define HWS_BLOCKED_CASE(NN)                                                            \
  case NN:                                                                              \
    if (rows)                                                                           \
      hipLaunchKernelGGL((fftRowsBlockedKernel<SIGN, NN>), dim3(H / 4, nbatch),         \
                         dim3(NN / 4), 0, stream, data, H, tw);                         \
    else                                                                                \
      hipLaunchKernelGGL((fftColsBlockedKernel<SIGN, NN>), dim3(W / 4, nbatch),         \
                         dim3(NN / 4), 0, stream, data, W, tw);                         \
    return true;
  switch (n) {
    HWS_BLOCKED_CASE(256)
    HWS_BLOCKED_CASE(512)
    HWS_BLOCKED_CASE(1024)
    HWS_BLOCKED_CASE(2048)
    HWS_BLOCKED_CASE(4096)
    default: return false;
  }
#undef HWS_BLOCKED_CASE
}
}  // namespace

// Sizes with compile-time blocked kernels (and their sparse variants).
bool fastBlockedSize(int n) { return n >= 256 && n <= 4096 && (n & (n - 1)) == 0; }

// The blocked layout is used whenever both sizes are multiples of 4 and one
// line of each fits the LDS of one runtime-radix workgroup (n <= 18308); the
// transform plans then also have to fit the workgroup's threads
// (blockedGenericFits: 16 values per thread, n up to about 15000).
bool blockedLayoutSupported(int W, int H) {
  if (fastBlockedSize(W) && fastBlockedSize(H)) return true;
  return W % 4 == 0 && H % 4 == 0 && W >= 16 && H >= 16 && blockedGenericLineFits(W) && blockedGenericLineFits(H);
}


bool colsProjectGeneric(const hws_gridder* g) {
  return !(fastBlockedSize(g->W) && fastBlockedSize(g->H));
}

bool colsProjectSupported(const hws_gridder* g, int nLayersInPass) {
  if (!g->blocked || g->noFusedProject) return false;
  const int T = g->plan.tileSize;
  if (T < 4 || (T & (T - 1)) != 0) return false;
  int maxLds = 65536;
  (void)hipDeviceGetAttribute(&maxLds, hipDeviceAttributeMaxSharedMemoryPerBlock, g->cfg.device);
  if (colsProjectGeneric(g)) return colsProjectGenericSupported(g, nLayersInPass, size_t(maxLds));
  return colsProjectLds(g->H, nLayersInPass, g->H / T) <= size_t(maxLds);
}

hws_status launchColsProject(hws_gridder* g, const ColsProjectArgs& a, bool cplx,
                             const float2* layers, float* sum, float* comp, float* isum,
                             float* icomp) {
  if (a.nImg == 0 || a.nLayersInPass == 0) return HWS_OK;
  if (colsProjectGeneric(g))
    launchColsProjectGeneric(g, a, cplx, layers, sum, comp, isum, icomp);
  else if (!launchColsProjectPow2(g, a, cplx, layers, sum, comp, isum, icomp))
    return setLastError(g, HWS_ERR_UNSUPPORTED, "fused projection: height not supported");
  return checkHip(g, hipGetLastError(), "fused columns and projection launch");
}

hws_status fft2d(hws_gridder* g, float2* data, int nbatch, int sign, const FftSparse* sparse,
                 const ModelSource* model) {
  if (nbatch <= 0) return HWS_OK;
  const int W = g->W, H = g->H;  if (g->blocked && !(fastBlockedSize(W) && fastBlockedSize(H)))
    return fft2dGeneric(g, data, nbatch, sign, sparse, model);
  if (g->blocked) {
    const float2* twRow = sign > 0 ? g->rowPlan.twBackward : g->rowPlan.twForward;
    const float2* twCol = sign > 0 ? g->colPlan.twBackward : g->colPlan.twForward;
    bool ok;
    if (sign > 0 && sparse) {
      ok = false;
      switch (W) {
#define HWS_SPARSE_CASE(NN)                                                                    \
  case NN:                                                                                     \
    hipLaunchKernelGGL((fftRowsBlockedSparseKernel<+1, NN>), dim3(H / 4, nbatch), dim3(NN / 4), \
                       0, g->stream, data, H, twRow, sparse->occ, sparse->layer0,              \
                       sparse->tilesY, sparse->tshift);                                        \
    ok = true;                                                                                 \
    break;
        HWS_SPARSE_CASE(256)
        HWS_SPARSE_CASE(512)
        HWS_SPARSE_CASE(1024)
        HWS_SPARSE_CASE(2048)
        HWS_SPARSE_CASE(4096)
#undef HWS_SPARSE_CASE
        default: break;
      }
      bool cols = sparse->rowsOnly;
      if (!cols) switch (H) {
#define HWS_ROWSPARSE_COLS(NN)                                                                 \
  case NN:                                                                                     \
    hipLaunchKernelGGL((fftColsBlockedRowSparseKernel<+1, NN>), dim3(W / 4, nbatch),            \
                       dim3(NN / 4), 0, g->stream, data, W, twCol, sparse->rowLive,            \
                       sparse->layer0, sparse->tilesY, sparse->tshift);                        \
    cols = true;                                                                               \
    break;
        HWS_ROWSPARSE_COLS(256)
        HWS_ROWSPARSE_COLS(512)
        HWS_ROWSPARSE_COLS(1024)
        HWS_ROWSPARSE_COLS(2048)
        HWS_ROWSPARSE_COLS(4096)
#undef HWS_ROWSPARSE_COLS
        default: break;
      }
      ok = ok && cols;
    } else if (sign < 0 && sparse) {
      if (model && sparse->colNeed) {
        ok = launchModelLayersPow2(g, data, nbatch, twRow, *model, *sparse);
      } else if (model) {
        ok = false;
        const int ml = model->precision == HWS_PRECISION_REFERENCE ? modelLayers<true>()
                                                                   : modelLayers<false>();
        const dim3 mgrid(H / 4, (nbatch + ml - 1) / ml);
        switch (W) {
#define HWS_MODEL_ROWS(NN)                                                                      \
  case NN:                                                                                      \
    if (model->precision == HWS_PRECISION_REFERENCE)                                            \
      hipLaunchKernelGGL((fftRowsFromModelKernel<-1, NN, true>), mgrid, dim3(NN / 4), 0,         \
                         g->stream, data, H, nbatch, twRow, *model);                            \
    else                                                                                        \
      hipLaunchKernelGGL((fftRowsFromModelKernel<-1, NN, false>), mgrid, dim3(NN / 4), 0,        \
                         g->stream, data, H, nbatch, twRow, *model);                            \
    ok = true;                                                                                  \
    break;
          HWS_MODEL_ROWS(256)
          HWS_MODEL_ROWS(512)
          HWS_MODEL_ROWS(1024)
          HWS_MODEL_ROWS(2048)
          HWS_MODEL_ROWS(4096)
#undef HWS_MODEL_ROWS
          default: break;
        }
      } else {
        ok = launchBlocked<-1>(W, true, data, W, H, nbatch, twRow, g->stream);
      }
      bool cols = false;
      switch (H) {
#define HWS_SPARSE_COLS(NN)                                                                    \
  case NN:                                                                                     \
    hipLaunchKernelGGL((fftColsBlockedSparseKernel<-1, NN>), dim3(W / 4, nbatch), dim3(NN / 4), \
                       0, g->stream, data, W, twCol, sparse->occ, sparse->layer0,              \
                       sparse->tilesY, sparse->tshift);                                        \
    cols = true;                                                                               \
    break;
        HWS_SPARSE_COLS(256)
        HWS_SPARSE_COLS(512)
        HWS_SPARSE_COLS(1024)
        HWS_SPARSE_COLS(2048)
        HWS_SPARSE_COLS(4096)
#undef HWS_SPARSE_COLS
        default: break;
      }
      ok = ok && cols;
    } else if (sign > 0)
      ok = launchBlocked<+1>(W, true, data, W, H, nbatch, twRow, g->stream) &&
           launchBlocked<+1>(H, false, data, W, H, nbatch, twCol, g->stream);
    else
      ok = launchBlocked<-1>(W, true, data, W, H, nbatch, twRow, g->stream) &&
           launchBlocked<-1>(H, false, data, W, H, nbatch, twCol, g->stream);
    if (!ok) return setLastError(g, HWS_ERR_UNSUPPORTED, "blocked layout size not supported");
    return checkHip(g, hipGetLastError(), "fft blocked launch");
  }
  int maxLds = 65536;
  (void)hipDeviceGetAttribute(&maxLds, hipDeviceAttributeMaxSharedMemoryPerBlock, g->cfg.device);
  const float2* twRow = sign > 0 ? g->rowPlan.twBackward : g->rowPlan.twForward;
  const float2* twCol = sign > 0 ? g->colPlan.twBackward : g->colPlan.twForward;
  bool rowsDone = false, colsDone = false;
  if (sign > 0) {
    rowsDone = dispatchPow2<+1>(W, data, W, H, nbatch, twRow, twCol, true, g->stream);
    colsDone = dispatchPow2<+1>(H, data, W, H, nbatch, twRow, twCol, false, g->stream);
  } else {
    rowsDone = dispatchPow2<-1>(W, data, W, H, nbatch, twRow, twCol, true, g->stream);
    colsDone = dispatchPow2<-1>(H, data, W, H, nbatch, twRow, twCol, false, g->stream);
  }
  if (rowsDone || colsDone) {
    hws_status st = checkHip(g, hipGetLastError(), "fft pow2 launch");
    if (st != HWS_OK) return st;
  }
  // rows: as many whole rows per block as fit 4096 values (at least one)
  if (!rowsDone) {
    int rows = std::max(1, 4096 / W);
    rows = std::min(rows, H);
    const int threads = threadsFor(g->rowPlan, rows);
    const size_t lds = size_t(rows) * ldsPitch(W) * sizeof(float2);
    if (threads == 0 || lds > size_t(maxLds))
      return setLastError(g, HWS_ERR_UNSUPPORTED, "row transform does not fit one workgroup");
    dim3 grid((H + rows - 1) / rows, nbatch);
    const unsigned long long radices = packRadices(g->rowPlan);
    const float2* tw = sign > 0 ? g->rowPlan.twBackward : g->rowPlan.twForward;
    if (sign > 0)
      launchRowsPlain<+1>(threads, grid, lds, g->stream, data, W, H, rows, radices, tw);
    else
      launchRowsPlain<-1>(threads, grid, lds, g->stream, data, W, H, rows, radices, tw);
    hws_status st = checkHip(g, hipGetLastError(), "fft rows launch");
    if (st != HWS_OK) return st;
  }
  // columns: blocks of bc columns, [bc][ldsPitch(H)] in LDS
  if (!colsDone) {
    int bc = std::max(1, 8192 / H);
    bc = std::min(std::min(bc, 16), W);
    while (bc > 1 && size_t(bc) * ldsPitch(H) * sizeof(float2) > size_t(maxLds)) --bc;
    int threads = threadsFor(g->colPlan, bc);
    while (threads == 0 && bc > 1) threads = threadsFor(g->colPlan, --bc);
    const size_t lds = size_t(bc) * size_t(ldsPitch(H)) * sizeof(float2);
    if (threads == 0 || lds > size_t(maxLds))
      return setLastError(g, HWS_ERR_UNSUPPORTED, "column transform does not fit one workgroup");
    const int nColBlocks = (W + bc - 1) / bc;
    dim3 grid(nColBlocks, nbatch);
    const unsigned long long radices = packRadices(g->colPlan);
    const float2* tw = sign > 0 ? g->colPlan.twBackward : g->colPlan.twForward;
    if (sign > 0)
      launchColsPlain<+1>(threads, grid, lds, g->stream, data, W, H, bc, nColBlocks, radices, tw);
    else
      launchColsPlain<-1>(threads, grid, lds, g->stream, data, W, H, bc, nColBlocks, radices, tw);
    hws_status st = checkHip(g, hipGetLastError(), "fft cols launch");
    if (st != HWS_OK) return st;
  }
  return HWS_OK;
}

}  // namespace hws
