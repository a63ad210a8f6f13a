// Device building blocks of the layer transforms: butterflies, the blocked
// layout's compile-time Stockham stages (memory to memory, and registers to
// registers for the kernels that fuse a transform with what precedes or
// follows it) and what the runtime-radix stages share. Included by the
// transform sources only (each holds its own kernels).
#ifndef HWS_FFT_DEVICE_H
#define HWS_FFT_DEVICE_H

#include "hws_internal.h"

namespace hws {

namespace {

// The butterflies and twiddle products fuse only where written (fmaf), so a
// transform computes the same bits in every kernel that inlines it; left to
// itself, the compiler contracts a product into the following sum in some
// inlining contexts and not in others.
__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
#pragma clang fp contract(off)
  return make_float2(fmaf(a.x, b.x, -(a.y * b.y)), fmaf(a.x, b.y, a.y * b.x));
}
__device__ __forceinline__ float2 cadd(float2 a, float2 b) {
  return make_float2(a.x + b.x, a.y + b.y);
}
__device__ __forceinline__ float2 csub(float2 a, float2 b) {
  return make_float2(a.x - b.x, a.y - b.y);
}
// multiply by sign * i
template <int SIGN>
__device__ __forceinline__ float2 mulI(float2 a) {
  return SIGN > 0 ? make_float2(-a.y, a.x) : make_float2(a.y, -a.x);
}

template <int SIGN, int R>
struct Butterfly;

template <int SIGN>
struct Butterfly<SIGN, 2> {
  __device__ __forceinline__ static void run(float2* v) {
#pragma clang fp contract(off)
    float2 a = v[0], b = v[1];
    v[0] = cadd(a, b);
    v[1] = csub(a, b);
  }
};

template <int SIGN>
struct Butterfly<SIGN, 4> {
  __device__ __forceinline__ static void run(float2* v) {
#pragma clang fp contract(off)
    float2 a0 = cadd(v[0], v[2]), a1 = csub(v[0], v[2]);
    float2 b0 = cadd(v[1], v[3]), b1 = mulI<SIGN>(csub(v[1], v[3]));
    v[0] = cadd(a0, b0);
    v[2] = csub(a0, b0);
    v[1] = cadd(a1, b1);
    v[3] = csub(a1, b1);
  }
};

template <int SIGN>
struct Butterfly<SIGN, 8> {
  __device__ __forceinline__ static void run(float2* v) {
#pragma clang fp contract(off)
    // radix-2 over even/odd, then radix-4 on each half
    float2 e[4] = {v[0], v[2], v[4], v[6]};
    float2 o[4] = {v[1], v[3], v[5], v[7]};
    Butterfly<SIGN, 4>::run(e);
    Butterfly<SIGN, 4>::run(o);
    const float h = 0.70710678118654752440f;
    // o[k] *= w8^k, w8 = exp(SIGN * 2 pi i / 8)
    o[1] = make_float2(h * (o[1].x - SIGN * o[1].y), h * (o[1].y + SIGN * o[1].x));
    o[2] = mulI<SIGN>(o[2]);
    o[3] = make_float2(h * (-o[3].x - SIGN * o[3].y), h * (-o[3].y + SIGN * o[3].x));
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      v[k] = cadd(e[k], o[k]);
      v[k + 4] = csub(e[k], o[k]);
    }
  }
};

// Odd radix: direct DFT with exp(SIGN 2 pi i k/R) constants.
template <int SIGN, int R>
struct Butterfly {
  __device__ __forceinline__ static void run(float2* v) {
#pragma clang fp contract(off)
    float2 res[R];
#pragma unroll
    for (int k = 0; k < R; ++k) {
      float2 acc = v[0];
#pragma unroll
      for (int r = 1; r < R; ++r) {
        const int m = (r * k) % R;
        float s, c;
        // constants folded at compile time
        c = (float)__builtin_cos(2.0 * 3.14159265358979323846 * m / R);
        s = (float)(SIGN * __builtin_sin(2.0 * 3.14159265358979323846 * m / R));
        acc = cadd(acc, cmul(v[r], make_float2(c, s)));
      }
      res[k] = acc;
    }
#pragma unroll
    for (int k = 0; k < R; ++k) v[k] = res[k];
  }
};

constexpr int kMaxValues = 16;  // complex values held per thread per stage

// LDS position of element e of a line of the runtime-radix transforms: one
// pad value after every 16, so that the first stage's writes (stride R = 16,
// 8, 4 or 2 values across the lanes) fall in distinct banks.
__device__ __forceinline__ int lp(int e) { return e + (e >> 4); }

// Line pitch (in values) of those transforms for length n: the padded length
// plus one.
__host__ __device__ constexpr int ldsPitch(int n) { return n + (n >> 4) + 1; }

// Division by a divisor that is the same on every lane: x / d ==
// umulhi(x, ceil(2^32 / d)) for d >= 2 whenever x * d < 2^32 (here x and d
// stay below 2^16).
struct UniformDiv {
  uint32_t m;
  int d;
};
__device__ __forceinline__ UniformDiv uniformDiv(int d) {
  return UniformDiv{d > 1 ? 0xFFFFFFFFu / uint32_t(d) + 1u : 0u, d};
}
__device__ __forceinline__ int divBy(int x, UniformDiv u) {
  return u.d == 1 ? x : int(__umulhi(uint32_t(x), u.m));
}

// ---- blocked layer layout: element (x, y) of a W x H layer is stored at
// ((y >> 2) * W + x) * 4 + (y & 3), i.e. groups of four rows interleaved.
// A row block (four rows) is then one contiguous run of 4W values and the
// four columns x0..x0+3 form 128-byte segments, so both passes of the 2-D
// transform read and write HBM fully coalesced. Each pass keeps four
// transforms of length N (N/4 threads, 16 values per thread) in flight:
// stage 0 reads HBM into registers, stages exchange through one padded LDS
// buffer, the last stage writes HBM. Radix 16 stages, then 8, 4 or 2.

__device__ __forceinline__ int padIdx(int e) { return e + (e >> 6); }

template <int SIGN>
struct Butterfly<SIGN, 16> {
  __device__ __forceinline__ static void run(float2* v) {
#pragma clang fp contract(off)
    // 4 x 4: DFT4 over stride-4 inputs, twiddle w16^(n1 k2), DFT4 again
    float2 a[4][4];
#pragma unroll
    for (int n2 = 0; n2 < 4; ++n2) {
#pragma unroll
      for (int n1 = 0; n1 < 4; ++n1) a[n2][n1] = v[n2 + 4 * n1];
      Butterfly<SIGN, 4>::run(a[n2]);  // a[n2][k1]
    }
    const float c1 = 0.92387953251128675613f, s1 = 0.38268343236508977173f;
    const float h = 0.70710678118654752440f;
    // twiddle a[n2][k1] *= w16^(n2 k1), w16 = exp(SIGN 2 pi i / 16)
    const float2 w1 = make_float2(c1, SIGN * s1), w2 = make_float2(h, SIGN * h),
                 w3 = make_float2(s1, SIGN * c1), w4 = make_float2(0.0f, float(SIGN)),
                 w6 = make_float2(-h, SIGN * h), w9 = make_float2(-c1, -SIGN * s1);
    a[1][1] = cmul(a[1][1], w1);
    a[1][2] = cmul(a[1][2], w2);
    a[1][3] = cmul(a[1][3], w3);
    a[2][1] = cmul(a[2][1], w2);
    a[2][2] = cmul(a[2][2], w4);
    a[2][3] = cmul(a[2][3], w6);
    a[3][1] = cmul(a[3][1], w3);
    a[3][2] = cmul(a[3][2], w6);
    a[3][3] = cmul(a[3][3], w9);
#pragma unroll
    for (int k1 = 0; k1 < 4; ++k1) {
      float2 b[4] = {a[0][k1], a[1][k1], a[2][k1], a[3][k1]};
      Butterfly<SIGN, 4>::run(b);
#pragma unroll
      for (int k2 = 0; k2 < 4; ++k2) v[k1 + 4 * k2] = b[k2];
    }
  }
};

template <bool ROWS>
__device__ __forceinline__ size_t blockedAddr(int pos, int f, int W) {
  // ROWS: pos = x, f = row in block; COLS: pos = y, f = column in block
  if (ROWS) return size_t(pos) * 4 + f;
  return (size_t(pos >> 2) * W + f) * 4 + (pos & 3);
}

// live (may be null): one flag per tile-sized stretch of the block's rows
// (rows pass: per uv tile along x) or columns (columns pass: per tile row
// along y), indexed by pos >> tshift (tshift = log2 of the tile edge).
// liveIn: cells of a stretch that is not live read as zero (their memory is
// not read, and need not have been written); otherwise they are not written.
// The layer cell (x, y) of a forward transform computed from the model image
// (the arithmetic of imageToLayersKernel, so the results are identical). REF:
// the reference precision (float n', FP64 sine and cosine).
template <bool REF>
__device__ __forceinline__ float2 modelCell(const ModelSource& ms, double w, int x, int y, int W,
                                           int H) {
  int yDest = y + H / 2;
  if (yDest >= H) yDest -= H;
  int xDest = (W - x) + W / 2;
  if (xDest >= W) xDest -= W;
  const double m = pixelM(yDest, H, ms.dm, ms.mShift);
  const double l = pixelL(xDest, W, ms.dl, ms.lShift);
  double np = nPrimeSeries(l, m);
  if (REF) np = double(float(np));
  const size_t src = size_t(yDest) * W + xDest;
  const float re = ms.re[src];
  const float imv = ms.cplx ? -ms.im[src] : 0.0f;
  return modelTerm<REF>(re, imv, ms.cplx != 0, w, np);
}

// Layers per workgroup of the model-fed rows pass: the workgroup reads the
// model rows of its row block once from memory and then from the L2 (the
// reference precision one: four take 128 registers for its 80).
template <bool REF>
constexpr int modelLayers() {
  return REF ? 1 : 4;
}

// A store the pass does not read back: marked non-temporal, so the stream of
// layer writes does not evict what the caches hold (the model image the
// forward rows pass reads for every layer).
__device__ __forceinline__ void streamStore(float2* p, float2 v) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  const f2 x = {v.x, v.y};
  __builtin_nontemporal_store(x, reinterpret_cast<f2*>(p));
}

// A load of a layer element the pass reads once (non-temporal).
__device__ __forceinline__ float2 streamLoad(const float2* p) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  const f2 v = __builtin_nontemporal_load(reinterpret_cast<const f2*>(p));
  return make_float2(v.x, v.y);
}

// MODEL (rows pass of a forward transform): the first stage computes its
// inputs from the model image (ms, w; y0 = the row block's first row)
// instead of reading the layer.
template <int SIGN, int R, int N, int NS, bool ROWS, int MODEL = 0>
__device__ __forceinline__ void blockedStage(float2* lds, float2* __restrict__ g, int W,
                                             const float2* __restrict__ tw, int tid,
                                             const unsigned char* live, int tshift,
                                             bool liveIn,
                                             const ModelSource* ms = nullptr, double w = 0.0,
                                             int y0 = 0, int H = 0) {
  constexpr int B = N / R;
  constexpr int T = N / 4;
  constexpr int PER = 16 / R;
  constexpr int TWSTEP = N / (NS * R);
  constexpr bool FIRST = NS == 1;
  constexpr bool LAST = NS * R == N;
  float2 v[PER][R];
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    const int bt = tid + q * T;
    const int f = bt & 3, b = bt >> 2;
    const int jm = b % NS;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int pos = b + r * B;
      float2 x;
      if (FIRST && MODEL)
        x = modelCell<MODEL == 2>(*ms, w, pos, y0 + f, W, H);
      else if (FIRST)
        // (the forward columns pass reads the rows pass's output once: a
        // non-temporal load; measured slower in the backward passes, whose
        // inputs the caches partly hold)
        x = (live && liveIn && !live[pos >> tshift])
                ? make_float2(0.0f, 0.0f)
                : (SIGN < 0 && !ROWS ? streamLoad(&g[blockedAddr<ROWS>(pos, f, W)])
                                     : g[blockedAddr<ROWS>(pos, f, W)]);
      else
        x = lds[padIdx(pos * 4 + f)];
      if (!FIRST && r != 0) x = cmul(x, tw[jm * r * TWSTEP]);
      v[q][r] = x;
    }
  }
  if (!FIRST) __syncthreads();  // every read of this stage precedes its writes
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    const int bt = tid + q * T;
    const int f = bt & 3, b = bt >> 2;
    const int jm = b % NS;
    Butterfly<SIGN, R>::run(v[q]);
    const int base = (b / NS) * NS * R + jm;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int pos = base + r * NS;
      if (LAST) {
        // columns pass of a forward transform: tiles nobody reads are not written
        if (live && !liveIn && !live[pos >> tshift]) continue;
        streamStore(&g[blockedAddr<ROWS>(pos, f, W)], v[q][r]);
      }
      else
        lds[padIdx(pos * 4 + f)] = v[q][r];
    }
  }
  if (!LAST) __syncthreads();
}

template <int SIGN, int N, bool ROWS, int NS = 1, int MODEL = 0>
__device__ __forceinline__ void blockedFft(float2* lds, float2* __restrict__ g, int W,
                                           const float2* __restrict__ tw, int tid,
                                           const unsigned char* live = nullptr,
                                           int tshift = 0, bool liveIn = true,
                                           const ModelSource* ms = nullptr,
                                           double w = 0.0, int y0 = 0, int H = 0) {
  if constexpr (NS < N) {
    constexpr int REM = N / NS;
    constexpr int R = (REM % 16 == 0) ? 16 : REM;  // 16s, then the remaining 8, 4 or 2
    static_assert(R == 16 || R == 8 || R == 4 || R == 2, "radix");
    blockedStage<SIGN, R, N, NS, ROWS, NS == 1 ? MODEL : 0>(lds, g, W, tw, tid, live, tshift,
                                                         liveIn, ms, w, y0, H);
    blockedFft<SIGN, N, ROWS, NS * R, MODEL>(lds, g, W, tw, tid, live, tshift, liveIn, ms, w, y0,
                                             H);
  }
}

// ---- the backward columns pass fused with the w-projection
// One Stockham stage of radix R over NF interleaved transforms of length N
// (NF N / 16 threads, 16 values per thread), as blockedStage but with
// registers for memory: the first stage takes its inputs from io
// (io[q R + r] = element b + r N / R of transform f, for bt = tid + q T,
// f = bt mod NF, b = bt / NF) and the last stage leaves its outputs there
// (io[q R + r] = element ((b / NS) NS R + b mod NS) + r NS of transform f).
template <int SIGN, int R, int N, int NS, int NF>
__device__ __forceinline__ void regStage(float2* lds, const float2* __restrict__ tw, int tid,
                                         const float2* in, float2* out) {
  constexpr int B = N / R;
  constexpr int T = NF * N / 16;
  constexpr int PER = 16 / R;
  constexpr int TWSTEP = N / (NS * R);
  constexpr bool FIRST = NS == 1;
  constexpr bool LAST = NS * R == N;
  float2 v[PER][R];
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    const int bt = tid + q * T;
    const int f = bt % NF, b = bt / NF;
    const int jm = b % NS;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      float2 x = FIRST ? in[q * R + r] : lds[padIdx((b + r * B) * NF + f)];
      if (!FIRST && r != 0) x = cmul(x, tw[jm * r * TWSTEP]);
      v[q][r] = x;
    }
  }
  // every read of this stage precedes its writes (and, in the first stage,
  // the previous transform's last reads precede this one's writes: that
  // stage synchronised between its reads and its outputs)
  if (!FIRST) __syncthreads();
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    const int bt = tid + q * T;
    const int f = bt % NF, b = bt / NF;
    const int jm = b % NS;
    Butterfly<SIGN, R>::run(v[q]);
    const int base = (b / NS) * NS * R + jm;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (LAST)
        out[q * R + r] = v[q][r];
      else
        lds[padIdx((base + r * NS) * NF + f)] = v[q][r];
    }
  }
  if (!LAST) __syncthreads();
}

// The transform of in (consumed by the first stage) into out; afterFirst()
// runs once the first stage has read in (in may then be overwritten, e.g. by
// the loads of the next transform's inputs).
template <int SIGN, int N, int NF, int NS = 1, class F>
__device__ __forceinline__ void regFft(float2* lds, const float2* __restrict__ tw, int tid,
                                       const float2* in, float2* out, F&& afterFirst) {
  if constexpr (NS < N) {
    constexpr int REM = N / NS;
    constexpr int R = (REM % 16 == 0) ? 16 : REM;
    static_assert(R == 16 || R == 8 || R == 4 || R == 2, "radix");
    regStage<SIGN, R, N, NS, NF>(lds, tw, tid, in, out);
    if constexpr (NS == 1) afterFirst();
    regFft<SIGN, N, NF, NS * R>(lds, tw, tid, in, out, afterFirst);
  }
}

// The last stage of regFft over length N: its radix and stride.
template <int N>
struct LastStage {
  static constexpr int p16() {
    int p = 1;
    while ((N / p) % 16 == 0) p *= 16;
    return p;
  }
  static constexpr int R = N / p16() == 1 ? 16 : N / p16();
  static constexpr int NS = N / R;
};

constexpr int kProjectColumns = 2;  // columns per workgroup of the fused pass

// Buffer-resource word 3 for raw (untyped) buffer loads on CDNA.
constexpr int kRawBufferFlags = 0x00020000;
// An offset past every buffer: such a buffer load returns zero without a
// memory access.
constexpr uint32_t kOffsetOutOfRange = 0xFFFFFFF0u;

}  // namespace

// Lines (rows or columns) per workgroup, threads and LDS of the transforms.
unsigned long long packRadices(const FftPlan& plan);
int threadsFor(const FftPlan& plan, int nfft, bool close = false);

// hws_fft_fused.hip: the fused power-of-two kernels; false where the size has
// none.
bool launchColsProjectPow2(hws_gridder* g, const ColsProjectArgs& a, bool cplx,
                           const float2* layers, float* sum, float* comp, float* isum,
                           float* icomp);
size_t colsProjectLds(int H, int nLayersInPass, int tilesY);
bool launchModelLayersPow2(hws_gridder* g, float2* data, int nbatch, const float2* tw,
                           const ModelSource& model, const FftSparse& sparse);

// hws_fft_generic.hip: the blocked runtime-radix kernels.
bool blockedGenericLineFits(int n);
bool colsProjectGenericSupported(const hws_gridder* g, int nLayersInPass, size_t maxLds);
void launchColsProjectGeneric(hws_gridder* g, const ColsProjectArgs& a, bool cplx,
                              const float2* layers, float* sum, float* comp, float* isum,
                              float* icomp);
hws_status fft2dGeneric(hws_gridder* g, float2* data, int nbatch, int sign,
                        const FftSparse* sparse, const ModelSource* model);

}  // namespace hws

#endif
