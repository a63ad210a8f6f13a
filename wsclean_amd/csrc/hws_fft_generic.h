// The blocked runtime-radix stages, shared by the sources that hold their
// kernels (hws_fft_generic.hip, hws_fft_generic_fused.hip).
#ifndef HWS_FFT_GENERIC_H
#define HWS_FFT_GENERIC_H

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

}  // namespace

// hws_fft_generic_fused.hip: the forward rows pass from the model for every
// layer (threads and lines per workgroup as for the other rows passes).
void launchModelLayersGeneric(int threads, int lines, dim3 grid, size_t lds, hipStream_t st,
                              float2* data, int W, int H, int nbatch, unsigned long long rad,
                              const float2* tw, const ModelSource& ms, const uint32_t* colNeed,
                              int tshift);

}  // namespace hws

#endif
