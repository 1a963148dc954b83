// Commit of a decode step to a sliding-window KV cache (gfx950): the update of
// nanolab's Attention.forward_cached (nanolab/mixers.py:435-450), which keeps
// of the cached rows and the T new ones those at positions < sinks or
// >= end - tail, in their order.
//
//   cache_plan_kernel   one workgroup lists the live rows (their index in the
//                       concatenation [cache | new] and their position) and
//                       stores their count where the host can read it;
//   cache_gather_kernel copies the live rows of K and V into the new cache in
//                       one launch, 16 bytes a thread.
//
// Both are bound by launch latency at the sizes a window cache has (at most
// window - 1 rows a head stay), so what counts is the number of launches and
// host waits: the chain of tensor operations (masks, cat, boolean indexing of
// K, V and the positions) took about 30 launches and three waits a step.
// Measured, SWA(64, 4) one-token steps at B16 H12 D64 bf16, committed:
// 180.3 -> 44.5 us a step (the step's own kernel is 6 us of it).
#include "attn_common.h"

namespace mi {

// Row i of [cache | new] is at pos[i] (i when pos is null) for i < Lc and at
// start + i - Lc beyond. The order of the rows is kept: a workgroup-wide
// prefix count in chunks of 256 rows.
__global__ void __launch_bounds__(256)
cache_plan_kernel(const long long* __restrict__ pos, int Lc, int n, long long start, long long lo,
                  long long sinks, int* __restrict__ rows, long long* __restrict__ pos_out,
                  int* __restrict__ count) {
  __shared__ int part[2][4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int base = 0;
  for (int i0 = 0, it = 0; i0 < n; i0 += 256, it ^= 1) {
    const int i = i0 + tid;
    long long at = 0;
    if (i < n) at = i >= Lc ? start + (i - Lc) : pos ? pos[i] : i;
    const bool live = i < n && (at < sinks || at >= lo);
    const unsigned long long m = __ballot(live);
    if (lane == 0) part[it][wave] = __popcll(m);
    __syncthreads();   // `part` alternates: the next chunk writes the other half
    int before = base + __popcll(m & ((1ull << lane) - 1ull));
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      if (w < wave) before += part[it][w];
      base += part[it][w];
    }
    if (live) {
      rows[before] = i;
      pos_out[before] = at;
    }
  }
  if (tid == 0) {
    *count = base;
    __threadfence_system();   // `count` may be host memory
  }
}

// out[t][b][h][r] (t = 0: K, 1: V; [B, Hkv, n, D] each) = row rows[r] of
// [cache | new]. One thread per 16-byte chunk; C chunks per row.
__global__ void __launch_bounds__(256)
cache_gather_kernel(const char* __restrict__ kc, const char* __restrict__ vc,
                    const char* __restrict__ kn, const char* __restrict__ vn,
                    const int* __restrict__ rows, char* __restrict__ ko, char* __restrict__ vo,
                    CommitParams p) {
  const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
  if (t >= p.total) return;
  const int c = (int)(t % p.chunks);
  long long u = t / p.chunks;
  const int r = (int)(u % p.n);
  u /= p.n;
  const int h = (int)(u % p.Hkv);
  u /= p.Hkv;
  const int b = (int)(u % p.B);
  const bool is_v = u >= p.B;
  const int i = rows[r];
  const long long row_bytes = 16LL * p.chunks;
  const char* src;
  if (i < p.Lc) {
    src = (is_v ? vc + b * p.v_sb + h * p.v_sh : kc + b * p.k_sb + h * p.k_sh) + i * row_bytes;
  } else {
    src = (is_v ? vn : kn) + (((long long)b * p.T + (i - p.Lc)) * p.Hkv + h) * row_bytes;
  }
  char* dst = (is_v ? vo : ko) + (((long long)b * p.Hkv + h) * p.n + r) * row_bytes;
  *reinterpret_cast<u32x4*>(dst + 16 * c) = *reinterpret_cast<const u32x4*>(src + 16 * c);
}

hipError_t launch_cache_plan(const long long* pos, int Lc, int T, long long start, long long lo,
                             long long sinks, int* rows, long long* pos_out, int* count,
                             hipStream_t st) {
  hipLaunchKernelGGL(cache_plan_kernel, dim3(1), dim3(256), 0, st, pos, Lc, Lc + T, start, lo,
                     sinks, rows, pos_out, count);
  return hipGetLastError();
}

hipError_t launch_cache_gather(const void* kc, const void* vc, const void* kn, const void* vn,
                               const int* rows, void* ko, void* vo, const CommitParams& p,
                               hipStream_t st) {
  if (p.total <= 0) return hipSuccess;
  hipLaunchKernelGGL(cache_gather_kernel, dim3((unsigned)((p.total + 255) / 256)), dim3(256), 0,
                     st, (const char*)kc, (const char*)vc, (const char*)kn, (const char*)vn, rows,
                     (char*)ko, (char*)vo, p);
  return hipGetLastError();
}

}  // namespace mi
