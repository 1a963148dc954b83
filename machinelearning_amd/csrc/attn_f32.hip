// float32 attention for grids that leave the chip idle, and for long walks (gfx950):
// forward, dQ (with the delta pass) and dK/dV whose workgroups split the walk.
//
// v_mfma_f32_32x32x2f32 takes 64 cycles for 4 KFLOP, so a float32 wave is
// bound by its serial chain of MFMAs: 128 per 32 x 64 tile forward, 256 in
// dK/dV. The tiled kernels (attn_fwd.hip, attn_bwd.hip) give one workgroup 128
// rows and every wave the whole walk over the other side; at B4 H4 S256 that is
// 32 workgroups on 256 CUs and a chain of up to four 64-key tiles a wave.
// Here a workgroup owns 32 rows and its four waves take every fourth 32-row
// tile of the walk, with their own partial results, summed through LDS in wave
// order at the end (no atomics: bitwise reproducible). Four times the
// workgroups, a quarter of the chain.
//
// No LDS staging: a tile's MFMA operands come straight from global memory (L2)
// into registers. The contraction over head dims may visit them in any order
// that both operands share, so a lane's natural rows are 16-byte loads (chunk j
// of lane half g: head dims 8j + 4g .. +3, four MFMAs); the transposed operands
// (column d = 32 dt + l32 of row crow(s, g)) are loads of 32 consecutive floats.
// Loads go through a buffer resource that ends at row S of the head: rows past
// it read as zeros. Two waves a SIMD (D <= 64) hide those loads; the MFMA chain
// then bounds the kernels (causal B8 H12 S1024 D64: 103 TFLOP/s forward and, all seven
// products counted, 97 backward, of the 157 that float32 MFMA peaks at).
//
// Which launches take it, and the times of both sides: f32_split_walk below.
#include "attn_common.h"

namespace mi {

namespace {

constexpr int kWaves = 4;

typedef __amdgpu_buffer_rsrc_t Buf;

// Rows [0, S) of one head of a [B, S, heads, D] float tensor.
struct Head {
  Buf r;
  unsigned rb;     // bytes from one row to the next
};
__device__ __forceinline__ Head head_of(const float* base, int b, int S, long long rs, int h, int D) {
  Head x;
  float* p = const_cast<float*>(base) + (long long)b * S * rs + (long long)h * D;
  x.r = __builtin_amdgcn_make_buffer_rsrc(p, 0, (int)(((long long)(S - 1) * rs + D) * 4), 0x00020000);
  x.rb = (unsigned)(rs * 4);
  return x;
}

// Row row0 + l32, chunk 8j + 4g: c[j][e] is head dim 8j + 4g + e.
template <int D>
__device__ __forceinline__ void load_rows(f32x4 (&c)[D / 8], const Head& x, int row0, int l32, int g) {
  const unsigned off = (unsigned)(row0 + l32) * x.rb + 16u * g;
#pragma unroll
  for (int j = 0; j < D / 8; ++j)
    c[j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(x.r, off + 32u * j, 0, 0));
}
// Rows row0 + crow(s, g) of columns 32 dt + l32.
template <int D>
__device__ __forceinline__ void load_cols(float (&t)[16][D / 32], const Head& x, int row0, int l32, int g) {
  const unsigned off = (unsigned)(row0 + 4 * g) * x.rb + 4u * l32;
#pragma unroll
  for (int s = 0; s < 16; ++s)
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt)
      t[s][dt] = __builtin_bit_cast(
          float, __builtin_amdgcn_raw_buffer_load_b32(x.r, off + crow_off(s) * x.rb + 128u * dt, 0, 0));
}

// acc += rows . cols over the head dims (32 x 32).
template <int D>
__device__ __forceinline__ f32x16 dot_rows(const f32x4 (&a)[D / 8], const f32x4 (&b)[D / 8], f32x16 acc) {
#pragma unroll
  for (int j = 0; j < D / 8; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) acc = Mfma32<float>::mma(a[j][e], b[j][e], acc);
  return acc;
}

__device__ __forceinline__ float halves(float x) { return x + __shfl_xor(x, 32); }

// A wave's 32 x D partial (acc[dt] register r: column 32 dt + crow(r, g) of row
// l32) into LDS rows of D + 4 floats.
template <int D>
__device__ __forceinline__ void put_partial(float* dst, const f32x16 (&acc)[D / 32], int l32, int g) {
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      *reinterpret_cast<f32x4*>(dst + l32 * (D + 4) + dt * 32 + 8 * j + 4 * g) =
          f32x4{acc[dt][4 * j], acc[dt][4 * j + 1], acc[dt][4 * j + 2], acc[dt][4 * j + 3]};
}

}  // namespace

template <int D, bool BLK>
__global__ void __launch_bounds__(256)
attn_f32_fwd_kernel(const float* __restrict__ Q, const float* __restrict__ K,
                    const float* __restrict__ V, float* __restrict__ O, float* __restrict__ LSE,
                    AttnParams p) {
  constexpr int DT = D / 32;
  __shared__ __attribute__((aligned(16))) float part[kWaves][32 * (D + 4)];
  __shared__ float ml[2][kWaves][32];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, g = lane >> 5;
  const WorkItem wi = work_item(p.nblk, p.B * p.H, p.div_wi, p.causal, p.wi_blocks_fastest);
  const int b = (int)fdiv((unsigned)wi.bh, p.div_h), h = wi.bh - b * p.H;
  const int hkv = (int)fdiv((unsigned)h, p.div_group);
  const int q0 = wi.blk * 32, qi = q0 + l32;

  const Head hK = head_of(K, b, p.S, p.kv_rs, hkv, D), hV = head_of(V, b, p.S, p.kv_rs, hkv, D);
  f32x4 qf[D / 8], kr[D / 8];
  float vc[16][DT];
  load_rows<D>(qf, head_of(Q, b, p.S, p.q_rs, h, D), q0, l32, g);

  int kbeg = 0, kend = p.S;
  if (p.causal) kend = min(p.S, causal_key_end<BLK>(p, q0 + 31) + 1);
  if (p.window > 0) kbeg = max(0, q0 - p.window + 1);
  const int t_begin = kbeg / 32, t_end = (kend + 31) / 32;
  const int key_hi = p.causal ? min(causal_key_end<BLK>(p, qi), p.S - 1) : p.S - 1;
  const int key_lo = p.window > 0 ? qi - p.window + 1 : 0;
  const int all_hi = p.causal ? min(causal_key_end<BLK>(p, q0), p.S - 1) : p.S - 1;

  f32x16 oacc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) oacc[dt] = zero16();
  float m_run = -1e30f, l_run = 0.f;    // as attn_fwd.hip: raw-score max, lane-local sum
  const float c = p.scale_log2;
  int t = t_begin + wave;
  if (t < t_end) {
    load_rows<D>(kr, hK, t * 32, l32, g);
    load_cols<D>(vc, hV, t * 32, l32, g);
  }
  for (; t < t_end; t += kWaves) {
    const int k0 = t * 32;
    f32x16 s = dot_rows<D>(kr, qf, zero16());
    if (t + kWaves < t_end) load_rows<D>(kr, hK, (t + kWaves) * 32, l32, g);
    if (k0 + 31 > all_hi || (p.window > 0 && k0 <= q0 + 31 - p.window))
      mask_rows(s, key_lo - (k0 + 4 * g), key_hi - (k0 + 4 * g), -INFINITY);
    float mx = s[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    if (wave_any(mx > m_run + p.resc_th)) {
      const float m_new = fmaxf(m_run, mx);
      const float alpha = fast_exp2((m_run - m_new) * c);
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[dt][r] *= alpha;
      m_run = m_new;
    }
    const float mc = m_run * c;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = fast_exp2(fmaf(s[r], c, -mc));
      l_run += s[r];
    }
#pragma unroll
    for (int r = 0; r < 16; ++r)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) oacc[dt] = Mfma32<float>::mma(vc[r][dt], s[r], oacc[dt]);
    if (t + kWaves < t_end) load_cols<D>(vc, hV, (t + kWaves) * 32, l32, g);
  }

  // Merge the waves' (max, sum, O) in wave order: eight threads per row.
  const float l_tot = halves(l_run);
  if (g == 0) {
    ml[0][wave][l32] = m_run;
    ml[1][wave][l32] = l_tot;
  }
  put_partial<D>(part[wave], oacc, l32, g);
  __syncthreads();
  const int row = tid >> 3, qr = q0 + row;
  if (qr >= p.S) return;
  float m = ml[0][0][row], l = 0.f, wt[kWaves];
#pragma unroll
  for (int w = 1; w < kWaves; ++w) m = fmaxf(m, ml[0][w][row]);
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    wt[w] = fast_exp2((ml[0][w][row] - m) * c);
    l = fmaf(wt[w], ml[1][w][row], l);
  }
  const float inv = gate_sigmoid(p, b, qr, h) / l;
  float* dst = O + ((long long)b * p.S + qr) * p.q_rs + (long long)h * D;
#pragma unroll
  for (int i = 0; i < D / 32; ++i) {
    const int d = 4 * ((tid & 7) + 8 * i);
    f32x4 a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(&part[w][row * (D + 4) + d]);
#pragma unroll
      for (int e = 0; e < 4; ++e) a[e] = fmaf(wt[w], x[e], a[e]);
    }
    *reinterpret_cast<f32x4*>(dst + d) = f32x4{a[0] * inv, a[1] * inv, a[2] * inv, a[3] * inv};
  }
  if ((tid & 7) == 0) LSE[((long long)b * p.H + h) * p.S + qr] = m * p.scale + logf(l);
}

// dQ of 32 queries. With p.o it also computes their Delta = rowsum(dO * O) -
// dLSE and writes the workspace's two planes (Delta, -LSE / scale), which
// dK/dV reads: the backward then needs no delta launch.
template <int D, bool BLK>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(D <= 64 ? 2 : 1, 8)))
attn_f32_dq_kernel(const float* __restrict__ Q, const float* __restrict__ K,
                   const float* __restrict__ V, const float* __restrict__ dO,
                   const float* __restrict__ LSE, const float* __restrict__ Delta,
                   float* __restrict__ dQ, AttnParams p) {
  constexpr int DT = D / 32;
  __shared__ __attribute__((aligned(16))) float part[kWaves][32 * (D + 4)];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, g = lane >> 5;
  const WorkItem wi = work_item(p.nblk, p.B * p.H, p.div_wi, p.causal, p.wi_blocks_fastest);
  const int b = (int)fdiv((unsigned)wi.bh, p.div_h), h = wi.bh - b * p.H;
  const int hkv = (int)fdiv((unsigned)h, p.div_group);
  const int q0 = wi.blk * 32, qi = q0 + l32;

  const Head hK = head_of(K, b, p.S, p.kv_rs, hkv, D), hV = head_of(V, b, p.S, p.kv_rs, hkv, D);
  f32x4 qf[D / 8], dof[D / 8], kr[D / 8], vr[D / 8];
  float kc[16][DT];
  load_rows<D>(qf, head_of(Q, b, p.S, p.q_rs, h, D), q0, l32, g);
  load_rows<D>(dof, head_of(dO, b, p.S, p.q_rs, h, D), q0, l32, g);

  int kbeg = 0, kend = p.S;
  if (p.causal) kend = min(p.S, causal_key_end<BLK>(p, q0 + 31) + 1);
  if (p.window > 0) kbeg = max(0, q0 - p.window + 1);
  const int t_begin = kbeg / 32, t_end = (kend + 31) / 32;
  const int key_hi = p.causal ? min(causal_key_end<BLK>(p, qi), p.S - 1) : p.S - 1;
  const int key_lo = p.window > 0 ? qi - p.window + 1 : 0;
  const int all_hi = p.causal ? min(causal_key_end<BLK>(p, q0), p.S - 1) : p.S - 1;
  int t = t_begin + wave;
  if (t < t_end) {
    load_rows<D>(kr, hK, t * 32, l32, g);
    load_rows<D>(vr, hV, t * 32, l32, g);
    load_cols<D>(kc, hK, t * 32, l32, g);
  }

  const long long ridx = ((long long)b * p.H + h) * p.S + qi;
  float L2 = INFINITY, Dq = 0.f;
  if (p.o) {
    f32x4 of[D / 8];
    load_rows<D>(of, head_of(reinterpret_cast<const float*>(p.o), b, p.S, p.q_rs, h, D), q0, l32, g);
    float dot = 0.f;
#pragma unroll
    for (int j = 0; j < D / 8; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) dot = fmaf(of[j][e], dof[j][e], dot);
    Dq = halves(dot);
    if (qi < p.S) {
      const float L = LSE[ridx];
      L2 = L * kLog2e;
      if (p.dlse) Dq -= p.dlse[ridx];
      if (wave == 0 && g == 0) {
        p.ws_out[ridx] = Dq;
        p.ws_out[(long long)p.B * p.H * p.S + ridx] = L * (-1.f / p.scale);
      }
    }
  } else if (qi < p.S) {
    L2 = LSE[ridx] * kLog2e;
    Dq = Delta[ridx];
  }

  f32x16 dqacc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) dqacc[dt] = zero16();
  const float c = p.scale_log2;
  for (; t < t_end; t += kWaves) {
    const int k0 = t * 32;
    const bool more = t + kWaves < t_end;
    f32x16 s = dot_rows<D>(kr, qf, zero16());
    if (more) load_rows<D>(kr, hK, (t + kWaves) * 32, l32, g);
    f32x16 ds = dot_rows<D>(vr, dof, zero16());
    if (more) load_rows<D>(vr, hV, (t + kWaves) * 32, l32, g);
#pragma unroll
    for (int r = 0; r < 16; ++r) ds[r] = fast_exp2(fmaf(s[r], c, -L2)) * (ds[r] - Dq);
    if (k0 + 31 > all_hi || (p.window > 0 && k0 <= q0 + 31 - p.window))
      mask_rows(ds, key_lo - (k0 + 4 * g), key_hi - (k0 + 4 * g), 0.f);
#pragma unroll
    for (int r = 0; r < 16; ++r)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) dqacc[dt] = Mfma32<float>::mma(kc[r][dt], ds[r], dqacc[dt]);
    if (more) load_cols<D>(kc, hK, (t + kWaves) * 32, l32, g);
  }

  put_partial<D>(part[wave], dqacc, l32, g);
  __syncthreads();
  const int row = tid >> 3, qr = q0 + row;
  if (qr >= p.S) return;
  float* dst = dQ + ((long long)b * p.S + qr) * p.q_rs + (long long)h * D;
#pragma unroll
  for (int i = 0; i < D / 32; ++i) {
    const int d = 4 * ((tid & 7) + 8 * i);
    f32x4 a = *reinterpret_cast<const f32x4*>(&part[0][row * (D + 4) + d]);
#pragma unroll
    for (int w = 1; w < kWaves; ++w) a += *reinterpret_cast<const f32x4*>(&part[w][row * (D + 4) + d]);
    *reinterpret_cast<f32x4*>(dst + d) = a * p.scale;
  }
}

// dK / dV of 32 keys: the walk over (head of the group, query tile) is split.
template <int D, bool BLK>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(D <= 64 ? 2 : 1, 8)))
attn_f32_dkdv_kernel(const float* __restrict__ Q, const float* __restrict__ K,
                     const float* __restrict__ V, const float* __restrict__ dO,
                     const float* __restrict__ LSE, const float* __restrict__ Delta,
                     float* __restrict__ dK, float* __restrict__ dV, AttnParams p) {
  constexpr int DT = D / 32;
  __shared__ __attribute__((aligned(16))) float part[kWaves][32 * (D + 4)];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, g = lane >> 5;
  const WorkItem wi = work_item(p.nblk, p.B * p.Hkv, p.div_wi, false, p.wi_blocks_fastest);
  const int b = (int)fdiv((unsigned)wi.bh, p.div_hkv), hkv = wi.bh - b * p.Hkv;
  const int k0 = wi.blk * 32, kj = k0 + l32;

  f32x4 kf[D / 8], vf[D / 8];
  load_rows<D>(kf, head_of(K, b, p.S, p.kv_rs, hkv, D), k0, l32, g);
  load_rows<D>(vf, head_of(V, b, p.S, p.kv_rs, hkv, D), k0, l32, g);

  int qbeg = 0, qend = p.S;
  if (p.causal) qbeg = causal_query_begin<BLK>(p, k0);
  if (p.window > 0) qend = min(p.S, k0 + 31 + p.window);
  const int tq_begin = qbeg / 32;
  const int ntq = max(0, (qend + 31) / 32 - tq_begin);
  const int niter = p.group * ntq;
  const int q_lo = p.causal ? causal_query_begin<BLK>(p, kj) : 0;
  const int q_hi = p.window > 0 ? min(p.S - 1, kj + p.window - 1) : p.S - 1;
  // Queries that see every key of the block.
  const int all_lo = p.causal ? causal_query_begin<BLK>(p, k0 + 31) : 0;
  const int all_hi = p.window > 0 ? min(p.S - 1, k0 + p.window - 1) : p.S - 1;

  f32x16 dkacc[DT], dvacc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) {
    dkacc[dt] = zero16();
    dvacc[dt] = zero16();
  }
  const float c = p.scale_log2;
  f32x4 qr[D / 8], orr[D / 8];
  const Buf rows = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(LSE), 0, (int)((long long)p.B * p.H * p.S * 4), 0x00020000);
  const Buf deltas = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(Delta), 0, (int)((long long)p.B * p.H * p.S * 4), 0x00020000);
  // The next tile's rows are loaded under this tile's products where the
  // registers allow it (D = 32), else at the tile's start.
  constexpr bool AHEAD = D <= 32;
  // Iteration it: head hkv * group + it / ntq, query tile tq_begin + it % ntq.
  int gh = 0, tq = wave;
  auto settle = [&]() __attribute__((always_inline)) {
    while (tq >= ntq && gh < p.group) {
      tq -= ntq;
      ++gh;
    }
  };
  if (niter > 0) settle();
  if (AHEAD && wave < niter) {
    load_rows<D>(qr, head_of(Q, b, p.S, p.q_rs, hkv * p.group + gh, D), (tq_begin + tq) * 32, l32, g);
    load_rows<D>(orr, head_of(dO, b, p.S, p.q_rs, hkv * p.group + gh, D), (tq_begin + tq) * 32, l32, g);
  }
  for (int it = wave; it < niter; it += kWaves) {
    const int h = hkv * p.group + gh, q0 = (tq_begin + tq) * 32;
    const Head hQ = head_of(Q, b, p.S, p.q_rs, h, D), hO = head_of(dO, b, p.S, p.q_rs, h, D);
    float qc[16][DT], oc[16][DT];
    if constexpr (AHEAD) {
      load_cols<D>(oc, hO, q0, l32, g);
      load_cols<D>(qc, hQ, q0, l32, g);
    } else {
      load_rows<D>(qr, hQ, q0, l32, g);
      load_rows<D>(orr, hO, q0, l32, g);
    }
    f32x4 L4[4], D4[4];
    const unsigned voff = (unsigned)((((long long)b * p.H + h) * p.S + q0 + 4 * g) * 4);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      L4[j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rows, voff + 32u * j, 0, 0));
      D4[j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(deltas, voff + 32u * j, 0, 0));
    }
    f32x16 s = dot_rows<D>(qr, kf, zero16());
    f32x16 ds = dot_rows<D>(orr, vf, zero16());
    if constexpr (!AHEAD) {
      load_cols<D>(oc, hO, q0, l32, g);
      load_cols<D>(qc, hQ, q0, l32, g);
    }
    tq += kWaves;
    settle();
    if (AHEAD && it + kWaves < niter) {
      const int hn = hkv * p.group + gh;
      load_rows<D>(qr, head_of(Q, b, p.S, p.q_rs, hn, D), (tq_begin + tq) * 32, l32, g);
      load_rows<D>(orr, head_of(dO, b, p.S, p.q_rs, hn, D), (tq_begin + tq) * 32, l32, g);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = fast_exp2(fmaf(s[r], c, -(L4[r >> 2][r & 3] * kLog2e)));
      ds[r] = s[r] * (ds[r] - D4[r >> 2][r & 3]);
    }
    // Both are masked: past row S the LSE and Delta read here are another head's.
    if (q0 < all_lo || q0 + 31 > all_hi) {
      mask_rows(s, q_lo - (q0 + 4 * g), q_hi - (q0 + 4 * g), 0.f);
      mask_rows(ds, q_lo - (q0 + 4 * g), q_hi - (q0 + 4 * g), 0.f);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        dvacc[dt] = Mfma32<float>::mma(oc[r][dt], s[r], dvacc[dt]);
        dkacc[dt] = Mfma32<float>::mma(qc[r][dt], ds[r], dkacc[dt]);
      }
  }

  const int row = tid >> 3, kr = k0 + row;
  auto store = [&](float* base, const f32x16 (&acc)[DT], float sc) __attribute__((always_inline)) {
    put_partial<D>(part[wave], acc, l32, g);
    __syncthreads();
    if (kr < p.S) {
      float* dst = base + ((long long)b * p.S + kr) * p.kv_rs + (long long)hkv * D;
#pragma unroll
      for (int i = 0; i < D / 32; ++i) {
        const int d = 4 * ((tid & 7) + 8 * i);
        f32x4 a = *reinterpret_cast<const f32x4*>(&part[0][row * (D + 4) + d]);
#pragma unroll
        for (int w = 1; w < kWaves; ++w) a += *reinterpret_cast<const f32x4*>(&part[w][row * (D + 4) + d]);
        *reinterpret_cast<f32x4*>(dst + d) = a * sc;
      }
    }
  };
  store(dK, dkacc, p.scale);
  __syncthreads();
  store(dV, dvacc, 1.f);
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
namespace {

AttnParams f32_params(AttnParams p, long long heads) {
  p.nblk = (p.S + 31) / 32;
  p.wi_blocks_fastest = !p.causal;
  p.div_wi = p.wi_blocks_fastest ? work_item_div_blocks(p.nblk) : work_item_div(heads);
  return p;
}

template <typename F>
hipError_t f32_dispatch(int D, bool blk, F&& f) {
  auto by_blk = [&](auto d) {
    if (blk) f(d, std::true_type{});
    else f(d, std::false_type{});
    return hipGetLastError();
  };
  switch (D) {
    case 32: return by_blk(std::integral_constant<int, 32>{});
    case 64: return by_blk(std::integral_constant<int, 64>{});
    case 128: return by_blk(std::integral_constant<int, 128>{});
  }
  return hipErrorInvalidValue;
}

}  // namespace

// Modelled time of a launch here over that on the 128-row kernels: walk rows that the
// busiest of 256 CUs passes, whole workgroups to a CU (a causal launch's last ones
// are its shortest). Four waves of a 128-row workgroup each walk all of it, in
// 64-row tiles; here they share it in 32-row tiles.
static double split_share(const AttnParams& p, int heads) {
  const auto up = [](long long a, long long b) { return (a + b - 1) / b; };
  const long long bh = (long long)p.B * heads, n128 = up(p.S, 128), n32 = up(p.S, 32);
  if (p.window > 0 && p.window < p.S - 31) {
    const long long tiled = up(p.window + 127LL, 64) * 64 + 32, split = up(up(p.window + 31LL, 32) + 1, 4) * 32;
    return (double)(up(n32 * bh, 256) * split) / (double)(up(n128 * bh, 256) * tiled);
  }
  const long long all = up(p.S, 64) * 64, each = up(n32, 4) * 32;
  if (!p.causal) return (double)(up(n32 * bh, 256) * each) / (double)(up(n128 * bh, 256) * all);
  const long long m = n32 / 4, tiled = 64 * n128 * (n128 - 1) + all,
                  split = 32 * (2 * m * (m + 1) + (n32 % 4) * (m + 1));
  const long long t = up(bh * tiled, 256 * 128) * 128, u = up(bh * split, 256 * 32) * 32;
  return (double)(u > each ? u : each) / (double)(t > all ? t : all);
}

// Whether a float32 launch of `heads` (query heads; kv heads for dK/dV) takes these
// kernels. Two things decide (`grid` counts the 128-row kernels' workgroups, `walk` the
// rows of the other side a row can see). What the split saves: few workgroups, or rounds of
// them that end half empty, which split_share models. What it costs: a merge, the
// tiles that four waves no longer share (so more L2 traffic), and at D >= 64 one or
// two waves per SIMD (and 4 / 15 spilled registers in dQ / dK/dV at D = 64): little on a
// long walk, 10-25% on one of 100-250 rows of a chip that is full either way. The
// limits are measured over 2100 shapes, each pass and D: none taken is over 5%
// slower, three over 2.5%. 128-row kernels | these, fwd and bwd us, * the one taken:
//   causal  D64  grid 32    S256     28.7 |   8.7*    95.8 |  28.4*
//           D64  grid 768   S1024     158 |   126*     507 |   470*
//           D32  grid 768   S1024    86.8 |  64.6*     291 |   237*
//           D64  grid 504   S256                       137*|   151
//           D128 grid 288   S1024     182 |   119*     606 |   416*
//           D128 grid 1488  S256      271*|   276      984*|  1017
//           D128 grid 3072  S2048    2357 |  2228*    7995*|  8691
//   full    D64  grid 960   S1024     324 |   277*    1066 |   976*
//           D64  grid 1488  S256      142*|   140      488*|   557
//           D32  grid 1488  S256                       239*|   265
//           D64  grid 3000  S128      164*|   189
//           D128 grid 264   S256      109 |    79*     370 |   266*
//           D128 grid 252   S128     36.5*|  45.1      129*|   143
//   window  D64  grid 2048  256 of 4096 254 | 215*     843*|   861
//           D128 grid 192   64 of 2048 45.5 | 28.1*    158 |  99.8*
// Offsets inside a head and the row vectors are 32-bit here (S <= 2 GiB of rows); larger
// tensors stay with the others too.
bool f32_split_walk(const AttnParams& p, int D, int heads, bool backward) {
  const long long row_bytes = 4LL * (p.q_rs > p.kv_rs ? p.q_rs : p.kv_rs);
  if ((p.S + 32LL) * row_bytes > 0x7fffffffLL) return false;
  if (4LL * (p.S + 32LL) * p.B * p.H > 0x7fffffffLL) return false;
  const long long grid = (p.S + 127LL) / 128 * p.B * heads;
  const long long walk = p.window > 0 && p.window < p.S - 31 ? p.window + 31LL : p.S;
  if (grid >= 512) {
    if (!backward ? walk < 128 : walk < 256 || (grid >= 1536 && walk < 2048)) return false;
  }
  if (walk <= 64) return true;
  const long long rows = walk * (p.H / heads);   // dK/dV walks every query head of the group
  // Walks of one full 128-row workgroup and at most half of another.
  const bool half = walk > 128 && walk <= 192;
  const bool few = grid <= 448 && rows > 128;
  double limit = 9.0;
  if (!p.causal && backward) {
    if (D == 32 && (grid <= 256 || half)) limit = 9.0;
    else if (D == 64 && grid <= 256 && rows >= 384 && rows <= 512) limit = 1.01;
    else if (rows <= 128) limit = 0.7;
    else if (rows <= 256) limit = D == 32 ? 0.89 : 0.8;
    else if (rows <= (D == 128 ? 1024 : 512)) limit = 0.98;
  } else if (!p.causal) {
    if (D == 128) limit = walk <= 256 ? 0.85 : walk <= 400 ? 0.98 : 9.0;
    else if (walk <= 128) limit = grid <= 256 ? 1.01 : 0.9;
    else if (walk <= 256 && !half) limit = 0.95;
  } else if (backward) {
    if (D >= 64 && grid > 2048) return false;
    if (D >= 64 && rows <= 640 && !(few || (grid <= 448 && D == 64))) limit = 0.96;
  } else if (D == 128 && walk <= 512 && !few) {
    limit = 0.95;
  }
  return split_share(p, heads) <= limit;
}

hipError_t launch_f32_fwd(int D, const void* q, const void* k, const void* v, void* o, float* lse,
                          const AttnParams& pa, hipStream_t st) {
  const AttnParams p = f32_params(pa, (long long)pa.B * pa.H);
  const dim3 grid((unsigned)((long long)p.nblk * p.B * p.H));
  return f32_dispatch(D, p.block > 1, [&](auto d, auto blk) {
    hipLaunchKernelGGL((attn_f32_fwd_kernel<decltype(d)::value, decltype(blk)::value>), grid,
                       dim3(256), 0, st, (const float*)q, (const float*)k, (const float*)v,
                       (float*)o, lse, p);
  });
}

hipError_t launch_f32_dq(int D, const void* q, const void* k, const void* v, const void* dout,
                         const float* lse, const float* delta, void* dq, const AttnParams& pa,
                         hipStream_t st) {
  const AttnParams p = f32_params(pa, (long long)pa.B * pa.H);
  const dim3 grid((unsigned)((long long)p.nblk * p.B * p.H));
  return f32_dispatch(D, p.block > 1, [&](auto d, auto blk) {
    hipLaunchKernelGGL((attn_f32_dq_kernel<decltype(d)::value, decltype(blk)::value>), grid,
                       dim3(256), 0, st, (const float*)q, (const float*)k, (const float*)v,
                       (const float*)dout, lse, delta, (float*)dq, p);
  });
}

hipError_t launch_f32_dkdv(int D, const void* q, const void* k, const void* v, const void* dout,
                           const float* lse, const float* delta, void* dk, void* dv,
                           const AttnParams& pa, hipStream_t st) {
  const AttnParams p = f32_params(pa, (long long)pa.B * pa.Hkv);
  const dim3 grid((unsigned)((long long)p.nblk * p.B * p.Hkv));
  return f32_dispatch(D, p.block > 1, [&](auto d, auto blk) {
    hipLaunchKernelGGL((attn_f32_dkdv_kernel<decltype(d)::value, decltype(blk)::value>), grid,
                       dim3(256), 0, st, (const float*)q, (const float*)k, (const float*)v,
                       (const float*)dout, lse, delta, (float*)dk, (float*)dv, p);
  });
}

}  // namespace mi
