// Decode projections on the fp32 residual stream (few rows): y = epilogue(rowscale o (a W^T)), bf16 a [M, K],
// W [N, K], M <= 64. One workgroup = 8 to 64 output columns, its waves over K (in-workgroup split, summed in
// wave order); what is around the product:
//
//   kStore    y = bf16
//   kRelu2    y = bf16(relu(.)^2)
//   kGate     y = bf16(gelu_tanh(.) * table[ids[m], off + n])
//   kStream   x[m, n] += .   (fp32 stream, in place);  y = bf16(x * (offset + norm_w[n])), or bf16(x);
//             ssq[m, block] = sum of x^2 over the block's columns
//   kPost     norms after the sums: x[m, n] holds the last sum, its norm x_prev = x * res_w * rstd(res_ssq) is
//             applied here; x <- alpha x_prev + . + bias;  y = bf16(x * norm_w[n]);  ssq as above
//   kGeglu    y = bf16(gelu_tanh(. gate) * . up), W = [gate rows; up rows]
//   kCap      y = fp32 cap * tanh(. / cap)
//
// A norm between two projections costs no launch: the producer (kStream, kPost) writes x * (offset + w)
// and the partial sums of squares, the consumer scales its rows by rsqrt(mean(x^2) + eps) (`ssq_in`).
//
// Bound by the weights' bytes, for small ones by a launch's fixed latency. Both operands arrive by LDS-DMA in
// rings that belong to one wave each (no barrier in the loop): a stage is 64 k, one instruction brings 8 rows x
// 128 bytes, i.e. whole cache lines with 8 consecutive lanes on each. Fragments read straight from memory put 16
// rows into 16 consecutive lanes, which costs the address path a cycle per lane: at 16 rows it moved 16 bytes
// per clock and CU, weights and activations together. The epilogue's operands are fetched before the loop.
// Measured in a replayed graph, us, direct fragments -> this (2048 x 8192 stream add, 8192 x 2048 relu^2,
// 2048 x 2048 stream add): 8 rows 15.2 -> 8.3, 9.9 -> 8.3, 6.2 -> 4.7; 16 rows 18.1 -> 10.3, 12.2 -> 9.9,
// 6.8 -> 5.1; 32 rows 26.2 -> 14.3, 18.2 -> 11.3, 8.8 -> 6.4.
#include "mix_params.h"
#include "mma.h"

namespace dla {
namespace {

enum { kStore = 0, kRelu2 = 1, kGate = 2, kStream = 3, kPost = 4, kGeglu = 5, kCap = 6 };

template <int N>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// 1 / rms of every row of a wave's share from n partial sums of squares of K columns: the first 256 of them are
// loaded by `RowScales` itself, side by side, and summed by `to`
template <int MT, int WV>
struct RowScales {
  static constexpr int R = (16 * MT + WV - 1) / WV;
  float v[R][4];
  __device__ __forceinline__ void load(const float* ssq, int n, int M) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
    for (int j = 0; j < R; ++j)
#pragma unroll
      for (int u = 0; u < 4; ++u)
        v[j][u] = lane + 64 * u < n ? ssq[static_cast<int64_t>(min(wave + j * WV, M - 1)) * n + lane + 64 * u] : 0.f;
  }
  __device__ __forceinline__ void to(float* rstd, const float* ssq, int n, int M, int K, float eps) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
    for (int j = 0; j < R; ++j) {
      float s = (v[j][0] + v[j][1]) + (v[j][2] + v[j][3]);
      for (int i = lane + 256; i < n; i += 64) s += ssq[static_cast<int64_t>(min(wave + j * WV, M - 1)) * n + i];
      s = wave_sum(s);
      if (lane == 0 && wave + j * WV < 16 * MT) rstd[wave + j * WV] = rsqrtf(s / K + eps);
    }
  }
};

// MG: groups of 8 rows of a. TC x NTL: columns per tile (8 or 16) x tiles. D: stages in a wave's ring. WV: waves.
template <int MG, int TC, int NTL, int D, int WV, int EPI>
__global__ __launch_bounds__(64 * WV) void stream_gemm_kernel(StreamGemmParams p) {
  constexpr int NW = EPI == kGeglu ? 2 : 1;  // weight rows per output column
  constexpr int CG = NTL * TC / 8, G = MG + NW * CG, MT = (MG + 1) / 2, NACC = NW * NTL * MT;
  static_assert(D >= 1 && D <= 4 && (D - 1) * G < 64, "loads in flight");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  __shared__ float rstd[16 * MT], rres[16 * MT];
  using M = Mma<bf16_t>;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * (TC * NTL);
  const int stages = (p.K + 63) / 64, per = (stages + WV - 1) / WV;
  const int s0 = wave * per, s1 = min(s0 + per, stages);
  // A ring slot holds G groups of 8 rows x 64 k. Lane l brings 16 bytes of row l / 8: chunk (l % 8) ^ (l / 8),
  // so that the fragments' reads (one chunk of 16 rows at a time) spread over the banks.
  bf16_t* ring = reinterpret_cast<bf16_t*>(smem) + wave * (D * G * 512);
  const int row8 = lane >> 3, ch = (lane & 7) ^ row8;
  const bf16_t* src[G];
#pragma unroll
  for (int i = 0; i < MG; ++i) src[i] = p.a + static_cast<int64_t>(min(8 * i + row8, p.M - 1)) * p.K;
#pragma unroll
  for (int i = 0; i < NW * CG; ++i)
    src[MG + i] = p.w + (static_cast<int64_t>(min(n0 + 8 * (i % CG) + row8, p.N - 1)) + static_cast<int64_t>(i / CG) * p.N) * p.K;
  auto issue = [&](int s, int slot) {
    int k = 64 * s + 8 * ch;
    k = k < p.K ? k : 0;  // (past K: any weights, times a's zeros below)
#pragma unroll
    for (int i = 0; i < G; ++i) {
      const auto* from = (const __attribute__((address_space(1))) void*)(src[i] + k);
      auto* to = (__attribute__((address_space(3))) void*)(ring + (slot * G + i) * 512);
      if (i >= MG && p.nt) __builtin_amdgcn_global_load_lds(from, to, 16, 0, 2);
      else __builtin_amdgcn_global_load_lds(from, to, 16, 0, 0);
    }
  };
  // this lane's outputs: entry ti = wave + o WV of (tile, row tile, i)
  constexpr int NO = (4 * MT * NTL + WV - 1) / WV;
  auto place = [&](int o, int& ti, int& m, int& n) {
    ti = wave + o * WV;
    m = 16 * ((ti >> 2) % MT) + 4 * g + (ti & 3);
    n = n0 + (ti >> 2) / MT * TC + r;
    return ti < 4 * MT * NTL && m < p.M && n < p.N && r < TC;
  };
  float xv[NO], cv[NO];  // the stream's value; the gate's factor or the bias
  bf16_t nw[NO], rw[NO];
  int64_t id[EPI == kGate ? NO : 1];
#pragma unroll
  for (int o = 0; o < NO; ++o) {
    int ti, m, n;
    const bool ok = place(o, ti, m, n);
    xv[o] = cv[o] = 0.f;
    nw[o] = rw[o] = 0;
    if constexpr (EPI == kStream || EPI == kPost) {
      if (ok) xv[o] = p.x[static_cast<int64_t>(m) * p.N + n];
      if (ok && p.norm_w) nw[o] = p.norm_w[n];
    }
    if constexpr (EPI == kPost) {
      if (ok && p.res_ssq) rw[o] = p.res_w[n];
      if (ok && p.bias) cv[o] = bf2f(p.bias[n]);
    }
    if constexpr (EPI == kGate) id[o] = ok ? p.ids[m] : -1;
  }
  RowScales<MT, WV> in_scale, res_scale;
  if (p.ssq_in) in_scale.load(p.ssq_in, p.nssq, p.M);
  if constexpr (EPI == kPost) {
    if (p.res_ssq) res_scale.load(p.res_ssq, p.nres, p.M);
  }
#pragma unroll
  for (int d = 0; d < D; ++d) issue(s0 + d, d);  // (a wave with fewer stages brings what it does not read)
  if constexpr (EPI == kGate) {  // (needs the ids: behind the first stages, not in front of them)
#pragma unroll
    for (int o = 0; o < NO; ++o) {
      int ti, m, n;
      place(o, ti, m, n);
      if (id[o] >= 0 && id[o] < p.vocab) cv[o] = bf2f(p.table[id[o] * p.ldt + p.off + n]);
    }
  }
  if (p.ssq_in) in_scale.to(rstd, p.ssq_in, p.nssq, p.M, p.K, p.eps);
  if constexpr (EPI == kPost) {
    if (p.res_ssq) res_scale.to(rres, p.res_ssq, p.nres, p.M, p.N, p.eps);
  }
  f32x4 acc[NACC];
#pragma unroll
  for (int i = 0; i < NACC; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  int slot = 0;
  for (int s = s0; s < s1; ++s) {
    // the oldest stage has landed once only the younger ones' loads are in flight
    const int young = min(D, s1 - s) - 1;
    if (D > 3 && young == 3) wait_loads<(D > 3 ? 3 * G : 0)>();
    else if (D > 2 && young == 2) wait_loads<(D > 2 ? 2 * G : 0)>();
    else if (D > 1 && young == 1) wait_loads<(D > 1 ? G : 0)>();
    else wait_loads<0>();
    const bf16_t* b = ring + slot * (G * 512);
    auto frag = [&](int group, int row, int h) {  // k 32 h + 8 g .. of a row
      return M::row(b + (group * 8 + row) * 64 + ((4 * h + g) ^ (row & 7)) * 8);
    };
    s16x8 af[2][MT], wf[2][NW * NTL];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int t = 0; t < MT; ++t) af[h][t] = frag(2 * t, 2 * t + 1 < MG ? r : r & 7, h);
#pragma unroll
      for (int q = 0; q < NW * NTL; ++q) wf[h][q] = frag(MG + q * (TC / 8), TC == 16 ? r : r & 7, h);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slot is read: its next stage may overwrite it
    if (s + D < s1) issue(s + D, slot);
    slot = slot + 1 == D ? 0 : slot + 1;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const bool in = 64 * s + 32 * h + 8 * g < p.K;
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const s16x8 a = in ? af[h][t] : M::zero();
#pragma unroll
        for (int q = 0; q < NW * NTL; ++q) acc[q * MT + t] = M::mma(a, wf[h][q], acc[q * MT + t]);
      }
    }
  }
  float* red = reinterpret_cast<float*>(smem);
  wait_loads<0>();
  __syncthreads();  // (every ring is read, and nothing is on its way into one)
#pragma unroll
  for (int q = 0; q < NACC; ++q)
#pragma unroll
    for (int i = 0; i < 4; ++i) red[((wave * NACC + q) * 4 + i) * 64 + lane] = acc[q][i];
  __syncthreads();
#pragma unroll
  for (int o = 0; o < NO; ++o) {
    int ti, m, n;
    const bool ok = place(o, ti, m, n);
    if (ti >= 4 * MT * NTL) continue;
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < WV; ++w) v += red[(w * NACC * 4 + ti) * 64 + lane];
    const float rs = p.ssq_in ? rstd[m] : 1.f;
    v *= rs;
    const int64_t at = static_cast<int64_t>(m) * p.N + n;
    if constexpr (EPI == kRelu2) {
      v = fmaxf(v, 0.f);
      v *= v;
    }
    if constexpr (EPI == kGate) v = gelu_tanh(v) * cv[o];
    if constexpr (EPI == kGeglu) {
      float up = 0.f;
#pragma unroll
      for (int w = 0; w < WV; ++w) up += red[((w * NACC + MT * NTL) * 4 + ti) * 64 + lane];
      v = gelu_tanh(v) * (up * rs);
    }
    if constexpr (EPI == kCap) {
      if (ok) p.yf[at] = p.cap * tanhf(v / p.cap);
      continue;
    }
    if constexpr (EPI == kStream || EPI == kPost) {
      float sq = 0.f;
      if (ok) {
        float x = xv[o];
        if constexpr (EPI == kPost) {
          if (p.res_ssq) x *= rres[m] * bf2f(rw[o]);
          x = p.alpha * x + v;
          if (p.bias) x += cv[o];
        } else {
          x += v;
        }
        p.x[at] = x;
        sq = x * x;
        v = p.norm_w ? x * (p.offset + bf2f(nw[o])) : x;
      }
#pragma unroll
      for (int d = 1; d < TC; d <<= 1) sq += __shfl_xor(sq, d, 64);
      // one partial sum per tile of TC columns
      if (r == 0 && m < p.M) p.ssq[static_cast<int64_t>(m) * (gridDim.x * NTL) + blockIdx.x * NTL + (ti >> 2) / MT] = sq;
    }
    if (ok) p.y[at] = f2bf(v);
  }
}

template <int MG, int TC, int NTL, int D, int WV, int EPI>
void go(const StreamGemmParams& p, hipStream_t st) {
  constexpr int NW = EPI == kGeglu ? 2 : 1, G = MG + NW * NTL * TC / 8, NACC = NW * NTL * ((MG + 1) / 2);
  constexpr int lds = WV * 1024 * (D * G > NACC ? D * G : NACC);
  static_assert(lds <= 150 * 1024, "LDS");
  if (lds > 64 * 1024)
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(stream_gemm_kernel<MG, TC, NTL, D, WV, EPI>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  stream_gemm_kernel<MG, TC, NTL, D, WV, EPI><<<(p.N + TC * NTL - 1) / (TC * NTL), 64 * WV, lds, st>>>(p);
}

enum Tile { kT8, kT16, kT16Deep, kT32, kT64 };

// Columns per workgroup. Every workgroup reads all of a for its columns, so wide tiles save L2 traffic and narrow
// ones fill the 256 CUs. us at 8 / 16 / 32 / 48 rows:
//   8 columns, up to 128 tiles of 16 (2048 x 8192: 8.5 / 10.3 / 14.2 / 18.7 against 10.1 / 12.1 / 16.1 / 20.2 with 16;
//   below K = 2048 there is nothing to share out: 2048 x 128 2.6 / 2.5 / 2.7 / 3.4 against 2.4 / 2.3 / 2.3 / 3.4);
//   32 columns from 17 rows on for more tiles than CUs (8192 x 2048: 10.1 / 11.9 at 32 / 48 rows against 14.4 / 17.6
//   with 16), and at 9 to 16 rows from 320 tiles on (5120 x 2048: 6.9 against 7.9);
//   64 columns from 33 rows on where 32 would not fit the CUs at once (16384 x 4096: 26.4 against 35.3 at 48 rows).
// Four waves with deeper rings instead of eight take long rows (4096 x 16384: 27.6 / 28.8 / 35.2 / 43.3 against 31.3 /
// 31.7 / 44.4 / 48.2) and, with few rows, many tiles (32000 x 2048: 21.7 against 23.7); two workgroups of them fit a
// CU where one of eight does, which decides at 17 to 32 rows beyond 256 workgroups (8208 x 2048: 257 of them).
Tile choose(const StreamGemmParams& p, int epi) {
  const int tiles = (p.N + 15) / 16, M = p.M;
  if (epi == kGeglu) return M <= 16 ? kT16Deep : kT32;
  if (epi == kGate || (tiles <= 128 && p.K >= 2048)) return kT8;
  if (p.K >= 8192) return kT16Deep;
  if (M <= 8) return tiles >= 1024 && p.K <= 2048 ? kT16Deep : kT16;
  if (M <= 16) return tiles >= 320 ? kT32 : kT16;
  if (M > 32 && tiles > 512) return kT64;
  return tiles > 256 ? kT32 : kT16;
}

template <int EPI>
void launch(const StreamGemmParams& p, Tile t, hipStream_t st) {
  const int M = p.M;
  if constexpr (EPI == kGeglu) {
    if (M <= 8) go<1, 16, 1, 3, 4, EPI>(p, st);
    else if (M <= 16) go<2, 16, 1, 3, 4, EPI>(p, st);
    else if (M <= 32) go<4, 16, 2, 1, 8, EPI>(p, st);
    else if (M <= 48) go<6, 16, 2, 1, 8, EPI>(p, st);
    else go<8, 16, 2, 1, 8, EPI>(p, st);
  } else {
    if (t == kT8) {
      if (M <= 8) go<1, 8, 1, 4, 8, EPI>(p, st);
      else if (M <= 16) go<2, 8, 1, 3, 8, EPI>(p, st);
      else if (M <= 32) go<4, 8, 1, 2, 8, EPI>(p, st);
      else if (M <= 48) go<6, 8, 1, 2, 8, EPI>(p, st);
      else go<8, 8, 1, 2, 8, EPI>(p, st);
    } else if constexpr (EPI != kGate) {
      if (t == kT16) {
        if (M <= 8) go<1, 16, 1, 2, 8, EPI>(p, st);
        else if (M <= 16) go<2, 16, 1, 2, 8, EPI>(p, st);
        else if (M <= 32) go<4, 16, 1, 2, 8, EPI>(p, st);
        else if (M <= 48) go<6, 16, 1, 2, 8, EPI>(p, st);
        else go<8, 16, 1, 2, 4, EPI>(p, st);
      } else if (t == kT16Deep) {
        if (M <= 8) go<1, 16, 1, 4, 4, EPI>(p, st);
        else if (M <= 16) go<2, 16, 1, 4, 4, EPI>(p, st);
        else if (M <= 32) go<4, 16, 1, 3, 4, EPI>(p, st);
        else if (M <= 48) go<6, 16, 1, 3, 4, EPI>(p, st);
        else go<8, 16, 1, 2, 4, EPI>(p, st);
      } else if (t == kT32) {
        if (M <= 16) go<2, 16, 2, 3, 4, EPI>(p, st);
        else if (M <= 32 && p.N > 32 * 256) go<4, 16, 2, 2, 4, EPI>(p, st);
        else if (M <= 32) go<4, 16, 2, 2, 8, EPI>(p, st);
        else if (M <= 48) go<6, 16, 2, 1, 8, EPI>(p, st);
        else go<8, 16, 2, 1, 8, EPI>(p, st);
      } else {
        if (M <= 48) go<6, 16, 4, 1, 8, EPI>(p, st);
        else go<8, 16, 4, 1, 8, EPI>(p, st);
      }
    }
  }
}

}  // namespace

int stream_gemm_partials(const StreamGemmParams& p, int epi) {
  const Tile t = choose(p, epi);
  if (t == kT8) return (p.N + 7) / 8;
  const int ntl = t == kT64 ? 4 : t == kT32 ? 2 : 1;
  return (p.N + 16 * ntl - 1) / (16 * ntl) * ntl;
}

void launch_stream_gemm(const StreamGemmParams& q, int epi, hipStream_t st) {
  StreamGemmParams p = q;
  // Weights are used once a step: from 8 MB on they pass the caches by (8192 x 2048 at 8 rows: 8.3 us against 8.7;
  // 16384 x 4096: 21.9 against 24.3; but 1344 x 2048: 4.0 against 3.6, 3072 x 768: 3.2 against 3.1)
  p.nt = static_cast<int64_t>(p.N) * p.K * (epi == kGeglu ? 4 : 2) >= 8 << 20;
  const Tile t = choose(p, epi);
  if (epi == kStore) launch<kStore>(p, t, st);
  else if (epi == kRelu2) launch<kRelu2>(p, t, st);
  else if (epi == kGate) launch<kGate>(p, t, st);
  else if (epi == kStream) launch<kStream>(p, t, st);
  else if (epi == kPost) launch<kPost>(p, t, st);
  else if (epi == kGeglu) launch<kGeglu>(p, t, st);
  else launch<kCap>(p, t, st);
}

}  // namespace dla
