// Token embedding gather (forward) and deterministic scatter-add (backward) for gfx950 (SURVEY
// K1). Reference: the HF `nn.Embedding` of every model forward (src/training/train_*.py); eager
// PyTorch's backward materialises a dense [V, H] gradient (zero-fill + sort-based segment sum),
// then autograd adds it into `.grad`: two passes over V x H (1 GB at Llama-3's 128256 x 4096)
// per micro-batch for a few thousand touched rows.
//
// Forward: one wave per token row, 16-byte loads/stores (the table row is contiguous).
// Backward: the token ids arrive sorted (with the inverse permutation) from a device sort, so all
// occurrences of a token are adjacent. The wave at the FIRST position of each run sums the run's
// dY rows in sorted order (fixed order: bitwise reproducible, no float atomics) and adds the sum
// into the gradient row in place -- straight into the training engine's flat main-grad buffer
// (bf16 or fp32), so untouched rows cost nothing. The sorted positions are cut into chunks of
// kEmbChunk, one wave each: a run that lies inside one chunk is summed and added by that wave
// directly; a longer run (a frequent token) leaves one fp32 partial per chunk in a scratch slab,
// folded in chunk order by a second pass, so a hot token does not serialise the pass (cdna guide
// Appendix B "Scatter / gather / embedding": split long lists, sum per destination in a fixed order).
// What both passes cost is round trips, not bytes, so each wave first learns its runs from one load of ids (lane =
// position) and then asks for rows in batches. 8 x 1000 padded tokens of width 768: 45 + 148 us with loops over
// positions (one dependent load after the other; the pad id's run is the longest), 14 + 7 so; 4 x 1024 tokens of
// width 4096: 165 + 170 us, 21 + 8 so.
#include "common.h"

namespace dla {

constexpr int kEmbChunk = 16;  // sorted positions per backward wave

__global__ __launch_bounds__(256) void embed_fwd_kernel(const bf16_t* __restrict__ w, int64_t ldw,
                                                        const int64_t* __restrict__ ids, int64_t N,
                                                        int H, int64_t V, bf16_t* __restrict__ out,
                                                        int* __restrict__ bad) {
  const int64_t row = blockIdx.x * 4ll + (threadIdx.x >> 6);
  if (row >= N) return;
  const int lane = threadIdx.x & 63;
  const int64_t id = ids[row];
  bf16_t* dst = out + row * static_cast<int64_t>(H);
  if (id < 0 || id >= V) {
    // out-of-range id: never read outside the table. The row is zeros and the sticky error word
    // is set (vector store from lane 0); ops/embedding.py raises on it at the next host sync.
    for (int c = lane * 8; c < H; c += 512) store_bf16x8(dst + c, bf16x8{});
    if (lane == 0) bad[0] = 1;
    return;
  }
  const bf16_t* src = w + id * ldw;
  for (int c = lane * 8; c < H; c += 512) store_bf16x8(dst + c, load_bf16x8(src + c));
}

// lane `l`'s 64-bit value, wave-uniform
__device__ __forceinline__ int64_t emb_lane(int64_t v, int l) {
  const uint32_t lo = __builtin_amdgcn_readlane(static_cast<int>(v), l);
  const uint32_t hi = __builtin_amdgcn_readlane(static_cast<int>(v >> 32), l);
  return static_cast<int64_t>((static_cast<uint64_t>(hi) << 32) | lo);
}

template <typename G>
__device__ __forceinline__ void emb_store_sum(G* g, const G* old, const float* a) {
  if constexpr (sizeof(G) == 4) {
    *reinterpret_cast<f32x4*>(g) = f32x4{old[0] + a[0], old[1] + a[1], old[2] + a[2], old[3] + a[3]};
    *reinterpret_cast<f32x4*>(g + 4) = f32x4{old[4] + a[4], old[5] + a[5], old[6] + a[6], old[7] + a[7]};
  } else {
    float r[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) r[e] = bf2f(old[e]) + a[e];
    store_bf16x8(reinterpret_cast<bf16_t*>(g), pack_bf16x8(r));
  }
}
template <typename G>
__device__ __forceinline__ void emb_load8(const G* g, G* v) {
  if constexpr (sizeof(G) == 4) {
    const f32x4 x = *reinterpret_cast<const f32x4*>(g), y = *reinterpret_cast<const f32x4*>(g + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[e] = x[e];
      v[4 + e] = y[e];
    }
  } else {
    const bf16x8 x = load_bf16x8(reinterpret_cast<const bf16_t*>(g));
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = x[e];
  }
}

// Pass 1: wave per chunk of kEmbChunk sorted positions and 512 columns. Each run piece [p, q) in the chunk is
// summed in order; a run wholly inside the chunk is added into grad here, a piece of a run that
// crosses a chunk boundary goes to scratch[p] (fp32 [H]) for pass 2.
template <typename G>
__global__ __launch_bounds__(256) void embed_bwd_partial_kernel(
    const int64_t* __restrict__ sid, const int64_t* __restrict__ perm, const bf16_t* __restrict__ dy,
    int64_t N, int H, int64_t V, float* __restrict__ scratch, G* __restrict__ grad, int64_t ldg) {
  const int64_t chunk = blockIdx.x * 4ll + (threadIdx.x >> 6);
  const int64_t p0 = chunk * kEmbChunk;
  if (p0 >= N) return;
  const int lane = threadIdx.x & 63, c = blockIdx.y * 512 + lane * 8;
  const int n = static_cast<int>(N - p0 < kEmbChunk ? N - p0 : kEmbChunk);
  // lane l + 1: id of position p0 + l, with the neighbours on both sides (-1 past the ends; a table's id is >= 0)
  const int64_t at = p0 - 1 + lane;
  const int64_t id = lane <= kEmbChunk + 1 && at >= 0 && at < N ? sid[at] : -1;
  const int64_t row = lane < n ? perm[p0 + lane] : 0;
  const int64_t next = __shfl_down(id, 1, 64);
  const uint64_t edge = __builtin_amdgcn_ballot_w64(id != next);  // bit l: positions p0 + l - 1 and p0 + l differ
  const uint64_t valid = __builtin_amdgcn_ballot_w64(id >= 0 && id < V) >> 1;
  const bool open_lo = !(edge & 1);  // the chunk's first run starts before it
  const uint32_t ends = static_cast<uint32_t>(edge >> 1) & ((1u << n) - 1);  // position l is its run's last
  constexpr int KB = kEmbChunk / 2;  // rows asked for at a time
  float a[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  int start = 0;
  const bool in = c < H;
#pragma unroll
  for (int h = 0; h < kEmbChunk; h += KB) {
    bf16x8 v[KB];
    G old[KB][8];
#pragma unroll
    for (int k = 0; k < KB; ++k) {
      const int l = h + k;
      if (l >= n || !((valid >> l) & 1)) continue;  // (flagged by the forward: no gradient)
      if (in) v[k] = load_bf16x8(dy + emb_lane(row, l) * H + c);
      if (in && ((ends >> l) & 1)) emb_load8(grad + emb_lane(id, l + 1) * ldg + c, old[k]);
    }
#pragma unroll
    for (int k = 0; k < KB; ++k) {
      const int l = h + k;
      if (l >= n) continue;
      if ((valid >> l) & 1) {
        if (in) {
#pragma unroll
          for (int e = 0; e < 8; ++e) a[e] += bf2f(v[k][e]);
        }
        if (((ends >> l) & 1) || l == n - 1) {  // the run's last position, or the last of its piece here
          const bool whole = ((ends >> l) & 1) && !(start == 0 && open_lo);
          if (in && whole) {
            emb_store_sum(grad + emb_lane(id, l + 1) * ldg + c, old[k], a);
          } else if (in) {
            float* dst = scratch + (p0 + start) * H + c;
            *reinterpret_cast<f32x4*>(dst) = f32x4{a[0], a[1], a[2], a[3]};
            *reinterpret_cast<f32x4*>(dst + 4) = f32x4{a[4], a[5], a[6], a[7]};
          }
        }
      }
      if ((ends >> l) & 1) {
        start = l + 1;
#pragma unroll
        for (int e = 0; e < 8; ++e) a[e] = 0.f;
      }
    }
  }
}

// Pass 2: wave per chunk boundary and 512 columns. The first boundary inside a run (its head lies in the chunk before)
// folds the run's pieces (head, then each chunk start inside the run, in order) and adds them into grad[id].
template <typename G>
__global__ __launch_bounds__(256) void embed_bwd_fold_kernel(const int64_t* __restrict__ sid,
                                                             int64_t N, int H, int64_t V,
                                                             const float* __restrict__ scratch,
                                                             G* __restrict__ grad, int64_t ldg) {
  const int64_t b = (blockIdx.x * 4ll + (threadIdx.x >> 6) + 1) * kEmbChunk;
  if (b >= N) return;
  const int lane = threadIdx.x & 63, c = blockIdx.y * 512 + lane * 8;
  // lane l: id of position b - 17 + l
  const int64_t at = b - kEmbChunk - 1 + lane;
  const int64_t mine = lane <= kEmbChunk + 1 && at >= 0 ? sid[at] : -1;
  const int64_t id = emb_lane(mine, kEmbChunk + 1);
  if (id < 0 || id >= V) return;
  const uint64_t same = __builtin_amdgcn_ballot_w64(mine == id);
  if (!((same >> kEmbChunk) & 1) || (same & 1)) return;  // no run across b, or one that an earlier boundary folds
  const int64_t p = b - __builtin_popcountll(same & ((1ull << (kEmbChunk + 1)) - 1));  // (ids are sorted)
  // end of the run: the number of positions after b that hold its id, 64 probes at a time
  int64_t lo = b + 1, hi = N;  // first position in [lo, hi] that is not the run's
  while (lo < hi) {
    const int64_t step = (hi - lo + 63) >> 6, q = lo + lane * step;
    const int k = __builtin_popcountll(__builtin_amdgcn_ballot_w64(q < hi && sid[q] == id));
    if (k == 0) {
      hi = lo;
    } else {
      const int64_t past = lo + k * step;
      lo = lo + (k - 1) * step + 1;
      hi = past < hi ? past : hi;
    }
  }
  const int64_t end = lo;
  if (c >= H) return;
  G old[8];
  emb_load8(grad + id * ldg + c, old);
  float a[8];
  {
    const float* src = scratch + p * H + c;
    const f32x4 x0 = *reinterpret_cast<const f32x4*>(src), x1 = *reinterpret_cast<const f32x4*>(src + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      a[e] = 0.f + x0[e];
      a[4 + e] = 0.f + x1[e];
    }
  }
  const float* src = scratch + b * H + c;
  const int64_t step = static_cast<int64_t>(kEmbChunk) * H;
  int64_t left = (end - b + kEmbChunk - 1) / kEmbChunk;  // pieces from b on
  constexpr int U = 16;
  for (; left >= U; left -= U, src += U * step) {
    f32x4 x[U][2];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      x[u][0] = *reinterpret_cast<const f32x4*>(src + u * step);
      x[u][1] = *reinterpret_cast<const f32x4*>(src + u * step + 4);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < 8; ++e) a[e] += x[u][e >> 2][e & 3];
  }
  for (; left > 0; --left, src += step) {
    const f32x4 x0 = *reinterpret_cast<const f32x4*>(src), x1 = *reinterpret_cast<const f32x4*>(src + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      a[e] += x0[e];
      a[4 + e] += x1[e];
    }
  }
  emb_store_sum(grad + id * ldg + c, old, a);
}

void launch_embed_fwd(const bf16_t* w, int64_t ldw, const int64_t* ids, int64_t N, int H, int64_t V,
                      bf16_t* out, int* bad, hipStream_t st) {
  if (N == 0) return;
  embed_fwd_kernel<<<static_cast<unsigned>((N + 3) / 4), 256, 0, st>>>(w, ldw, ids, N, H, V, out, bad);
}

void launch_embed_bwd(const int64_t* sid, const int64_t* perm, const bf16_t* dy, int64_t N, int H,
                      int64_t V, float* scratch, void* grad, bool grad_f32, int64_t ldg, hipStream_t st) {
  if (N == 0) return;
  const int64_t chunks = (N + kEmbChunk - 1) / kEmbChunk;
  const unsigned cols = static_cast<unsigned>((H + 511) / 512);
  const dim3 g1(static_cast<unsigned>((chunks + 3) / 4), cols), g2(static_cast<unsigned>((chunks + 2) / 4), cols);
  if (grad_f32) {
    embed_bwd_partial_kernel<float><<<g1, 256, 0, st>>>(sid, perm, dy, N, H, V, scratch, static_cast<float*>(grad), ldg);
    if (chunks > 1) embed_bwd_fold_kernel<float><<<g2, 256, 0, st>>>(sid, N, H, V, scratch, static_cast<float*>(grad), ldg);
  } else {
    embed_bwd_partial_kernel<bf16_t><<<g1, 256, 0, st>>>(sid, perm, dy, N, H, V, scratch, static_cast<bf16_t*>(grad), ldg);
    if (chunks > 1) embed_bwd_fold_kernel<bf16_t><<<g2, 256, 0, st>>>(sid, N, H, V, scratch, static_cast<bf16_t*>(grad), ldg);
  }
}

}  // namespace dla
