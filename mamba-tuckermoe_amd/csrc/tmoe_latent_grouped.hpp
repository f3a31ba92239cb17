// The latent expert contraction (tmoe_latent.hpp) grouped by expert: each token meets
// only the k experts it selected instead of all E of them (bf16; r3 and r2 multiples
// of 128).
//
//   k_latent_count, k_latent_sort   the tokens ordered by their set of experts (k <= 2: the pair
//                    (lo, hi)), in row tiles of 128 tokens of one pair, and the B k
//                    (token, slot) entries ordered by expert, in chunks
//   k_latent_pair    C_j = A G_{e_j} for both slots j of a pair's tokens in one
//                    tile: forward (A = x) out = p_0 C_0 + p_1 C_1; backward
//                    (A = dout, G transposed) dx = p_0 C_0 + p_1 C_1 and
//                    dp_j = x . C_j, so no (B, E r3) product is stored
//   k_latent_scale   xs[i] = R(p x) of entry i, in expert order (the A rows of dG)
//   k_latent_dge     dG[e] = sum over e's entries of xs^T dout, one fp32 plane per
//                    chunk of entries; both operands have K (entries) as their slow
//                    axis and are read transposed from LDS (ds_read_b64_tr_b16)
//   k_latent_finish  dG = the sum of each expert's planes, in chunk order;
//                    dp = the sum of its column tiles' parts
//
// Measured at 16384 tokens, E 8, k 2, r3 256, r2 1024 (MI355X; one kernel trace of either form):
//   forward    pairs 38.7, sort 12.3, G's transpose among its counts (dense: product 67.8, G
//              transposed 5.6, weights 4.3)
//   dx and dp  39.1 (dense: H 83.5, dx / dp 30.9)
//   dG         xs 6.8, products 35.5, planes and dp 8.7, both sorts of the backward 10.9 (dense:
//              transposes 34.8, products 132.8, planes 5.3, weights and the zero bias 7.9)
// These kernel times add to 152 us (dense 373); a forward and backward in a stream without the
// trace take 149 (dense 348).
//
// The sort is a stable counting sort on integers, so every sum has a fixed order. An
// index outside [0, E) selects nothing (weight 0, dp 0).
#pragma once

#include "tmoe_latent.hpp"

namespace tmoe {
namespace dev {

constexpr int kLatBM = 128;              // tokens of a row tile of k_latent_pair
constexpr int kLatMaxE = 64;
constexpr int kLatMaxKeys = kLatMaxE * (kLatMaxE + 1) / 2;
constexpr int kLatSwap = 1 << 30;        // order[]: the token's slot 0 is the pair's hi

struct LatentSort {
  const int64_t* idx;
  const void* p;                // bf16 or fp32
  bool p_f32;
  int64_t B;
  int E, k;
  int pair_blocks, exp_blocks;  // work-groups of each sort (exp_blocks 0: forward)
  int chunk;                    // entries per dG chunk (at most)
  int *pair_hist, *exp_hist;    // key counts per work-group
  int* meta;                    // [0]: row tiles, [1]: dG chunks
  int4* tiles;                  // (start, tokens, expert lo, expert hi) per row tile
  int* order;                   // (B) token | kLatSwap, by pair
  int4* chunks;                 // (start, entries, expert, 0) per chunk
  int2* exp_chunks;             // (first chunk, chunks) per expert
  int* etok;                    // (B k) token of an entry, by expert
  float* ew;                    // (B k) its probability
};

// The pair of experts of token b (lo <= hi); swap: slot 0 selects hi.
__device__ __forceinline__ void latent_pair_of(const LatentSort& s, int64_t b, int& lo, int& hi,
                                               bool& swap) {
  const int64_t i0 = s.idx[b * s.k], i1 = s.k == 2 ? s.idx[b * 2 + 1] : i0;
  const bool v0 = i0 >= 0 && i0 < s.E, v1 = i1 >= 0 && i1 < s.E;
  const int a = v0 ? (int)i0 : (v1 ? (int)i1 : 0), c = v1 ? (int)i1 : a;
  swap = a > c;
  lo = swap ? c : a;
  hi = swap ? a : c;
}
// exclusive scan of v over the wave; total: the wave's sum
__device__ __forceinline__ int wave_scan_excl(int v, int lane, int& total) {
  int x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(x, o);
    if (lane >= o) x += y;
  }
  total = __shfl(x, 63);
  return x - v;
}

// A stable counting sort of n items over nblk <= kSortBlocks work-groups, in two
// launches: count_keys stores the key counts of range blk in row blk of hist; sort_range
// adds the rows (those of earlier ranges give its items' first places) and places its
// range, kSortSpan items at a time: the keys into LDS, their places by the first wave in
// order, the items by every thread. One launch whose work-groups each count every item
// took 16 us for 16384 tokens, its LDS atomics most of it.
// start[key] is the key's first place (start[nkeys] = n); emit(pos, i).
constexpr int kSortThreads = 256, kSortSpan = 1024, kSortBlocks = 64, kSortBatch = 16;
__device__ __forceinline__ void sort_span(int64_t n, int blk, int nblk, int64_t& lo, int64_t& hi) {
  const int64_t span = ((n + (int64_t)nblk * 64 - 1) / ((int64_t)nblk * 64)) * 64;
  lo = blk * span < n ? blk * span : n;
  hi = lo + span < n ? lo + span : n;
}
template <class Key>
__device__ __forceinline__ void count_keys(int64_t n, int nkeys, int blk, int nblk, int* cnt,
                                           int* hist, Key key) {
  const int tid = threadIdx.x, nt = (int)blockDim.x;
  int64_t lo, hi;
  sort_span(n, blk, nblk, lo, hi);
  for (int i = tid; i < nkeys; i += nt) cnt[i] = 0;
  __syncthreads();
  for (int64_t i = lo + tid; i < hi; i += nt) atomicAdd(cnt + key(i), 1);
  __syncthreads();
  for (int i = tid; i < nkeys; i += nt) hist[(int64_t)blk * nkeys + i] = cnt[i];
}
template <class Key, class Emit>
__device__ __forceinline__ void sort_range(int64_t n, int nkeys, int blk, int nblk, int* before,
                                           int* rest, int* start, int* span_buf, const int* hist,
                                           Key key, Emit emit) {
  constexpr int kItems = kSortSpan / kSortThreads, kParts = kSortBlocks / kSortBatch;
  const int tid = threadIdx.x, lane = tid & 63;
  int64_t lo, hi;
  sort_span(n, blk, nblk, lo, hi);
  // a thread's items of a span: key and payload, loaded ahead of the places
  int kk[kItems], pay[kItems];
  auto load = [&](int64_t s0, int m) {
#pragma unroll
    for (int u = 0; u < kItems; ++u) {
      const int i = tid + u * kSortThreads;
      if (i < m) kk[u] = key(s0 + i, pay[u]);
    }
  };
  auto span_of = [&](int64_t s0) { return (int)(hi - s0 < kSortSpan ? hi - s0 : kSortSpan); };
  if (lo < hi) load(lo, span_of(lo));
  for (int i = tid; i < nkeys; i += kSortThreads) before[i] = rest[i] = 0;
  __syncthreads();
  for (int t = tid; t < nkeys * kParts; t += kSortThreads) {   // kSortBatch rows of one key
    const int i = t % nkeys, r0 = t / nkeys * kSortBatch;
    int h[kSortBatch];
#pragma unroll
    for (int u = 0; u < kSortBatch; ++u)
      h[u] = hist[(int64_t)(r0 + u < nblk ? r0 + u : nblk - 1) * nkeys + i];
    int bf = 0, rs = 0;
#pragma unroll
    for (int u = 0; u < kSortBatch; ++u) {
      bf += r0 + u < blk ? h[u] : 0;
      rs += r0 + u >= blk && r0 + u < nblk ? h[u] : 0;
    }
    if (bf) atomicAdd(before + i, bf);
    if (rs) atomicAdd(rest + i, rs);
  }
  __syncthreads();
  if (tid < 64) {
    int carry = 0;
    for (int b = 0; b < nkeys; b += 64) {
      const int q = b + lane;
      const int bf = q < nkeys ? before[q] : 0;
      int total;
      const int ex = wave_scan_excl(q < nkeys ? bf + rest[q] : 0, lane, total) + carry;
      if (q < nkeys) {
        start[q] = ex;
        before[q] = ex + bf;   // the next place of this range's items
      }
      carry += total;
    }
    if (lane == 0) start[nkeys] = carry;
  }
  for (int64_t s0 = lo; s0 < hi; s0 += kSortSpan) {
    const int m = span_of(s0);
    if (s0 > lo) load(s0, m);
#pragma unroll
    for (int u = 0; u < kItems; ++u)
      if (tid + u * kSortThreads < m) span_buf[tid + u * kSortThreads] = kk[u];
    __syncthreads();
    if (tid < 64) {
      volatile int* next = before;
      for (int b = 0; b < m; b += 64) {
        const bool valid = b + lane < m;
        const int kv = valid ? span_buf[b + lane] : nkeys;
        uint64_t same = ~0ull;   // lanes with this lane's key
        for (int bit = 1; bit <= nkeys; bit <<= 1) {
          const uint64_t q = __ballot((kv & bit) != 0);
          same &= (kv & bit) ? q : ~q;
        }
        const int rank = __popcll(same & ((1ull << lane) - 1));
        if (valid) {
          const int pos = next[kv] + rank;
          span_buf[b + lane] = pos;
          if (rank == __popcll(same) - 1) next[kv] = pos + 1;
        }
        __builtin_amdgcn_wave_barrier();
      }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kItems; ++u)
      if (tid + u * kSortThreads < m)
        emit(span_buf[tid + u * kSortThreads], s0 + tid + u * kSortThreads, pay[u]);
    __syncthreads();
  }
}

__device__ __forceinline__ int latent_pair_keys(const LatentSort& s) {
  return s.k == 2 ? s.E * (s.E + 1) / 2 : s.E;
}
__device__ __forceinline__ int latent_pair_key(const LatentSort& s, int lo, int hi) {
  return s.k == 2 ? lo * s.E - lo * (lo - 1) / 2 + (hi - lo) : lo;
}
__device__ __forceinline__ int latent_key_of(const LatentSort& s, int64_t b, int& pay) {
  int lo, hi;
  bool sw;
  latent_pair_of(s, b, lo, hi, sw);
  pay = (int)b | (sw ? kLatSwap : 0);
  return latent_pair_key(s, lo, hi);
}
// an entry's expert; those that select nothing come last (key E)
__device__ __forceinline__ int latent_exp_of(const LatentSort& s, int64_t i) {
  const int64_t e = s.idx[i];
  return e >= 0 && e < s.E ? (int)e : s.E;
}

// The counts of both sorts; the work-groups past them transpose G (forward): GT (r2, E r3)
// in 32 x 32 tiles.
__global__ __launch_bounds__(kSortThreads) void k_latent_count(LatentSort s,
                                                               const uint16_t* __restrict__ G,
                                                               uint16_t* __restrict__ GT,
                                                               int64_t rows, int64_t cols) {
  __shared__ int cnt[kLatMaxKeys];
  const int tb = (int)blockIdx.x - s.pair_blocks - s.exp_blocks;
  if (tb >= 0) {
    uint16_t(*tile)[33] = reinterpret_cast<uint16_t(*)[33]>(cnt);
    const int nc = (int)(cols / 32);   // rows and cols are multiples of 32
    const int64_t r0 = (int64_t)(tb / nc) * 32, c0 = (int64_t)(tb % nc) * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    for (int y = ty; y < 32; y += 8) tile[y][tx] = G[(r0 + y) * cols + c0 + tx];
    __syncthreads();
    for (int y = ty; y < 32; y += 8) GT[(c0 + y) * rows + r0 + tx] = tile[tx][y];
    return;
  }
  if ((int)blockIdx.x < s.pair_blocks)
    count_keys(s.B, latent_pair_keys(s), (int)blockIdx.x, s.pair_blocks, cnt, s.pair_hist,
               [&](int64_t b) {
                 int pay;
                 return latent_key_of(s, b, pay);
               });
  else
    count_keys(s.B * s.k, s.E + 1, (int)blockIdx.x - s.pair_blocks, s.exp_blocks, cnt, s.exp_hist,
               [&](int64_t i) { return latent_exp_of(s, i); });
}

__global__ __launch_bounds__(kSortThreads) void k_latent_sort(LatentSort s) {
  __shared__ int before[kLatMaxKeys], rest[kLatMaxKeys], start[kLatMaxKeys + 1], buf[kSortSpan];
  const int tid = threadIdx.x, lane = tid & 63;
  if ((int)blockIdx.x < s.pair_blocks) {
    const int E = s.E, nkeys = latent_pair_keys(s);
    auto key_of = [&](int lo, int hi) { return latent_pair_key(s, lo, hi); };
    sort_range(
        s.B, nkeys, (int)blockIdx.x, s.pair_blocks, before, rest, start, buf, s.pair_hist,
        [&](int64_t b, int& pay) { return latent_key_of(s, b, pay); },
        [&](int pos, int64_t, int pay) { s.order[pos] = pay; });
    if (blockIdx.x != 0) return;
    __syncthreads();
    if (tid < 64) {   // rest[key] = the key's first row tile
      int carry = 0;
      for (int b = 0; b < nkeys; b += 64) {
        const int kk = b + lane;
        const int n = kk < nkeys ? (start[kk + 1] - start[kk] + kLatBM - 1) / kLatBM : 0;
        int total;
        const int ex = wave_scan_excl(n, lane, total);
        if (kk < nkeys) rest[kk] = ex + carry;
        carry += total;
      }
      if (lane == 0) s.meta[0] = carry;
    }
    __syncthreads();
    for (int t = tid; t < E * E; t += (int)blockDim.x) {
      const int lo = t / E, hi = t - lo * E;
      if (s.k == 2 ? hi < lo : hi != lo) continue;
      const int kk = key_of(lo, hi);
      int at = start[kk], left = start[kk + 1] - at;
      for (int r = rest[kk]; left > 0; ++r, at += kLatBM, left -= kLatBM)
        s.tiles[r] = make_int4(at, left < kLatBM ? left : kLatBM, lo, hi);
    }
    return;
  }
  // entries (b, j) by expert
  const int blk = (int)blockIdx.x - s.pair_blocks;
  sort_range(
      s.B * s.k, s.E + 1, blk, s.exp_blocks, before, rest, start, buf, s.exp_hist,
      [&](int64_t i, int& pay) {
        pay = __float_as_int(s.p_f32 ? static_cast<const float*>(s.p)[i]
                                     : load_as_f32(static_cast<const uint16_t*>(s.p) + i));
        return latent_exp_of(s, i);
      },
      [&](int pos, int64_t i, int pay) {
        s.etok[pos] = (int)(i / s.k);
        s.ew[pos] = __int_as_float(pay);
      });
  if (blk != 0) return;
  __syncthreads();
  if (tid < 64) {   // E <= 64: one lane per expert
    const int n = lane < s.E ? start[lane + 1] - start[lane] : 0;
    const int nch = (n + s.chunk - 1) / s.chunk;
    int total;
    const int first = wave_scan_excl(nch, lane, total);
    if (lane == 0) s.meta[1] = total;
    if (lane < s.E) {
      s.exp_chunks[lane] = make_int2(first, nch);
      int at = start[lane];
      for (int c = 0; c < nch; ++c) {   // even pieces
        const int end = start[lane] + (int)((int64_t)n * (c + 1) / nch);
        s.chunks[first + c] = make_int4(at, end - at, lane, 0);
        at = end;
      }
    }
  }
}

struct LatentPair {
  const char* A;          // x (B, r3) or dout (B, r2): K-contiguous rows
  int64_t a_row;          // bytes
  const char* Bt;         // rows of N, K-contiguous: forward G^T (r2, E r3), backward G
  int64_t b_row, b_exp;   // bytes between rows and between experts
  int nkt;                // K tiles of 64
  int N;                  // r2 or r3
  const int* meta;
  const int4* tiles;
  const int* order;
  const int64_t* idx;
  const void* p;
  bool p_f32;
  int E;
  uint16_t* out;          // (B, N)
  const uint16_t* x;      // backward: (B, N)
  float* dpp;             // backward: (parts, B k) partial dp, part = 32 columns of x
  int64_t dp_plane;       // B k
};

// One row tile (128 tokens of one pair) x 128 product columns: 128 / NSLOT columns of
// each slot's expert. 4 waves of 64 x 64; with two slots a wave's two column blocks are
// the same 32 columns of its slots' products, so that the weighted sum and dp stay in
// a lane. Bound by the latency of one K tile's DMA (about 1.2 us a K tile and round of
// work-groups), not by its 17 GFLOP (7 us) or its 306 MB from L2. Both operands arrive by LDS
// DMA (the token rows gathered by each lane's own row addresses) in two stages of one 64-wide
// K tile; 64 KB of LDS and <= 256 registers a wave put two work-groups on a compute unit,
// one's loads under the other's MFMAs.
template <int NSLOT, bool BWD>
__global__ __launch_bounds__(256, 2) void k_latent_pair(LatentPair q) {
  constexpr int CS = 128 / NSLOT;
  constexpr int kStage = 256 * 8;   // u32x4 slots: 128 A rows, 128 B rows
  __shared__ u32x4 smem[2 * kStage];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  // row tile rt's column tiles all run on XCD rt % 8: its gathered rows stay in that L2
  const int ncol = q.N / CS;
  const int i0 = (int)blockIdx.x >> 3;
  const int rt = (i0 / ncol) * 8 + ((int)blockIdx.x & 7), ct = i0 % ncol;
  if (rt >= q.meta[0]) return;
  const int4 d = q.tiles[rt];
  const char *ap[4], *bp[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int blk = wave * 4 + j, r = blk * 8 + (lane >> 3), ch = dma_chunk(lane, blk);
    const int tok = q.order[d.x + (r < d.y ? r : d.y - 1)] & (kLatSwap - 1);
    ap[j] = q.A + tok * q.a_row + ch * 16;
    const int slot = NSLOT == 2 ? (r >> 5) & 1 : 0;
    const int col = NSLOT == 2 ? ct * CS + (r >> 6) * 32 + (r & 31) : ct * CS + r;
    bp[j] = q.Bt + col * q.b_row + (slot ? d.w : d.z) * q.b_exp + ch * 16;
  }
  auto dma = [&](int stage) __attribute__((always_inline)) {
    u32x4* s = smem + stage * kStage;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      __builtin_amdgcn_global_load_lds((gbl_cvptr)ap[j], (lds_vptr)(s + (wave * 4 + j) * 64), 16, 0, 0);
      __builtin_amdgcn_global_load_lds((gbl_cvptr)bp[j], (lds_vptr)(s + 1024 + (wave * 4 + j) * 64),
                                       16, 0, 0);
      ap[j] += kTileKBytes;
      bp[j] += kTileKBytes;
    }
  };
  dma(0);
  // this lane's rows: the slots' probabilities, in the tile's expert order, and (backward)
  // its x values
  float pw[2][NSLOT];
  int64_t src[2];         // b k
  bool sw[2];             // the pair's first expert is the token's slot 1
  uint2 xv[2][NSLOT == 2 ? 4 : 8];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = wm * 64 + i * 32 + (lane & 31);
    const int o = q.order[d.x + (r < d.y ? r : d.y - 1)];
    const int64_t b = o & (kLatSwap - 1);
    sw[i] = (o & kLatSwap) != 0;
    src[i] = b * NSLOT;
#pragma unroll
    for (int j = 0; j < NSLOT; ++j) {
      const int64_t at = b * NSLOT + (NSLOT == 2 && sw[i] ? 1 - j : j);
      const int64_t e = q.idx[at];
      const float v = q.p_f32 ? static_cast<const float*>(q.p)[at]
                              : load_as_f32(static_cast<const uint16_t*>(q.p) + at);
      pw[i][j] = e >= 0 && e < q.E ? v : 0.f;
    }
    if constexpr (BWD) {
#pragma unroll
      for (int c = 0; c < (NSLOT == 2 ? 4 : 8); ++c) {
        const int col = ct * CS + wn * (NSLOT == 2 ? 32 : 64) + (c >> 2) * 32 + 8 * (c & 3) +
                        4 * (lane >> 5);
        xv[i][c] = *reinterpret_cast<const uint2*>(q.x + b * q.N + col);
      }
    }
  }
  f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = zero16();
  for (int kt = 0; kt < q.nkt; ++kt) {
    wait_vm_lds<0>();   // K tile kt is in LDS; this wave's reads of the other stage are done
    lds_barrier();
    if (kt + 1 < q.nkt) dma((kt + 1) & 1);
    const u32x4* s = smem + (kt & 1) * kStage;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const int ch = ks * 2 + (lane >> 5);
      u32x4 af[2], bf[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        af[i] = s[lds_slot(wm * 64 + i * 32 + (lane & 31), ch)];
        bf[i] = s[lds_slot(128 + wn * 64 + i * 32 + (lane & 31), ch)];
      }
      // transposed blocks: lane = token row, elements = 4 runs of 4 columns
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) mma(acc[i][j], bf[j], af[i], EltBF16{});
    }
  }
  mfma_drain();
  if constexpr (BWD) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int r = wm * 64 + i * 32 + (lane & 31);
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        float v = 0.f;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const uint2 u = xv[i][NSLOT == 2 ? c : 4 * j + c];
          v += bf16_bits_to_f32(u.x & 0xffffu) * acc[i][j][4 * c] +
               bf16_bits_to_f32(u.x >> 16) * acc[i][j][4 * c + 1] +
               bf16_bits_to_f32(u.y & 0xffffu) * acc[i][j][4 * c + 2] +
               bf16_bits_to_f32(u.y >> 16) * acc[i][j][4 * c + 3];
        }
        v += __shfl_xor(v, 32);
        if (lane < 32 && r < d.y) {
          const int slot = NSLOT == 2 ? (sw[i] ? 1 - j : j) : 0;
          const int part = NSLOT == 2 ? ct * 2 + wn : (ct * 2 + wn) * 2 + j;
          q.dpp[part * q.dp_plane + src[i] + slot] = v;
        }
      }
    }
  }
  // out tile (128 x CS bf16) through LDS, stored as 16-byte chunks of whole rows
  constexpr int RB = CS * 2 + 16;
  lds_barrier();
  char* st = reinterpret_cast<char*>(smem);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = wm * 64 + i * 32 + (lane & 31);
#pragma unroll
    for (int j = 0; j < 2 / NSLOT; ++j)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[e] = pw[i][0] * acc[i][j][4 * c + e];
          if constexpr (NSLOT == 2) v[e] += pw[i][1] * acc[i][1][4 * c + e];
        }
        const int col = wn * (64 / NSLOT) + j * 32 + 8 * c + 4 * (lane >> 5);
        uint2 u;
        u.x = pack_bf16x2(v[0], v[1]);
        u.y = pack_bf16x2(v[2], v[3]);
        *reinterpret_cast<uint2*>(st + r * RB + col * 2) = u;
      }
  }
  __syncthreads();
  constexpr int CPR = CS / 8;
  for (int c = tid; c < d.y * CPR; c += 256) {
    const int r = c / CPR, ch = c - r * CPR;
    const int64_t b = q.order[d.x + r] & (kLatSwap - 1);
    *reinterpret_cast<u32x4*>(q.out + b * q.N + ct * CS + ch * 8) =
        *reinterpret_cast<const u32x4*>(st + r * RB + ch * 16);
  }
}

// xs (n, r3): xs[i] = R(ew[i] x[etok[i]]), one 16-byte chunk a thread.
__global__ __launch_bounds__(256) void k_latent_scale(const uint16_t* __restrict__ x,
                                                      const int* __restrict__ etok,
                                                      const float* __restrict__ ew, int64_t n,
                                                      int r3, uint16_t* __restrict__ xs,
                                                      u32x4* __restrict__ zero, int zero_chunks) {
  const int cpr = r3 / 8;
  const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (c < zero_chunks) zero[c] = u32x4{0u, 0u, 0u, 0u};
  const int64_t i = c / cpr;
  if (i >= n) return;
  const int ch = (int)(c - i * cpr);
  const u32x4 v = *reinterpret_cast<const u32x4*>(x + (int64_t)etok[i] * r3 + ch * 8);
  const float w = ew[i];
  u32x4 o;
#pragma unroll
  for (int j = 0; j < 4; ++j)
    o[j] = pack_bf16x2(bf16_bits_to_f32(v[j] & 0xffffu) * w, bf16_bits_to_f32(v[j] >> 16) * w);
  *reinterpret_cast<u32x4*>(xs + i * r3 + ch * 8) = o;
}

struct LatentDg {
  const char* xs;         // (B k, r3) by expert
  const char* dout;       // (B, r2)
  const int* etok;
  const int* meta;
  const int4* chunks;
  const char* zero;       // 256 zero bytes
  float* planes;          // (chunks, r3, r2)
  int r3, r2;
};

// Plane of one chunk: a 128 (rows of G) x 128 tile, K = the chunk's entries in K tiles
// of 64. LDS holds both operands as they lie in memory, 64 entry rows of 256 bytes, by
// DMA (dout's rows gathered); an MFMA fragment (8 entries of one column a lane) is two
// transposed 64-bit reads. Within a K tile LDS row 4 (4 w + j) + s holds entry
// 16 w + 4 s + j (the same for both operands), so that a lane's DMA rows are four
// consecutive entries. Past the chunk's end both are a row of zeros: dout's last row again would
// give NaN where that row is not finite.
__global__ __launch_bounds__(256, 2) void k_latent_dge(LatentDg q) {
  constexpr int kStage = 2 * 64 * 16;   // u32x4 slots: 64 rows x 16 chunks, twice
  __shared__ u32x4 smem[2 * kStage];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int ntm = q.r3 / 128, ntn = q.r2 / 128, per = ntm * ntn;
  // a chunk's tiles share its rows: all on XCD chunk % 8
  const int i0 = (int)blockIdx.x >> 3;
  const int c = (i0 / per) * 8 + ((int)blockIdx.x & 7), t = i0 % per;
  if (c >= q.meta[1]) return;
  const int tm = t / ntn, tn = t - tm * ntn;
  const int4 d = q.chunks[c];
  const int sub = lane >> 4;
  const int chunk = tr_dma_chunk(lane);
  const int64_t a_row = (int64_t)q.r3 * 2, b_row = (int64_t)q.r2 * 2;
  const char* abase = q.xs + d.x * a_row + tm * 256 + chunk * 16;
  const char* bbase = q.dout + tn * 256 + chunk * 16;
  // entries past the end: a zero row of either
  const int64_t za = q.zero + chunk * 16 - abase, zb = q.zero + chunk * 16 - bbase;
  const int k0 = wave * 16 + sub * 4;   // this lane's first entry of a K tile
  const int nkt = (d.y + 63) / 64;
  int tok[4];
  auto load_tok = [&](int kt) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int k = kt * 64 + k0 + j;
      tok[j] = q.etok[d.x + (k < d.y ? k : d.y - 1)];
    }
  };
  const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) u32x4*)smem;
  auto dma = [&](int kt, int stage) __attribute__((always_inline)) {
    const uint32_t s = lds0 + stage * (kStage * 16);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int k = kt * 64 + k0 + j;
      const bool in = k < d.y;
      const int64_t oa = in ? k * a_row : za, ob = in ? tok[j] * b_row : zb;
      __builtin_amdgcn_global_load_lds((gbl_cvptr)(abase + oa),
                                       (lds_vptr)(size_t)(s + (wave * 4 + j) * 1024), 16, 0, 0);
      __builtin_amdgcn_global_load_lds((gbl_cvptr)(bbase + ob),
                                       (lds_vptr)(size_t)(s + 16384 + (wave * 4 + j) * 1024), 16, 0,
                                       0);
    }
  };
  f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = zero16();
  load_tok(0);
  dma(0, 0);
  load_tok(1);
  for (int kt = 0; kt < nkt; ++kt) {
    wait_vm_lds<0>();
    lds_barrier();
    const uint32_t sa = lds0 + (kt & 1) * (kStage * 16);
    const uint32_t sb = sa + 64 * 256;
    // the whole K tile's fragments, then the next tile's DMA, then the MFMAs: the
    // compiler waits for every DMA in flight before a transposed read (it takes them
    // for aliases), so none is issued ahead of the reads
    u32x4 af[4][2], bf[4][2];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        af[ks][i] = tr_frag(sa, ks, wm * 2 + i, lane);
        bf[ks][i] = tr_frag(sb, ks, wn * 2 + i, lane);
      }
    __builtin_amdgcn_sched_barrier(0);
    if (kt + 1 < nkt) {
      dma(kt + 1, (kt + 1) & 1);
      load_tok(kt + 2);
    }
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) mma(acc[i][j], af[ks][i], bf[ks][j], EltBF16{});
  }
  mfma_drain();
  // a lane holds one column of sixteen rows: 128-byte runs of two rows a store
  float* out = q.planes + ((int64_t)c * q.r3 + tm * 128) * q.r2 + tn * 128;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e)
        out[(int64_t)(wm * 64 + i * 32 + acc_row(lane, e)) * q.r2 + wn * 64 + j * 32 + (lane & 31)] =
            acc[i][j][e];
}

// dG (E, per) bf16 from the experts' planes, four values a thread; work-groups from dp_blk0
// on instead sum the `parts` planes of dp (n values; an index outside [0, E): 0).
__global__ __launch_bounds__(256) void k_latent_finish(const float* __restrict__ planes,
                                                       const int2* __restrict__ exp_chunks,
                                                       int64_t per, int64_t total,
                                                       uint16_t* __restrict__ dG, int dp_blk0,
                                                       const float* __restrict__ dpp, int parts,
                                                       int64_t n, const int64_t* __restrict__ idx,
                                                       int E, void* __restrict__ dp, bool p_f32) {
  if ((int)blockIdx.x >= dp_blk0) {
    const int64_t i = (int64_t)((int)blockIdx.x - dp_blk0) * 256 + threadIdx.x;
    if (i >= n) return;
    float v = 0.f;
    for (int c = 0; c < parts; ++c) v += dpp[c * n + i];
    const int64_t e = idx[i];
    if (!(e >= 0 && e < E)) v = 0.f;
    if (p_f32) static_cast<float*>(dp)[i] = v;
    else store_from_f32(static_cast<uint16_t*>(dp) + i, v);
    return;
  }
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= total) return;
  const int64_t e = i / per, at = i - e * per;
  const int2 ch = exp_chunks[e];
  float4 v = {0.f, 0.f, 0.f, 0.f};
  for (int c = 0; c < ch.y; ++c) {
    const float4 u = *reinterpret_cast<const float4*>(planes + (int64_t)(ch.x + c) * per + at);
    v.x += u.x; v.y += u.y; v.z += u.z; v.w += u.w;
  }
  uint2 o;
  o.x = pack_bf16x2(v.x, v.y);
  o.y = pack_bf16x2(v.z, v.w);
  *reinterpret_cast<uint2*>(dG + i) = o;
}

}  // namespace dev
}  // namespace tmoe
