// Dispatch plan: a stable counting sort of the R = T*k route slots by expert,
// built without any host synchronisation.
//
// The flat slot array is cut into blocks of EB consecutive slots. Inside a
// block, every expert owns an EB-bit mask in LDS marking the slots routed to
// it (OR is order independent, so the masks are deterministic). A slot's rank
// among the block's slots of the same expert is the popcount of the mask bits
// below it, which is exactly the stable order of argsort(stable=True).
// Pass 1 writes per-block expert counts (and per-block counts of invalid ids),
// pass 2 scans them into per-(block, expert) bases and writes the plan's error
// count, pass 3 rebuilds the masks and scatters. Passes 2 and 3 are one kernel
// up to 1024 experts, 65536 block counts and 2048 blocks, all three are one where a single
// block takes the slots, and pass 2 is a launch of one workgroup otherwise.
// Every counter is written, not accumulated, so a plan needs no clearing launch.
#include "common.h"
#include "plan.h"

namespace mx {
namespace {

__device__ __forceinline__ void build_masks(const int64_t *top_idx, int64_t slot0, int n_slots,
                                            int E, int words, uint32_t *mask,
                                            int32_t *lds_err) {
  for (int i = threadIdx.x; i < E * words; i += blockDim.x) mask[i] = 0;
  __syncthreads();
  for (int p = threadIdx.x; p < n_slots; p += blockDim.x) {
    const int64_t e = top_idx[slot0 + p];
    if (e >= 0 && e < E) {
      atomicOr(&mask[e * words + (p >> 5)], 1u << (p & 31));
    } else if (lds_err && e != MX_ROUTE_DROPPED) {
      atomicAdd(lds_err, 1);
    }
  }
  __syncthreads();
}

__global__ __launch_bounds__(256) void plan_count_kernel(const int64_t *top_idx, int64_t R,
                                                         int E, int EB, int32_t *block_counts,
                                                         int32_t *block_err) {
  extern __shared__ uint32_t mask[];
  __shared__ int32_t n_err;
  if (threadIdx.x == 0) n_err = 0;
  const int words = EB >> 5;
  const int64_t slot0 = static_cast<int64_t>(blockIdx.x) * EB;
  const int n_slots = static_cast<int>(min<int64_t>(EB, R - slot0));
  build_masks(top_idx, slot0, n_slots, E, words, mask, &n_err);  // syncs before and after
  if (threadIdx.x == 0) block_err[blockIdx.x] = n_err;
  for (int e = threadIdx.x; e < E; e += blockDim.x) {
    int c = 0;
    for (int w = 0; w < words; ++w) c += __popc(mask[e * words + w]);
    block_counts[static_cast<int64_t>(blockIdx.x) * E + e] = c;
  }
}

// Block-wide exclusive scan of one int64 per thread (blockDim.x == 1024).
__device__ int64_t block_exclusive_scan(int64_t v, int64_t *shared, int64_t *total) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  int64_t x = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int64_t y = __shfl_up(x, off, 64);
    if (lane >= off) x += y;
  }
  if (lane == 63) shared[wid] = x;
  __syncthreads();
  if (threadIdx.x == 0) {
    int64_t run = 0;
    for (int w = 0; w < static_cast<int>(blockDim.x >> 6); ++w) {
      const int64_t s = shared[w];
      shared[w] = run;
      run += s;
    }
    shared[16] = run;
  }
  __syncthreads();
  const int64_t r = shared[wid] + x - v;
  *total = shared[16];
  __syncthreads();
  return r;
}

// The plan's error count, and its copy for the host (system scope: the host
// sees it while the stream is still busy). As a launch of its own after the
// layer this store took 4 us, and as long as the last workgroup slot took to
// come free beside another stream's work (14 us beside a GEMM).
__device__ __forceinline__ void store_errors(int32_t n, int32_t *err, int32_t *host_err) {
  *err = n;
  if (host_err) __hip_atomic_store(host_err, n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// One workgroup of 1024 threads. Thread t owns experts t, t + 1024, ...
// (E <= kPlanMaxExperts); the exclusive scans over experts run chunk by chunk
// of 1024 in expert order, carrying the running total. With E <= 1024 the
// per-block counts are summed and turned into per-block bases by G groups of
// E threads, each over a contiguous range of blocks (G = min(16, 1024 / E));
// with more experts each thread walks all blocks for each of its experts.
// kEpt: experts per thread the kernel is compiled for (1 when E <= 1024).
template <int kEpt>
__global__ __launch_bounds__(1024) void plan_scan_kernel(
    const int32_t *block_counts, const int32_t *block_err, int n_blocks, int E, int64_t n_rows,
    int tile_m, const int64_t *counts_in, int32_t *block_base, int64_t *seg, int2 *tiles,
    int32_t *num_tiles, int2 *tiles2, int32_t *num_tiles2, int2 *tiles2m, int32_t *num_tiles2m,
    int2 *tilesr, int32_t *num_tilesr, int32_t *err_counter, int32_t *host_err,
    int64_t *counts_out,
    int64_t *starts_out, int32_t *offsets_out) {
  __shared__ int64_t scan_tmp[32];
  __shared__ int32_t part[1024];     // [group][expert] block-range counts (E <= 1024)
  __shared__ int64_t start_s[1024];  // expert starts (E <= 1024)
  __shared__ int32_t n_err;
  const int t = threadIdx.x;
  if (t == 0) n_err = 0;
  __syncthreads();
  if (block_err) {
    int32_t c = 0;
    for (int b = t; b < n_blocks; b += blockDim.x) c += block_err[b];
    if (c) atomicAdd(&n_err, c);
  }
  const int ept = (E + 1023) / 1024;
  const bool small = E <= 1024;
  const int G = counts_in || !small ? 1 : max(1, min(16, 1024 / E));
  const int ge = small ? t / E : 0, ee = small ? t - ge * E : 0;
  const bool gact = !counts_in && small && G > 1 && ge < G;
  const int b_lo = gact ? static_cast<int>(static_cast<int64_t>(n_blocks) * ge / G) : 0;
  const int b_hi = gact ? static_cast<int>(static_cast<int64_t>(n_blocks) * (ge + 1) / G) : 0;
  if (gact) {
    // Unrolled so that several block counts are in flight at once: the loop is
    // latency bound (one workgroup, 16+ loads per thread).
    int32_t c = 0;
#pragma unroll 8
    for (int b = b_lo; b < b_hi; ++b) c += block_counts[static_cast<int64_t>(b) * E + ee];
    part[t] = c;
  }
  __syncthreads();
  int64_t count[kEpt], start[kEpt], seg_lo[kEpt], seg_hi[kEpt];
  int64_t carry = 0;
#pragma unroll
  for (int c = 0; c < kEpt; ++c) {
    count[c] = start[c] = seg_lo[c] = seg_hi[c] = 0;
    if (c >= ept) continue;  // uniform across the workgroup
    const int e = t + 1024 * c;
    if (e < E) {
      if (counts_in) {
        count[c] = counts_in[e];
        if (count[c] < 0 || count[c] > n_rows) {
          atomicAdd(&n_err, 1);
          count[c] = count[c] < 0 ? 0 : n_rows;
        }
      } else if (G > 1) {
        for (int gg = 0; gg < G; ++gg) count[c] += part[gg * E + e];
      } else {
        for (int b = 0; b < n_blocks; ++b) count[c] += block_counts[static_cast<int64_t>(b) * E + e];
      }
    }
    int64_t chunk_total = 0;
    start[c] = carry + block_exclusive_scan(count[c], scan_tmp, &chunk_total);
    carry += chunk_total;
    seg_lo[c] = start[c];
    seg_hi[c] = start[c] + count[c];
    if (counts_in) {
      // Rows beyond num_rows are never touched, even if the counts disagree.
      if (seg_lo[c] > n_rows) seg_lo[c] = n_rows;
      if (seg_hi[c] > n_rows) seg_hi[c] = n_rows;
    }
  }
  if (counts_in && t == 0 && carry != n_rows) atomicAdd(&n_err, 1);
  if (small && t < E) start_s[t] = start[0];
  __syncthreads();
  if (gact) {
    int64_t run = start_s[ee];
    for (int gg = 0; gg < ge; ++gg) run += part[gg * E + ee];
#pragma unroll 8
    for (int b = b_lo; b < b_hi; ++b) {
      const int64_t i = static_cast<int64_t>(b) * E + ee;
      block_base[i] = static_cast<int32_t>(run);
      run += block_counts[i];
    }
  }
#pragma unroll
  for (int c = 0; c < kEpt; ++c) {
    const int e = t + 1024 * c;
    if (c >= ept || e >= E) continue;
    if (!counts_in && G == 1) {
      int64_t run = start[c];
      for (int b = 0; b < n_blocks; ++b) {
        const int64_t i = static_cast<int64_t>(b) * E + e;
        block_base[i] = static_cast<int32_t>(run);
        run += block_counts[i];
      }
    }
    seg[e] = seg_lo[c];
    seg[E + e] = seg_hi[c];
    if (counts_out) counts_out[e] = count[c];
    if (starts_out) starts_out[e] = start[c];
    if (offsets_out) offsets_out[e] = static_cast<int32_t>(start[c] + count[c]);
  }
  // Lists: 0 = tile_m-row tiles, 1 = 2*tile_m-row tiles over all rows;
  // 2 = 2*tile_m-row tiles over each expert's rows but a final remainder of
  // at most tile_m rows, 3 = one tile_m-row tile for that remainder.
  for (int list = 0; list < 4; ++list) {
    const int tm = list == 0 || list == 3 ? tile_m : 2 * tile_m;
    int2 *out = list == 0 ? tiles : list == 1 ? tiles2 : list == 2 ? tiles2m : tilesr;
    int64_t tcarry = 0;
#pragma unroll
    for (int c = 0; c < kEpt; ++c) {
      if (c >= ept) continue;  // uniform
      const int e = t + 1024 * c;
      const int64_t n = e < E ? seg_hi[c] - seg_lo[c] : 0;
      const int64_t full = n / (2 * tile_m), rem = n - full * 2 * tile_m;
      int64_t my_tiles, first = seg_lo[c];
      if (list <= 1)
        my_tiles = (n + tm - 1) / tm;
      else if (list == 2)
        my_tiles = full + (rem > tile_m ? 1 : 0);
      else {
        my_tiles = rem > 0 && rem <= tile_m ? 1 : 0;
        first = seg_lo[c] + full * 2 * tile_m;
      }
      int64_t chunk_tiles = 0;
      const int64_t tile0 = tcarry + block_exclusive_scan(my_tiles, scan_tmp, &chunk_tiles);
      tcarry += chunk_tiles;
      for (int64_t j = 0; j < my_tiles; ++j)
        out[tile0 + j] = make_int2(e, static_cast<int>(first + j * tm));
    }
    if (threadIdx.x == 0) {
      int32_t *num = list == 0 ? num_tiles : list == 1 ? num_tiles2 : list == 2 ? num_tiles2m
                                                                               : num_tilesr;
      *num = static_cast<int32_t>(tcarry);
    }
  }
  __syncthreads();
  if (t == 0) store_errors(n_err, err_counter, host_err);
}

template <int SCORE_DTYPE>
__global__ __launch_bounds__(256) void plan_scatter_kernel(
    const int64_t *top_idx, const void *top_scores, int64_t R, int k, int E, int EB,
    const int32_t *block_base, int64_t *sort_positions, int64_t *sorted_token_indices,
    void *sorted_scores, int64_t *inverse_order, int32_t *row_token, int32_t *row_slot) {
  extern __shared__ uint32_t lds[];
  const int words = EB >> 5;
  uint32_t *mask = lds;
  // Per-word popcount prefixes sit in LDS when they fit next to the masks;
  // otherwise (many experts, EB <= 256: at most 7 words below a slot) each
  // slot adds up the popcounts of the words below its own.
  const bool lds_prefix = plan_prefix_in_lds(E, EB);
  uint32_t *prefix = lds + E * words;
  const int64_t slot0 = static_cast<int64_t>(blockIdx.x) * EB;
  const int n_slots = static_cast<int>(min<int64_t>(EB, R - slot0));
  build_masks(top_idx, slot0, n_slots, E, words, mask, nullptr);
  if (lds_prefix) {
    for (int e = threadIdx.x; e < E; e += blockDim.x) {
      uint32_t run = 0;
      for (int w = 0; w < words; ++w) {
        prefix[e * words + w] = run;
        run += __popc(mask[e * words + w]);
      }
    }
    __syncthreads();
  }
  const int32_t *base = block_base + static_cast<int64_t>(blockIdx.x) * E;
  for (int p = threadIdx.x; p < n_slots; p += blockDim.x) {
    const int64_t i = slot0 + p;
    const int64_t e = top_idx[i];
    if (e < 0 || e >= E) {
      if (inverse_order) inverse_order[i] = -1;
      continue;
    }
    const int w = p >> 5;
    const uint32_t below = mask[e * words + w] & ((1u << (p & 31)) - 1u);
    uint32_t pre = 0;
    if (lds_prefix) {
      pre = prefix[e * words + w];
    } else {
      for (int w2 = 0; w2 < w; ++w2) pre += __popc(mask[e * words + w2]);
    }
    const int64_t pos = base[e] + pre + __popc(below);
    const int64_t tok = i / k;
    if (sort_positions) sort_positions[pos] = i;
    if (sorted_token_indices) sorted_token_indices[pos] = tok;
    if (sorted_scores) {
      if (SCORE_DTYPE == MX_DTYPE_BF16)
        reinterpret_cast<uint16_t *>(sorted_scores)[pos] =
            reinterpret_cast<const uint16_t *>(top_scores)[i];
      else
        reinterpret_cast<float *>(sorted_scores)[pos] = reinterpret_cast<const float *>(top_scores)[i];
    }
    if (inverse_order) inverse_order[i] = pos;
    row_token[pos] = static_cast<int32_t>(tok);
    row_slot[pos] = static_cast<int32_t>(i);
  }
}

// Inclusive scan over a wave.
__device__ __forceinline__ int32_t wave_scan(int32_t x) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int32_t y = __shfl_up(x, off, 64);
    x += lane >= off ? y : 0;
  }
  return x;
}

// Exclusive scans of N values per thread of a 1024-thread workgroup; `total`
// receives the sums. `shared` holds 16 values per scan.
template <int N>
__device__ __forceinline__ void wg_exclusive_scan(const int32_t (&v)[N], int32_t (&before)[N],
                                                  int32_t (&total)[N], int32_t *shared) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  int32_t x[N];
#pragma unroll
  for (int i = 0; i < N; ++i) x[i] = wave_scan(v[i]);
  __syncthreads();  // the last use of `shared`
  if (lane == 63) {
#pragma unroll
    for (int i = 0; i < N; ++i) shared[16 * i + wid] = x[i];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const int32_t s = wave_scan(lane < 16 ? shared[16 * i + lane] : 0);  // over the waves
    const int32_t mine = __shfl(s, wid > 0 ? wid - 1 : 0, 64);
    before[i] = (wid > 0 ? mine : 0) + x[i] - v[i];
    total[i] = __shfl(s, 15, 64);
  }
}

// The plan in one kernel after the block counts, or in one kernel altogether
// when a single block holds every slot (n_blocks == 1, no counts passed).
// Latency is all there is to it (a few hundred KB at most), so the scan is not
// a launch of one workgroup between the counting and the scattering blocks:
// every scattering block reads all the block counts itself (at most
// kFusedCounts of them, from L2) and scans the experts, and one more block
// writes the segments and the tile lists meanwhile. Kernel traces, 64 experts,
// count + scan + scatter against this: 64 slots 19.4 -> 6.6 us and 1024 slots 15.4 ->
// 9.7 (one launch for three), 16384 slots 23.1 -> 13.9, 131072 slots 24.8 -> 17.7;
// 65536 slots of 128 experts 28.5 -> 23.0. Kernel times alone, without the gaps between
// them, 256 experts: 38400 slots 26.0 -> 14.0, 65536 slots (65536 block counts, the
// most) 30.4 -> 20.7; 98304 slots of 128 experts 27.8 -> 18.8. (With 64-bit scans unrolled over the
// waves the kernel spilled, and took 12.7 us for the 64 slots.)
constexpr int kFusedCounts = 65536;
// And at most so many blocks: each reads the counts of all, blocks^2 * experts
// counts together. Plan call with 4 and 8 experts, three kernels against this: 2048
// blocks (8388608 slots) 1226 / 1170 and 739 / 706 us, 4096 blocks 2376 / 2476 and
// 1450 / 1492.
constexpr int kFusedBlocks = 2048;
// Mask bits (E * EB) of a block: masks and prefixes take 32 KB of LDS.
constexpr int kFusedBits = 131072;

struct PlanFused {
  const int64_t *top_idx;
  const void *top_scores;
  int64_t R;
  int k, E, EB, n_blocks;
  const int32_t *block_counts, *block_err;
  PlanView v;
  int32_t *host_err;
  int64_t *counts, *starts;
  int32_t *offsets;
  int64_t *sort_positions, *sorted_token_indices;
  void *sorted_scores;
  int64_t *inverse_order;
};

template <int SCORE_DTYPE>
__global__ __launch_bounds__(1024) void plan_fused_kernel(PlanFused a) {
  extern __shared__ uint32_t lds[];
  __shared__ int32_t scan_tmp[64], part[1024], before_s[1024], base_s[1024];
  __shared__ int32_t n_err;
  const int t = threadIdx.x, E = a.E, words = a.EB >> 5;
  const bool single = a.n_blocks == 1;
  const int blk = blockIdx.x;
  const bool scatters = blk < a.n_blocks, lists = blk == static_cast<int>(gridDim.x) - 1;
  uint32_t *mask = lds, *prefix = lds + E * words;
  const int64_t slot0 = static_cast<int64_t>(blk) * a.EB;
  const int n_slots = static_cast<int>(min<int64_t>(a.EB, a.R - slot0));
  if (t == 0) n_err = 0;
  int32_t total = 0;  // rows of expert t
  if (scatters) {
    build_masks(a.top_idx, slot0, n_slots, E, words, mask, &n_err);
    if (words <= 16) {
      if (t < E) {
        for (int w = 0; w < words; ++w) {
          prefix[t * words + w] = total;
          total += __popc(mask[t * words + w]);
        }
      }
    } else {
      for (int e = t >> 6; e < E; e += 16) {
        int32_t run = 0;
        for (int w0 = 0; w0 < words; w0 += 64) {
          const int w = w0 + (t & 63);
          const int32_t c = w < words ? __popc(mask[e * words + w]) : 0;
          const int32_t x = wave_scan(c);
          if (w < words) prefix[e * words + w] = run + x - c;
          run += __shfl(x, 63, 64);
        }
        if ((t & 63) == 0) part[e] = run;
      }
      __syncthreads();
      if (t < E) total = part[t];
      __syncthreads();
    }
  }
  int32_t before = 0;  // rows of expert t in the blocks before this one
  if (!single) {
    // Groups of E threads, each over a contiguous range of blocks.
    const int G = max(1, min(16, 1024 / E)), g = t / E, e = t - g * E;
    int32_t all = 0, mine = 0;
    if (g < G) {
      const int lo = a.n_blocks * g / G, hi = a.n_blocks * (g + 1) / G;
#pragma unroll 8
      for (int b = lo; b < hi; ++b) {
        const int32_t c = a.block_counts[static_cast<int64_t>(b) * E + e];
        all += c;
        mine += b < blk ? c : 0;
      }
    }
    __syncthreads();
    part[t] = all;
    before_s[t] = mine;
    __syncthreads();
    total = 0;
    if (t < E)
      for (int q = 0; q < G; ++q) {
        total += part[q * E + t];
        before += before_s[q * E + t];
      }
    if (lists) {
      int32_t c = 0;
      for (int b = t; b < a.n_blocks; b += 1024) c += a.block_err[b];
      if (c) atomicAdd(&n_err, c);
    }
  }
  int32_t start_[1], rows_[1];
  wg_exclusive_scan<1>({total}, start_, rows_, scan_tmp);
  const int32_t start = start_[0];
  if (t < E) base_s[t] = start + before;
  __syncthreads();
  if (lists) {
    if (t < E) {
      a.v.seg[t] = start;
      a.v.seg[E + t] = start + total;
      if (a.counts) a.counts[t] = total;
      if (a.starts) a.starts[t] = start;
      if (a.offsets) a.offsets[t] = start + total;
    }
    // Tile counts of expert t in the four lists (as in plan_scan_kernel).
    constexpr int M = kPlanTileM;
    const int32_t full = total / (2 * M), rem = total - full * 2 * M;
    const int32_t n[4] = {(total + M - 1) / M, full + (rem > 0 ? 1 : 0), full + (rem > M ? 1 : 0),
                          rem > 0 && rem <= M ? 1 : 0};
    int32_t at[4], num[4];
    wg_exclusive_scan<4>(n, at, num, scan_tmp);
    for (int j = 0; j < n[0]; ++j) a.v.tiles[at[0] + j] = make_int2(t, start + j * M);
    for (int j = 0; j < n[1]; ++j) a.v.tiles2[at[1] + j] = make_int2(t, start + j * 2 * M);
    for (int j = 0; j < n[2]; ++j) a.v.tiles2m[at[2] + j] = make_int2(t, start + j * 2 * M);
    if (n[3]) a.v.tilesr[at[3]] = make_int2(t, start + full * 2 * M);
    if (t == 0) {
      *a.v.num_tiles = num[0];
      *a.v.num_tiles2 = num[1];
      *a.v.num_tiles2m = num[2];
      *a.v.num_tilesr = num[3];
      store_errors(n_err, a.v.err, a.host_err);
    }
  }
  if (!scatters) return;
  for (int p = t; p < n_slots; p += 1024) {
    const int64_t i = slot0 + p;
    const int64_t e = a.top_idx[i];
    if (e < 0 || e >= E) {
      if (a.inverse_order) a.inverse_order[i] = -1;
      continue;
    }
    const int w = static_cast<int>(e) * words + (p >> 5);
    const uint32_t below = mask[w] & ((1u << (p & 31)) - 1u);
    const int32_t pos = base_s[e] + static_cast<int32_t>(prefix[w]) + __popc(below);
    const uint32_t tok = static_cast<uint32_t>(i) / static_cast<uint32_t>(a.k);  // i < 2^31
    if (a.sort_positions) a.sort_positions[pos] = i;
    if (a.sorted_token_indices) a.sorted_token_indices[pos] = tok;
    if (a.sorted_scores) {
      if (SCORE_DTYPE == MX_DTYPE_BF16)
        reinterpret_cast<uint16_t *>(a.sorted_scores)[pos] =
            reinterpret_cast<const uint16_t *>(a.top_scores)[i];
      else
        reinterpret_cast<float *>(a.sorted_scores)[pos] =
            reinterpret_cast<const float *>(a.top_scores)[i];
    }
    if (a.inverse_order) a.inverse_order[i] = pos;
    a.v.row_token[pos] = static_cast<int32_t>(tok);
    a.v.row_slot[pos] = static_cast<int32_t>(i);
  }
}

// Slots per block when one block takes all R slots (a multiple of 32), or 0
// when it cannot. 4096 slots take one workgroup about as long as a counting
// launch of its own.
inline int single_block_slots(int E, int64_t R) {
  const int64_t eb = (R + 31) / 32 * 32;
  return E <= 1024 && R <= 4096 && E * eb <= kFusedBits ? static_cast<int>(eb) : 0;
}

constexpr int kPlanMaxEpt = kPlanMaxExperts / 1024;

}  // namespace

int slots_per_plan_block(int num_experts, int64_t rows) {
  // Masks + prefixes of E * EB bits each must fit in 64 KiB of LDS, and large
  // route counts are cut into at least 256 blocks (one workgroup per CU).
  int eb = 4096;
  while (eb > 256 && (static_cast<int64_t>(num_experts) * eb > 262144 || ceil_div(rows, eb) < 256))
    eb >>= 1;
  if (static_cast<int64_t>(num_experts) * eb <= 262144) return eb;
  // More than 1024 experts: the masks alone fill the 64 KiB (prefixes are
  // recounted per slot), so the blocks shrink to 32..128 slots.
  while (eb > 32 && static_cast<int64_t>(num_experts) * eb > 524288) eb >>= 1;
  return eb;
}

PlanLayout plan_layout(int64_t num_rows, int num_experts) {
  PlanLayout L;
  L.rows = num_rows;
  L.experts = num_experts;
  L.slots_per_block = slots_per_plan_block(num_experts, num_rows);
  L.blocks = static_cast<int>(ceil_div(num_rows, L.slots_per_block));
  L.max_tiles = ceil_div(num_rows, kPlanTileM) + num_experts;
  L.max_tiles2 = ceil_div(num_rows, kPlanTileM2) + num_experts;
  size_t off = 256;  // header: error counter, tile count
  L.off_block_counts = off;
  off = align_up(off + sizeof(int32_t) * L.blocks * num_experts, 256);
  L.off_block_base = off;
  off = align_up(off + sizeof(int32_t) * L.blocks * num_experts, 256);
  L.off_seg = off;
  off = align_up(off + sizeof(int64_t) * 2 * num_experts, 256);
  L.off_tiles = off;
  off = align_up(off + sizeof(int2) * L.max_tiles, 256);
  L.off_tiles2 = off;
  off = align_up(off + sizeof(int2) * L.max_tiles2, 256);
  L.off_tiles2m = off;
  off = align_up(off + sizeof(int2) * L.max_tiles2, 256);
  L.off_tilesr = off;
  off = align_up(off + sizeof(int2) * num_experts, 256);
  L.off_row_token = off;
  off = align_up(off + sizeof(int32_t) * num_rows, 256);
  L.off_row_slot = off;
  off = align_up(off + sizeof(int32_t) * num_rows, 256);
  L.off_block_err = off;
  off = align_up(off + sizeof(int32_t) * L.blocks, 256);
  L.bytes = off;
  return L;
}

PlanView plan_view(void *ws, const PlanLayout &L) {
  char *b = static_cast<char *>(ws);
  PlanView v;
  v.err = reinterpret_cast<int32_t *>(b);
  v.num_tiles = reinterpret_cast<int32_t *>(b) + 1;
  v.num_tiles2 = reinterpret_cast<int32_t *>(b) + 2;
  v.num_tiles2m = reinterpret_cast<int32_t *>(b) + 3;
  v.num_tilesr = reinterpret_cast<int32_t *>(b) + 4;
  v.block_counts = reinterpret_cast<int32_t *>(b + L.off_block_counts);
  v.block_base = reinterpret_cast<int32_t *>(b + L.off_block_base);
  v.seg = reinterpret_cast<int64_t *>(b + L.off_seg);
  v.tiles = reinterpret_cast<int2 *>(b + L.off_tiles);
  v.tiles2 = reinterpret_cast<int2 *>(b + L.off_tiles2);
  v.tiles2m = reinterpret_cast<int2 *>(b + L.off_tiles2m);
  v.tilesr = reinterpret_cast<int2 *>(b + L.off_tilesr);
  v.row_token = reinterpret_cast<int32_t *>(b + L.off_row_token);
  v.row_slot = reinterpret_cast<int32_t *>(b + L.off_row_slot);
  v.block_err = reinterpret_cast<int32_t *>(b + L.off_block_err);
  return v;
}

int build_plan(const int64_t *top_idx, const void *top_scores, int score_dtype,
               int64_t num_tokens, int top_k, int num_experts, int64_t *counts, int64_t *starts,
               int32_t *offsets, int64_t *sort_positions, int64_t *sorted_token_indices,
               void *sorted_scores, int64_t *inverse_order, void *workspace, hipStream_t s,
               int32_t *host_err) {
  const int64_t R = num_tokens * top_k;
  const PlanLayout L = plan_layout(R, num_experts);
  const PlanView v = plan_view(workspace, L);
  const int eb1 = R > 0 ? single_block_slots(num_experts, R) : 0;
  if (L.blocks > 0 && eb1 == 0) {
    const size_t lds = sizeof(uint32_t) * num_experts * (L.slots_per_block / 32);
    hipLaunchKernelGGL(plan_count_kernel, dim3(L.blocks), dim3(256), lds, s, top_idx, R,
                       num_experts, L.slots_per_block, v.block_counts, v.block_err);
  }
  // The fused kernel takes one expert per thread.
  if (eb1 > 0 || (L.blocks > 1 && num_experts <= 1024 &&
                  num_experts * L.slots_per_block <= kFusedBits && L.blocks <= kFusedBlocks &&
                  static_cast<int64_t>(L.blocks) * num_experts <= kFusedCounts)) {
    PlanFused a = {};
    a.top_idx = top_idx;
    a.top_scores = top_scores;
    a.R = R;
    a.k = top_k;
    a.E = num_experts;
    a.EB = eb1 > 0 ? eb1 : L.slots_per_block;
    a.n_blocks = eb1 > 0 ? 1 : L.blocks;
    a.block_counts = v.block_counts;
    a.block_err = v.block_err;
    a.v = v;
    a.host_err = host_err;
    a.counts = counts;
    a.starts = starts;
    a.offsets = offsets;
    a.sort_positions = sort_positions;
    a.sorted_token_indices = sorted_token_indices;
    a.sorted_scores = top_scores ? sorted_scores : nullptr;
    a.inverse_order = inverse_order;
    const size_t lds = 2 * sizeof(uint32_t) * num_experts * (a.EB / 32);
    const dim3 grid(eb1 > 0 ? 1 : L.blocks + 1);
    if (score_dtype == MX_DTYPE_BF16)
      hipLaunchKernelGGL(plan_fused_kernel<MX_DTYPE_BF16>, grid, dim3(1024), lds, s, a);
    else
      hipLaunchKernelGGL(plan_fused_kernel<MX_DTYPE_F32>, grid, dim3(1024), lds, s, a);
    return check_launch("mx_build_plan");
  }
  hipLaunchKernelGGL(num_experts <= 1024 ? plan_scan_kernel<1> : plan_scan_kernel<kPlanMaxEpt>,
                     dim3(1), dim3(1024), 0, s, v.block_counts,
                     L.blocks > 0 ? v.block_err : static_cast<int32_t *>(nullptr), L.blocks,
                     num_experts, R,
                     kPlanTileM, static_cast<const int64_t *>(nullptr), v.block_base, v.seg,
                     v.tiles, v.num_tiles, v.tiles2, v.num_tiles2, v.tiles2m, v.num_tiles2m,
                     v.tilesr, v.num_tilesr, v.err, host_err, counts, starts, offsets);
  if (L.blocks > 0) {
    const size_t lds = (plan_prefix_in_lds(num_experts, L.slots_per_block) ? 2 : 1) *
                       sizeof(uint32_t) * num_experts * (L.slots_per_block / 32);
    if (score_dtype == MX_DTYPE_BF16)
      hipLaunchKernelGGL(plan_scatter_kernel<MX_DTYPE_BF16>, dim3(L.blocks), dim3(256), lds, s,
                         top_idx, top_scores, R, top_k, num_experts, L.slots_per_block,
                         v.block_base, sort_positions, sorted_token_indices,
                         top_scores ? sorted_scores : nullptr, inverse_order, v.row_token,
                         v.row_slot);
    else
      hipLaunchKernelGGL(plan_scatter_kernel<MX_DTYPE_F32>, dim3(L.blocks), dim3(256), lds, s,
                         top_idx, top_scores, R, top_k, num_experts, L.slots_per_block,
                         v.block_base, sort_positions, sorted_token_indices,
                         top_scores ? sorted_scores : nullptr, inverse_order, v.row_token,
                         v.row_slot);
  }
  return check_launch("mx_build_plan");
}

int plan_from_counts(const int64_t *counts, int64_t num_rows, int num_experts, void *workspace,
                     hipStream_t s) {
  const PlanLayout L = plan_layout(num_rows, num_experts);
  const PlanView v = plan_view(workspace, L);
  hipLaunchKernelGGL(num_experts <= 1024 ? plan_scan_kernel<1> : plan_scan_kernel<kPlanMaxEpt>,
                     dim3(1), dim3(1024), 0, s,
                     static_cast<const int32_t *>(nullptr), static_cast<const int32_t *>(nullptr),
                     0, num_experts, num_rows,
                     kPlanTileM, counts, static_cast<int32_t *>(nullptr), v.seg, v.tiles,
                     v.num_tiles, v.tiles2, v.num_tiles2, v.tiles2m, v.num_tiles2m, v.tilesr,
                     v.num_tilesr, v.err, static_cast<int32_t *>(nullptr),
                     static_cast<int64_t *>(nullptr),
                     static_cast<int64_t *>(nullptr), static_cast<int32_t *>(nullptr));
  return check_launch("mx_plan_from_counts");
}

int validate_plan_args(const char *name, int64_t num_tokens, int top_k, int num_experts) {
  if (num_tokens < 0 || top_k <= 0 || top_k > 16) {
    set_error("%s: need num_tokens >= 0 and top_k in [1, 16]", name);
    return MX_ERR_INVALID;
  }
  if (num_experts <= 0 || num_experts > kPlanMaxExperts) {
    set_error("%s: num_experts must be in [1, %d], got %d", name, kPlanMaxExperts, num_experts);
    return MX_ERR_INVALID;
  }
  if (num_tokens * top_k >= (int64_t(1) << 31)) {
    set_error("%s: num_tokens * top_k must stay below 2^31", name);
    return MX_ERR_INVALID;
  }
  return MX_OK;
}

}  // namespace mx

using namespace mx;

extern "C" size_t mx_plan_workspace_size(int64_t num_tokens, int top_k, int num_experts) {
  if (num_tokens < 0 || top_k <= 0 || num_experts <= 0) return 0;
  return plan_layout(num_tokens * top_k, num_experts).bytes;
}

extern "C" int mx_build_plan(const int64_t *top_idx, const void *top_scores, int score_dtype,
                             int64_t num_tokens, int top_k, int num_experts, int64_t *counts,
                             int64_t *starts, int32_t *offsets, int64_t *sort_positions,
                             int64_t *sorted_token_indices, void *sorted_scores,
                             int64_t *inverse_order, void *workspace, void *stream) {
  clear_error();
  int rc = validate_plan_args("mx_build_plan", num_tokens, top_k, num_experts);
  if (rc) return rc;
  if (!workspace || (num_tokens > 0 && !top_idx)) {
    set_error("mx_build_plan: top_idx and workspace must be non-null");
    return MX_ERR_INVALID;
  }
  if (sorted_scores && !top_scores) {
    set_error("mx_build_plan: sorted_scores requires top_scores");
    return MX_ERR_INVALID;
  }
  return build_plan(top_idx, top_scores, score_dtype, num_tokens, top_k, num_experts, counts,
                    starts, offsets, sort_positions, sorted_token_indices, sorted_scores,
                    inverse_order, workspace, as_stream(stream));
}

extern "C" int mx_plan_from_counts(const int64_t *counts, int64_t num_rows, int num_experts,
                                   void *workspace, void *stream) {
  clear_error();
  int rc = validate_plan_args("mx_plan_from_counts", num_rows, 1, num_experts);
  if (rc) return rc;
  if (!counts || !workspace) {
    set_error("mx_plan_from_counts: counts and workspace must be non-null");
    return MX_ERR_INVALID;
  }
  return plan_from_counts(counts, num_rows, num_experts, workspace, as_stream(stream));
}

namespace {
__global__ void plan_publish_kernel(const int32_t *err, int32_t *host_slot) {
  __hip_atomic_store(host_slot, *err, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}
}  // namespace

// One thread that stores the count through the mapped pointer: a 4-byte copy
// to the host is a copy kernel of 4 us and an event of its own to wait for.
extern "C" int mx_publish_plan_errors(const void *workspace, int32_t *host_slot, void *stream) {
  clear_error();
  if (!workspace || !host_slot) {
    set_error("mx_publish_plan_errors: workspace and host slot must be non-null");
    return MX_ERR_INVALID;
  }
  hipLaunchKernelGGL(plan_publish_kernel, dim3(1), dim3(1), 0, as_stream(stream),
                     static_cast<const int32_t *>(workspace), host_slot);
  return check_launch("mx_publish_plan_errors");
}

extern "C" const int32_t *mx_plan_error_counter(const void *workspace) {
  return static_cast<const int32_t *>(workspace);
}
