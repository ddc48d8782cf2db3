// Top-k selection of the indexer, deepseek_v41_mlx/indexer.py:140-144, and the block-level
// candidate pre-filter, indexer.py:38-64.
//
// Order: the k best scores, ties broken by the lowest position (the rule the reference leaves
// to mx.argpartition, tests/test_parity.py:17-21), -0.0 equal to +0.0. Output positions are
// ascending, mapped to idx + offset when idx < lens and -1 otherwise.
//
// Many rows (a prompt chunk): topk_stripe_kernel, a workgroup sized to the row's length. Few rows
// (decode): one 1024-thread workgroup per score row. Rows of up to 32K scores (topk_reg_kernel) keep
// their keys in registers, J consecutive positions per thread, as order-preserving 32-bit keys;
// an MSD radix select over digits of 11, 11 and 10 bits finds the k-th best key T and how many
// T-valued keys to take, then one block scan of per-thread (greater, equal) counts gives each
// thread the rank of its first selection and it writes its selections in position order -- the
// output comes out sorted and ties resolve to the lowest positions by construction. Rows over
// 16K scores with k <= 2048 can go in two stages through a workspace (per-chunk lists of the
// chunk's best k, then a merge); candidate blocks run the same register core over block maxima.
// Longer rows fall back to topk_kernel (4-pass, 8-bit digits, keys re-read from memory).
#include "select.h"

namespace dsv41 {

struct SelShared {
  uint32_t hist[kSelWaves][256];
  uint32_t tot[256];
  uint32_t wsum[kSelWaves];
  uint32_t pick[2];
};

// Finds the k-th largest key among key(0..count) (1 <= k <= count). Returns T and sets
// *need = number of T-valued keys to take after all keys > T. All threads must call it.
template <typename KeyFn>
__device__ uint32_t radix_select(SelShared& sh, KeyFn key, int count, int k, int* need) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  uint32_t prefix = 0u, pmask = 0u;
  int kk = k;
  for (int pass = 0; pass < 4; ++pass) {
    const int shift = 24 - 8 * pass;
    for (int i = tid; i < kSelWaves * 256; i += kSelThreads) (&sh.hist[0][0])[i] = 0u;
    if (tid == 0) sh.pick[0] = sh.pick[1] = 0u;
    __syncthreads();
    for (int i = tid; i < count; i += kSelThreads) {
      const uint32_t kv = key(i);
      if ((kv & pmask) == prefix) atomicAdd(&sh.hist[wave][(kv >> shift) & 255u], 1u);
    }
    __syncthreads();
    if (tid < 256) {
      uint32_t c = 0u;
#pragma unroll
      for (int w = 0; w < kSelWaves; ++w) c += sh.hist[w][tid];
      sh.tot[tid] = c;
    }
    __syncthreads();
    uint32_t incl = 0u, mine = 0u;
    if (tid < 256) {
      // suffix sums over digits: thread t handles digit 255 - t
      mine = sh.tot[255 - tid];
      incl = wave_incl_scan(mine, lane);
      if (lane == 63) sh.wsum[wave] = incl;
    }
    __syncthreads();
    if (tid < 256) {
      for (int w = 0; w < wave; ++w) incl += sh.wsum[w];
      const uint32_t above = incl - mine;               // keys whose digit is > d
      if (above < (uint32_t)kk && (uint32_t)kk <= incl) {
        sh.pick[0] = 255u - (uint32_t)tid;
        sh.pick[1] = above;
      }
    }
    __syncthreads();
    prefix |= sh.pick[0] << shift;
    pmask |= 255u << shift;
    kk -= (int)sh.pick[1];
    __syncthreads();
  }
  *need = kk;
  return prefix;
}

// Ordered compaction: calls emit(i, rank) for each selected i in increasing i, where rank is
// its position among the selected. Selection: key > T, or key == T among the first `need`.
template <typename KeyFn, typename EmitFn>
__device__ void ordered_select(SelShared& sh, KeyFn key, int count, uint32_t T, int need, EmitFn emit) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  uint32_t gt_base = 0u, eq_base = 0u;
  for (int c0 = 0; c0 < count; c0 += kSelThreads) {
    const int i = c0 + tid;
    const uint32_t kv = i < count ? key(i) : 0u;
    const uint32_t gt = (i < count && kv > T) ? 1u : 0u;
    const uint32_t eq = (i < count && kv == T) ? 1u : 0u;
    const uint32_t packed = (gt << 16) | eq;
    const uint32_t incl = wave_incl_scan(packed, lane);
    if (lane == 63) sh.wsum[wave] = incl;
    __syncthreads();
    uint32_t wbase = 0u, total = 0u;
#pragma unroll
    for (int w = 0; w < kSelWaves; ++w) {
      const uint32_t ws = sh.wsum[w];
      if (w < wave) wbase += ws;
      total += ws;
    }
    const uint32_t excl = wbase + incl - packed;
    const uint32_t gt_before = gt_base + (excl >> 16);
    const uint32_t eq_before = eq_base + (excl & 0xFFFFu);
    if (gt || (eq && eq_before < (uint32_t)need))
      emit(i, (int)(gt_before + min(eq_before, (uint32_t)need)));
    gt_base += total >> 16;
    eq_base += total & 0xFFFFu;
    __syncthreads();
  }
}

// Rows of up to J*1024 scores: thread t holds the J consecutive positions t*J .. t*J+J-1 in
// registers (float4 loads), so the radix passes and the compaction touch memory only for
// histograms and the output. Digits are 11, 11 and 10 bits wide: an 11-bit leading digit (sign,
// exponent, two mantissa bits) spreads realistic score rows over enough bins that plain LDS
// atomics stay cheap, and the later passes count only keys sharing the chosen prefix.
// Histograms alternate between two buffers, so clearing the next one needs no extra barrier.
// Compaction: one block scan of the packed per-thread (greater, equal) counts gives every thread
// the number of selected positions before its own; it then walks its keys in position order.
// J keys of entries i0 .. i0+J-1 of a score row as order keys (float4 loads when `vec`: the row
// 16-byte aligned and i0 a multiple of 4), valid for j < nvalid.
template <int J>
__device__ __forceinline__ void load_keys(const float* x, int i0, int nvalid, int vec, uint32_t (&key)[J]) {
  static_assert(J % 4 == 0, "keys are loaded as float4");
  if (vec) {
#pragma unroll
    for (int q = 0; q < J / 4; ++q) {
      float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
      if (4 * q < nvalid) v = *reinterpret_cast<const float4*>(x + i0 + 4 * q);
      key[4 * q + 0] = order_key(v.x);
      key[4 * q + 1] = order_key(v.y);
      key[4 * q + 2] = order_key(v.z);
      key[4 * q + 3] = order_key(v.w);
    }
  } else {
#pragma unroll
    for (int j = 0; j < J; ++j) key[j] = j < nvalid ? order_key(x[i0 + j]) : 0u;
  }
}

template <int J>
__global__ __launch_bounds__(kSelThreads) void topk_reg_kernel(const float* __restrict__ scores,
                                                               int32_t* __restrict__ out, int n, int nb, int k,
                                                               int start_pos, int ratio, int offset, int vec) {
  __shared__ RegSelShared sh;
  const int64_t row = blockIdx.x;
  const float* x = scores + row * nb;
  int32_t* o = out + row * k;
  const int s = (int)(row % n);
  const int lens = (start_pos + s + 1) / ratio;
  const int i0 = threadIdx.x * J;
  const int nvalid = min(max(nb - i0, 0), J);   // keys j < nvalid are real positions
  if (k >= nb) {                                 // everything is selected, in order
    for (int j = 0; j < nvalid; ++j) o[i0 + j] = i0 + j < lens ? i0 + j + offset : -1;
    return;
  }
  uint32_t key[J];
  load_keys<J>(x, i0, nvalid, vec, key);
  select_top<J>(key, nvalid, k, sh, [&](uint32_t rank, int j) {
    const int i = i0 + j;
    o[rank] = i < lens ? i + offset : -1;
  });
}

// Long rows in two stages (the workspace form). Stage 1: each kTopkChunk-entry chunk of a row
// selects its own best min(k, chunk) entries under the same order and writes them, in position
// order, as (order key, position) at cand[row][chunk][rank] -- every entry of the row's best k
// is among its chunk's best k, so the chunk lists hold the answer. Stage 2 selects the row's k
// best from the concatenated lists (still in position order, so ties still resolve to the lowest
// positions), one workgroup per row, keys in registers. Stage 1 spreads a row over
// ceil(nb / chunk) workgroups instead of one; chunks are kTopkChunk entries, or twice that where
// k is above an eighth of kTopkChunk (the lists then stay at 4,096 entries per 32K-score row).
constexpr int kTopkChunk = 4096;

template <int J>   // chunk = J * kSelThreads entries
__global__ __launch_bounds__(kSelThreads) void topk_chunk_kernel(const float* __restrict__ scores,
                                                                 uint32_t* __restrict__ ckey,
                                                                 int32_t* __restrict__ cpos, int nb, int k,
                                                                 int chunks, int vec) {
  constexpr int CH = J * kSelThreads;
  __shared__ RegSelShared sh;
  const int64_t row = blockIdx.x / chunks;
  const int ch = (int)(blockIdx.x - row * chunks);
  const int base = ch * CH;
  const int count = min(CH, nb - base);
  const int kc = min(k, count);
  const float* x = scores + row * nb + base;
  const int64_t cbase = (row * chunks + ch) * (int64_t)k;
  const int i0 = threadIdx.x * J;
  const int nvalid = min(max(count - i0, 0), J);
  uint32_t key[J];
  load_keys<J>(x, i0, nvalid, vec, key);
  select_top<J>(key, nvalid, kc, sh, [&](uint32_t rank, int j) {
    ckey[cbase + rank] = order_key(x[i0 + j]);     // re-read: j is a run-time index
    cpos[cbase + rank] = base + i0 + j;
  });
}

template <int J>
__global__ __launch_bounds__(kSelThreads) void topk_merge_kernel(const uint32_t* __restrict__ ckey,
                                                                  const int32_t* __restrict__ cpos,
                                                                  int32_t* __restrict__ out, int n, int nb, int k,
                                                                  int chunks, int chunk, int start_pos, int ratio,
                                                                  int offset) {
  __shared__ RegSelShared sh;
  const int64_t row = blockIdx.x;
  // the lists of chunks 0..chunks-2 are full (k entries: chunk >= k), the last one holds
  // min(k, its count): the valid entries are the first m of the row's concatenation
  const int m = (chunks - 1) * k + min(k, nb - (chunks - 1) * chunk);
  const uint32_t* kr = ckey + row * (int64_t)chunks * k;
  const int32_t* pr = cpos + row * (int64_t)chunks * k;
  int32_t* o = out + row * k;
  const int s = (int)(row % n);
  const int lens = (start_pos + s + 1) / ratio;
  const int i0 = threadIdx.x * J;
  const int nvalid = min(max(m - i0, 0), J);
  // keys and positions are loaded together: the selection's output step then reads no memory
  uint32_t key[J];
  int32_t pos[J];
#pragma unroll
  for (int j = 0; j < J; ++j) {
    key[j] = j < nvalid ? kr[i0 + j] : 0u;
    pos[j] = j < nvalid ? pr[i0 + j] : 0;
  }
  select_top<J>(key, nvalid, k, sh, [&](uint32_t rank, int j) {
    int32_t i = 0;
#pragma unroll
    for (int t = 0; t < J; ++t) i = t == j ? pos[t] : i;   // j is a run-time index
    o[rank] = i < lens ? i + offset : -1;
  });
}

// Many rows (a prompt chunk's queries): one workgroup of NT threads per row, wave w holding the
// contiguous positions 64 J w .. + 64 J - 1 of the row in registers, 64 at a time (entry j of lane l:
// 64 (J w + j) + l). Against topk_reg_kernel's J consecutive positions per thread, the loads and the
// output are contiguous over the lanes, ranks come from ballots (two instructions per 64 entries
// instead of a loop over each thread's own), and a barrier holds 4 or 8 waves instead of 16 while the
// CU's other rows go on. Bound by issue: the per-entry code is straight-line vector code -- an entry
// that a pass does not count adds to a dummy word of its lane's bank instead of being branched
// around, and the scalar unit, which the CU's waves share, is left to the output step (with exec
// masks and uniform branches per entry the same kernel took 267 us at 8,192 rows x 10,240, 408 us at
// 8,192 x 16,384; topk_reg_kernel 238 and 271 us; this one 84.5 and 128.5 us, 4.8 and 4.3 TB/s of
// scores and positions).
//
// Entries past the row's end have key 0, below every real key but the all-ones NaN's, whose
// entries all precede them: they are never taken (k < nb: there are enough real entries).
//
// The first histogram leaves -inf out. Masked and not yet visible entries are most of many rows, and
// their additions to one bin went one lane at a time; where the k-th best is itself -inf (a query that
// sees fewer than k entries) the row is done after that histogram. 2,048 masked rows x 32,768, half of
// each -inf: 172 -> 86 us; a causal 8,192 x 10,240 chunk's top-2,048 104.5 -> 88 us.
template <int NT>
struct StripeShared {
  uint32_t hist[2][2048 + 64];   // the last 64 words: what a pass does not count
  uint32_t wsum[NT / 64];
  uint32_t pick[3];
};

constexpr uint32_t kNegInfKey = 0x007FFFFFu, kInfKey = 0xFF800000u;   // order_key of -INFINITY, INFINITY

// kStripeLists: stage 1 of the two-stage selection (below) over `chunks` chunks of `chunk` entries per
// row: workgroup (row, chunk) writes its chunk's best min(k, count) as (order key, position).
// kStripeBlocks: select_candidate_blocks (candidate_kernel's result) at 8 scores per block: entries are
// the blocks, an entry's key that of its maximum (+inf for the row's pinned last visible block), and
// the output the keep bytes of all the row's scores.
constexpr int kStripeRows = 0, kStripeLists = 1, kStripeBlocks = 2;

// Four scores, four keep words: rows start anywhere (nb odd), so their pieces are only as aligned as
// their elements, which global loads and stores allow.
typedef float f32x4_row __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x2_row __attribute__((ext_vector_type(2), aligned(1)));

// The largest of block blk's scores in a row x of nb, 8 scores per block; NaNs are passed over. A block
// of nothing but NaN gives NaN (nan_blocks) or -inf.
__device__ __forceinline__ float block8_max(const float* x, int blk, int nb, bool nan_blocks) {
  float m = -INFINITY;
  if (blk * 8 + 8 <= nb) {
    const f32x4_row u = *reinterpret_cast<const f32x4_row*>(x + blk * 8);
    const f32x4_row v = *reinterpret_cast<const f32x4_row*>(x + blk * 8 + 4);
    m = fmaxf(fmaxf(fmaxf(u[0], u[1]), fmaxf(u[2], u[3])), fmaxf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3])));
    return nan_blocks ? m : fmaxf(m, -INFINITY);
  }
  for (int t = blk * 8; t < nb; ++t) m = fmaxf(m, x[t]);
  return m;
}

// Block blk's keep bytes.
__device__ __forceinline__ void block8_keep(uint8_t* kr, int blk, int nb, bool keep) {
  if (blk * 8 + 8 <= nb) {
    const uint32_t w = keep ? 0x01010101u : 0u;
    *reinterpret_cast<u32x2_row*>(kr + blk * 8) = u32x2_row{w, w};
    return;
  }
  for (int t = blk * 8; t < nb; ++t) kr[t] = keep ? 1 : 0;
}

template <int NT, int J, int MODE>
__global__ __launch_bounds__(NT, 8) void topk_stripe_kernel(
    const float* __restrict__ scores, int32_t* __restrict__ out, int n, int row_len, int k_max, int start_pos,
    int ratio, int offset, int chunks, int chunk, uint32_t* __restrict__ ckey, int32_t* __restrict__ cpos,
    uint8_t* __restrict__ keep, const int32_t* __restrict__ lens_v, int nan_blocks) {
  constexpr bool LISTS = MODE == kStripeLists, BLOCKS = MODE == kStripeBlocks;
  constexpr int NBIN = 2048, NW = NT / 64, BPT = NBIN / NT;
  static_assert(BPT % 2 == 0, "a thread's bins are read 8 bytes at a time");
  __shared__ __align__(16) StripeShared<NT> sh;
  const uint32_t row = LISTS ? blockIdx.x / (unsigned)chunks : blockIdx.x;
  const int ch = LISTS ? (int)(blockIdx.x - row * (unsigned)chunks) : 0;
  const int nb = LISTS ? min(chunk, row_len - ch * chunk)              // entries of this selection
                       : (BLOCKS ? (row_len + 7) / 8 : row_len);
  const int k = LISTS ? min(k_max, nb) : k_max;
  const char* x = reinterpret_cast<const char*>(scores + (int64_t)row * row_len + ch * chunk);
  char* o = reinterpret_cast<char*>(out + (int64_t)row * k);
  const int64_t list = (int64_t)blockIdx.x * k_max;   // this chunk's list (LISTS)
  const int s = (int)(row % (unsigned)n);   // 32 bits: the 64-bit division is a long scalar routine
  const int lens = BLOCKS && lens_v ? lens_v[s] : (start_pos + s + 1) / ratio;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if constexpr (LISTS) {
    if (k == nb) {                                 // a last chunk of at most k entries goes whole (uniform)
      for (int t = tid; t < nb; t += NT) {
        ckey[list + t] = order_key(reinterpret_cast<const float*>(x)[t]);
        cpos[list + t] = ch * chunk + t;
      }
      return;
    }
  }
  const int last = BLOCKS && lens > 0 ? (lens - 1) / 8 : -1;
  const int pinned = last < nb ? last : -1;        // past the row's blocks: none, and no place taken
  int p0 = wave * (64 * J) + lane;                 // this lane's first position
  // The positions p0 + 64 j are formed again where they are used: kept, they would take J registers.
  auto forget = [&]() { asm volatile("" : "+v"(p0)); };
  uint32_t key[J];
#pragma unroll
  for (int j = 0; j < J; ++j) {
    if constexpr (BLOCKS)
      key[j] = __float_as_uint(block8_max(reinterpret_cast<const float*>(x), min(p0 + 64 * j, nb - 1), row_len,
                                           nan_blocks != 0));
    else
      key[j] = __float_as_uint(*reinterpret_cast<const float*>(x + (uint32_t)min(p0 + 64 * j, nb - 1) * 4u));
    if (j % 4 == 3) __builtin_amdgcn_sched_barrier(0);     // no more than 4 entries' temporaries at once
  }
  auto clear = [&](int b) {
    uint2* h = reinterpret_cast<uint2*>(sh.hist[b]);
#pragma unroll
    for (int i = 0; i < NBIN / 2 / NT; ++i) h[tid + i * NT] = make_uint2(0u, 0u);
  };
  clear(0);
  clear(1);
  forget();
#pragma unroll
  for (int j = 0; j < J; ++j) {
    key[j] = p0 + 64 * j < nb ? order_key(__uint_as_float(key[j])) : 0u;
    if constexpr (BLOCKS)                          // the pinned block
      if (p0 + 64 * j == pinned) key[j] = kInfKey;
    if (j % 4 == 3) __builtin_amdgcn_sched_barrier(0);
  }
  __syncthreads();

  uint32_t prefix = 0u;                            // resolved top bits of the k-th best key, in place
  int need = k;                                    // entries still to take from the prefix's bin
  bool whole = false;                              // the bin holds exactly `need` entries
  const uint32_t dummy = NBIN + lane;
  uint32_t c[BPT], tot, incl;
  // suffix scan from the highest digit down: thread t owns the BPT digits below 2048 - BPT * t
  auto scan = [&](const uint32_t* h) {
    const uint2* hv = reinterpret_cast<const uint2*>(h + NBIN - BPT * (tid + 1));
#pragma unroll
    for (int i = 0; i < BPT / 2; ++i) {
      const uint2 v = hv[BPT / 2 - 1 - i];
      c[2 * i] = v.y; c[2 * i + 1] = v.x;
    }
    tot = 0u;
#pragma unroll
    for (int b = 0; b < BPT; ++b) tot += c[b];
    incl = wave_incl_scan(tot, lane);
    if (lane == 63) sh.wsum[wave] = incl;
    __syncthreads();
  };
  auto wave_total = [&]() {
    uint32_t t = 0u;
#pragma unroll
    for (int w = 0; w < NW; ++w) t += sh.wsum[w];
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)t);
  };
#pragma unroll
  for (int pass = 0; pass < 3; ++pass) {
    const int shift = pass == 0 ? 21 : (pass == 1 ? 10 : 0);
    uint32_t* h = sh.hist[pass & 1];
    forget();
#pragma unroll
    for (int j = 0; j < J; ++j) {
      uint32_t bin;
      bool counts;
      if (pass == 0) {
        // -inf (masked or not yet visible entries, often most of a row) stays out: one bin would
        // take its additions one lane at a time. So do the keys below it (NaNs with the sign set)
        // and the entries past the end, key 0.
        bin = key[j] >> 21;
        counts = key[j] > kNegInfKey;
      } else if (pass == 1) {
        bin = (key[j] >> 10) & 2047u;
        counts = (key[j] ^ prefix) < (1u << 21);
      } else {
        bin = key[j] & 1023u;
        counts = (key[j] ^ prefix) < (1u << 10);
      }
      atomicAdd(&h[counts ? bin : dummy], 1u);
      if (j % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();                               // histogram complete
    if (pass == 1) clear(0);                       // for pass 2; its readers have passed a barrier
    scan(h);
    if (pass == 0) {
      const uint32_t above_inf = wave_total();
      if (above_inf < (uint32_t)need) {            // uniform: all of those are taken, the rest from -inf down
        uint32_t inf = 0u, low = kNegInfKey;       // low, sh21 opaque: nothing per entry is kept from above
        int sh21 = 21;
        asm volatile("" : "+s"(low), "+s"(sh21));
#pragma unroll
        for (int j = 0; j < J; ++j) inf += key[j] == low ? 1u : 0u;
        inf = wave_incl_scan(inf, lane);
        __syncthreads();                           // wsum read
        if (lane == 63) sh.wsum[wave] = inf;
        __syncthreads();
        if (wave_total() >= (uint32_t)need - above_inf) {   // the k-th best is -inf itself
          prefix = low;
          need -= (int)above_inf;
          __syncthreads();                         // wsum read
          break;
        }
        // the k-th best is a NaN below -inf: count every entry of the row
        __syncthreads();
        clear(0);
        __syncthreads();
        forget();
#pragma unroll
        for (int j = 0; j < J; ++j) {
          atomicAdd(&h[p0 + 64 * j < nb ? key[j] >> sh21 : dummy], 1u);
          if (j % 4 == 3) __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();
        scan(h);
      }
    }
    uint32_t above = incl - tot;
#pragma unroll
    for (int w = 0; w < NW; ++w) above += w < wave ? sh.wsum[w] : 0u;
    if (above < (uint32_t)need && (uint32_t)need <= above + tot) {   // one thread: its bins hold the k-th best
#pragma unroll
      for (int b = 0; b < BPT; ++b) {
        if (above < (uint32_t)need && (uint32_t)need <= above + c[b]) {
          sh.pick[0] = (uint32_t)(NBIN - 1 - BPT * tid - b);
          sh.pick[1] = above;
          sh.pick[2] = above + c[b] == (uint32_t)need ? 1u : 0u;
        }
        above += c[b];
      }
    }
    __syncthreads();
    prefix |= (uint32_t)__builtin_amdgcn_readfirstlane((int)sh.pick[0]) << shift;
    need -= __builtin_amdgcn_readfirstlane((int)sh.pick[1]);
    whole = __builtin_amdgcn_readfirstlane((int)sh.pick[2]) != 0;
    if (whole) break;                              // uniform; pick is written again only past two barriers
  }

  // whole: every key >= prefix is taken. Else all three digits are resolved: keys above, and the
  // first `need` entries of those equal.
  const uint32_t T = prefix;
  forget();
  auto emit = [&](uint64_t m, bool take, uint32_t base, int j) {
    const uint32_t rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, base));
    const int p = p0 + 64 * j;
    if constexpr (BLOCKS) {                        // a block of nothing but -inf or NaN is never kept
      if (p < nb)
        block8_keep(keep + (int64_t)row * row_len, p, row_len, take && key[j] > kNegInfKey && key[j] <= kInfKey);
    } else if constexpr (LISTS) {
      if (take) {
        *reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(ckey + list) + (rank << 2)) = key[j];
        *reinterpret_cast<int32_t*>(reinterpret_cast<char*>(cpos + list) + (rank << 2)) = ch * chunk + p;
      }
    } else {
      if (take) *reinterpret_cast<int32_t*>(o + (rank << 2)) = p < lens ? p + offset : -1;
    }
  };
  auto waves_before = [&](uint32_t mine) {         // the sum of `mine` (per lane) over the waves before this one
    const uint32_t incl = wave_incl_scan(mine, lane);
    if (lane == 63) sh.wsum[wave] = incl;          // last read before the final pass barrier
    __syncthreads();
    uint32_t before = 0u;
#pragma unroll
    for (int w = 0; w < NW; ++w) before += w < wave ? sh.wsum[w] : 0u;
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)before);
  };
  if (whole) {
    uint32_t cnt = 0u;
#pragma unroll
    for (int j = 0; j < J; ++j) cnt += key[j] >= T ? 1u : 0u;
    uint32_t base = waves_before(cnt);
    uint32_t T2 = T;                               // opaque: the compiler would keep J comparison masks from above
    asm volatile("" : "+s"(T2));
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const bool take = key[j] >= T2;
      const uint64_t m = __ballot(take);
      emit(m, take, base, j);
      base += (uint32_t)__popcll(m);
      if (j % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
  } else {
    uint32_t cnt = 0u;                             // above T << 16 | equal (at most 32,768 of either)
#pragma unroll
    for (int j = 0; j < J; ++j) cnt += (key[j] > T ? 0x10000u : 0u) + (key[j] == T ? 1u : 0u);
    const uint32_t before = waves_before(cnt);
    uint32_t eq = before & 0xFFFFu, base = (before >> 16) + min(eq, (uint32_t)need);
    uint32_t T2 = T;                               // opaque, as above
    asm volatile("" : "+s"(T2));
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const uint64_t e = __ballot(key[j] == T2);
      const uint32_t er = __builtin_amdgcn_mbcnt_hi((uint32_t)(e >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)e, eq));
      const bool take = key[j] > T2 || (key[j] == T2 && er < (uint32_t)need);
      const uint64_t m = __ballot(take);
      emit(m, take, base, j);
      base += (uint32_t)__popcll(m);
      eq += (uint32_t)__popcll(e);
      if (j % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// Rows longer than 32k scores: keys are re-read from memory in every pass.
__global__ __launch_bounds__(kSelThreads) void topk_kernel(const float* __restrict__ scores, int32_t* __restrict__ out,
                                                           int n, int nb, int k, int start_pos, int ratio,
                                                           int offset) {
  __shared__ SelShared sh;
  const int64_t row = blockIdx.x;
  const float* x = scores + row * nb;
  int32_t* o = out + row * k;
  const int s = (int)(row % n);
  const int lens = (start_pos + s + 1) / ratio;
  auto key = [&](int i) { return order_key(x[i]); };
  auto emit = [&](int i, int rank) {
    if (rank < k) o[rank] = i < lens ? i + offset : -1;
  };
  if (k >= nb) {  // everything is selected (k == nb)
    for (int i = threadIdx.x; i < nb; i += kSelThreads) emit(i, i);
    return;
  }
  int need = 0;
  const uint32_t T = radix_select(sh, key, nb, k, &need);
  ordered_select(sh, key, nb, T, need, emit);
}

constexpr int kMaxCandBlocks = 8192;
// Rows from which candidate blocks of 8 scores run on topk_stripe_kernel, us candidate_kernel -> stripe.
// 32,768 scores, 2,048 blocks kept: 64 rows 11.2 -> 10.3, 384 rows 21.8 -> 15.9, 2,048 rows 99.0 -> 63.6;
// 1,400 x 22,804 417 us with byte stores and scalar reads of the rows that are not 16-byte pieces, 52 us with
// element-aligned ones, 33.6 us on the stripe kernel. Up to 1,024 blocks the register kernel's one short
// pass wins until the rows fill the chip more than once (4,096 scores, 64 blocks kept: 64 rows 5.9 -> 6.4,
// 256 rows 6.6 -> 7.1, 384 rows 8.1 -> 7.3, 512 rows 8.7 -> 7.5).
static int64_t cand_stripe_from(int nblk) { return nblk > kSelThreads ? 64 : 384; }

// select_candidate_blocks on the register core: thread t holds the maxima of blocks t*J ..
// t*J+J-1 as order keys (the pinned block (lens-1)/bs as +inf); the best min(topk_blocks, nblk)
// blocks (ties -> lowest block) are marked, and a marked block is kept when its maximum is
// > -inf. Each thread then writes the keep bytes of its own blocks.
template <int J>
__global__ __launch_bounds__(kSelThreads) void candidate_kernel(const float* __restrict__ scores,
                                                                uint8_t* __restrict__ keep, int n, int nb,
                                                                int topk_blocks, int bs, const int32_t* lens_v,
                                                                int start_pos, int ratio, int nan_blocks) {
  __shared__ RegSelShared sh;
  __shared__ uint8_t marked[kMaxCandBlocks];
  const int64_t row = blockIdx.x;
  const float* x = scores + row * nb;
  const int s = (int)(row % n);
  const int lens = lens_v ? lens_v[s] : (start_pos + s + 1) / ratio;
  const int nblk = (nb + bs - 1) / bs;
  const int last = lens > 0 ? (lens - 1) / bs : -1;  // floor((lens - 1) / bs)
  const int j0 = threadIdx.x * J;
  const int nvalid = min(max(nblk - j0, 0), J);
  float bm[J];
  uint32_t key[J];
#pragma unroll
  for (int j = 0; j < J; ++j) {
    float m = -INFINITY;
    const int blk = j0 + j;
    if (j < nvalid) {
      if (bs == 8) {
        m = block8_max(x, blk, nb, nan_blocks != 0);
      } else {
        const int e = min(nb, (blk + 1) * bs);
        for (int t = blk * bs; t < e; ++t) m = fmaxf(m, x[t]);
      }
    }
    bm[j] = blk == last ? INFINITY : m;
    key[j] = order_key(bm[j]);
    if (j < nvalid) marked[blk] = 0;
  }
  const int kb = min(topk_blocks, nblk);
  if (kb >= nblk) {
#pragma unroll
    for (int j = 0; j < J; ++j)
      if (j < nvalid) marked[j0 + j] = 1;
  } else if (kb > 0) {
    select_top<J>(key, nvalid, kb, sh, [&](uint32_t, int j) { marked[j0 + j] = 1; });
  }
  __syncthreads();
  uint8_t* kr = keep + row * nb;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    if (j >= nvalid) continue;
    const int blk = j0 + j;
    const uint8_t v = (marked[blk] && bm[j] > -INFINITY) ? 1 : 0;
    if (bs == 8) {
      block8_keep(kr, blk, nb, v != 0);
    } else {
      const int e = min(nb, (blk + 1) * bs);
      for (int t = blk * bs; t < e; ++t) kr[t] = v;
    }
  }
}

}  // namespace dsv41

using namespace dsv41;

namespace dsv41 {
// Stage 2 of a two-stage selection over per-chunk lists of k (key, position) entries, `chunk`
// scores per chunk (>= k); also used by the indexer's fused decode form. chunks * k <= 32768.
int topk_merge_launch(const char* what, const uint32_t* ckey, const int32_t* cpos, int32_t* out, int64_t rows, int n,
                      int nb, int k, int chunks, int chunk, int start_pos, int ratio, int offset, hipStream_t stream) {
  const int64_t m = (int64_t)chunks * k;
  DSV41_REQUIRE(m <= 32 * kSelThreads && rows < (1ll << 31), DSV41_E_SHAPE, "%s: %lld candidates per row", what,
                (long long)m);
  const dim3 grid((unsigned)rows), block(kSelThreads);
#define DSV41_MERGE_CASE(J_)                                                                                  \
  if (m <= J_ * kSelThreads) {                                                                                \
    hipLaunchKernelGGL(topk_merge_kernel<J_>, grid, block, 0, stream, ckey, cpos, out, n, nb, k, chunks, chunk, \
                       start_pos, ratio, offset);                                                            \
    return check_launch(what);                                                                              \
  }
  DSV41_MERGE_CASE(4)
  DSV41_MERGE_CASE(8)
  DSV41_MERGE_CASE(16)
  DSV41_MERGE_CASE(32)
#undef DSV41_MERGE_CASE
  return set_error(DSV41_E_SHAPE, "%s: too many candidates", what);
}
}  // namespace dsv41

// How a selection over `rows` rows of nb scores runs.
struct TopkPlan {
  bool stripe;         // topk_stripe_kernel (the whole row, or stage 1)
  int chunks, chunk;   // two stages: per-chunk lists, then a merge (chunks 0: one stage)
};

constexpr int kStripeMax = 32 * kSelThreads;   // entries of the largest stripe workgroup

// Stripe workgroups win once the chip has rows enough to fill it, and earlier where a row would
// otherwise go in two stages (single calls, graph-replayed, 1,024-thread register kernel or two
// stages -> stripe):
//   4,096 scores, top-512:    256 rows 7.0 -> 7.5 us,   512 rows 9.1 -> 8.3,   8,192 rows 83.1 -> 38.2
//   10,240 scores, top-2,048: 256 rows 10.4 -> 11.5 us, 512 rows 18.0 -> 13.5, 8,192 rows 238.4 -> 84.5
//   16,384 scores, top-512:   256 rows 11.1 -> 11.7 us, 512 rows 19.7 -> 15.4, 8,192 rows 271.3 -> 128.5
//   32,768 scores, top-512:   32 rows 13.9 -> 15.4 us,  64 rows 16.2 -> 15.5,  2,048 rows 194.3 -> 79.9
// Rows over 32,768 scores go in two stages whose chunks are as few and as even as stripe workgroups
// can hold (65,536 scores, top-512: 64 rows 20.6 us either way, 128 rows 32.1 -> 21.8 us, 2,048 rows
// 386 -> 173.5 us).
//
// Fewer rows: rows longer than one 16-keys-per-thread workgroup holds go in two stages, with k at
// most half a chunk and the chunk lists small enough for one register workgroup.
// For 16 rows of 32,768 scores and k = 1,024 one 32-keys-per-thread workgroup per row is faster
// on scores already in cache (17.5-19.3 against 19.4-20.2 us), but inside a decode step, reading
// the scores the scoring kernel has just written, the two stages spread that read over 8
// workgroups per row and win: the 40-layer fp8 step took 1.163-1.166 ms against 1.190-1.195 ms.
//
// Rows over 24,576 scores whose two stages have short lists (k up to 1,024) win for a few rows more: 64 rows
// of 32,768 scores, two stages -> stripe, top-128 13.1 -> 14.8 us, top-512 15.5 -> 15.6, top-2,048 23.0 ->
// 16.0; 72 rows of 28,000, top-128 13.1 -> 14.8; 80 rows of 32,768, top-128 15.8 -> 14.8.
static int64_t stripe_from(int nb, int k) {
  if (nb <= 16 * kSelThreads) return 512;
  if (nb <= kStripeMax) return nb <= 24 * kSelThreads || k > 1024 ? 64 : 80;
  return 128;
}

static TopkPlan topk_plan(int64_t rows, int nb, int k, bool allow_two_stage) {
  TopkPlan p{false, 0, 0};
  if (k >= nb) return p;                           // everything is selected
  const bool many = rows >= stripe_from(nb, k);
  if (nb <= kStripeMax) {
    p.stripe = many;
    if (p.stripe) return p;
  }
  if (!allow_two_stage || nb <= 16 * kSelThreads) return p;
  if (nb > kStripeMax && many) {
    const int c = (nb + kStripeMax - 1) / kStripeMax;
    const int ch = ((nb + c - 1) / c + 63) / 64 * 64;
    if (k <= ch && (int64_t)c * k <= 32 * kSelThreads && (int64_t)(c - 1) * ch < nb && rows * c < (1ll << 31)) {
      p.stripe = true;
      p.chunks = c;
      p.chunk = ch;
      return p;
    }
  }
  if (2 * k > kTopkChunk) return p;
  // lists of more than 4,096 entries per row with 4,096-entry chunks: 8,192-entry chunks halve them
  const int ch = (int64_t)((nb + kTopkChunk - 1) / kTopkChunk) * k > 4 * kSelThreads ? 2 * kTopkChunk : kTopkChunk;
  const int c = (nb + ch - 1) / ch;
  if ((int64_t)c * k > 32 * kSelThreads) return p;
  p.chunks = c;
  p.chunk = ch;
  return p;
}

// Launches topk_stripe_kernel for selections of at most `len` entries on a grid of one workgroup each.
template <int MODE>
static void launch_stripe(int len, unsigned grid, const float* scores, int32_t* out, int n, int nb, int k,
                          int start_pos, int ratio, int offset, int chunks, int chunk, uint32_t* ckey, int32_t* cpos,
                          uint8_t* keep, const int32_t* lens, int nan_blocks, hipStream_t stream) {
#define DSV41_STRIPE_CASE(NT_, J_)                                                                                  \
  if (len <= NT_ * J_) {                                                                                            \
    hipLaunchKernelGGL((topk_stripe_kernel<NT_, J_, MODE>), dim3(grid), dim3(NT_), 0, stream, scores, out, n, nb, k, \
                       start_pos, ratio, offset, chunks, chunk, ckey, cpos, keep, lens, nan_blocks);                \
    return;                                                                                                         \
  }
  if constexpr (MODE == kStripeBlocks) {           // at most kMaxCandBlocks
    DSV41_STRIPE_CASE(256, 8)
    DSV41_STRIPE_CASE(256, 16)
    DSV41_STRIPE_CASE(512, 16)
  }
  if constexpr (MODE == kStripeRows) {             // chunks are longer than half of kStripeMax
    DSV41_STRIPE_CASE(256, 8)
    DSV41_STRIPE_CASE(256, 16)
    DSV41_STRIPE_CASE(256, 24)
    DSV41_STRIPE_CASE(256, 32)
    DSV41_STRIPE_CASE(256, 40)
    DSV41_STRIPE_CASE(512, 24)
    DSV41_STRIPE_CASE(512, 32)
  }
  if constexpr (MODE != kStripeBlocks) {
    DSV41_STRIPE_CASE(512, 40)
    DSV41_STRIPE_CASE(1024, 24)
    DSV41_STRIPE_CASE(1024, 32)
  }
#undef DSV41_STRIPE_CASE
}

static size_t topk_ws_bytes(int64_t rows, int chunks, int k) {
  const size_t list = ((size_t)rows * chunks * k * sizeof(uint32_t) + 255) & ~(size_t)255;
  return 2 * list;                               // order keys, then positions
}

static int topk_launch(const char* what, const float* scores, int32_t* out, int64_t rows, int32_t n, int32_t nb,
                       int32_t topk, int32_t start_pos, int32_t ratio, int32_t offset, void* workspace,
                       size_t workspace_bytes, bool allow_two_stage, hipStream_t stream) {
  DSV41_REQUIRE(scores && out, DSV41_E_ARG, "%s: null tensor", what);
  DSV41_REQUIRE(rows >= 0 && n > 0 && nb >= 0 && topk >= 0 && start_pos >= 0 && ratio > 0, DSV41_E_ARG,
                "%s: bad sizes", what);
  DSV41_REQUIRE(nb <= (1 << 22), DSV41_E_SHAPE, "%s: nb %d > 2^22", what, nb);
  DSV41_REQUIRE(rows < (1ll << 31), DSV41_E_ARG, "%s: too many rows", what);
  const int k = topk < nb ? topk : nb;
  if (rows == 0 || k == 0) return 0;
  const dim3 grid((unsigned)rows), block(kSelThreads);
  const int vec = (nb % 4 == 0 && aligned16(scores)) ? 1 : 0;
  TopkPlan plan = topk_plan(rows, nb, k, allow_two_stage);
  // Many rows in two stages where few take one (k over half a chunk): a caller without the workspace still
  // gets the one stage.
  if (plan.chunks && !topk_plan(1, nb, k, true).chunks &&
      !(workspace && aligned16(workspace) && workspace_bytes >= topk_ws_bytes(rows, plan.chunks, k)))
    plan = TopkPlan{false, 0, 0};
  if (plan.chunks) {
    const int chunks = plan.chunks, chunk = plan.chunk;
    const size_t need = topk_ws_bytes(rows, chunks, k);
    DSV41_REQUIRE(workspace && workspace_bytes >= need, DSV41_E_WORKSPACE, "%s: workspace of %zu bytes needed", what,
                  need);
    DSV41_REQUIRE(aligned16(workspace), DSV41_E_ARG, "%s: workspace must be 16-byte aligned", what);
    DSV41_REQUIRE(rows * chunks < (1ll << 31), DSV41_E_ARG, "%s: too many row chunks", what);
    uint32_t* ckey = reinterpret_cast<uint32_t*>(workspace);
    int32_t* cpos = reinterpret_cast<int32_t*>(reinterpret_cast<uint8_t*>(workspace) + need / 2);
    const dim3 cgrid((unsigned)(rows * chunks));
    if (plan.stripe)
      launch_stripe<kStripeLists>(chunk, cgrid.x, scores, out, n, nb, k, start_pos, ratio, offset, chunks, chunk, ckey,
                                  cpos, nullptr, nullptr, 0, stream);
    else if (chunk == kTopkChunk)
      hipLaunchKernelGGL(topk_chunk_kernel<kTopkChunk / kSelThreads>, cgrid, block, 0, stream, scores, ckey, cpos, nb, k,
                         chunks, vec);
    else
      hipLaunchKernelGGL(topk_chunk_kernel<2 * kTopkChunk / kSelThreads>, cgrid, block, 0, stream, scores, ckey, cpos,
                         nb, k, chunks, vec);
    int rc = check_launch(what);
    if (rc) return rc;
    return topk_merge_launch(what, ckey, cpos, out, rows, n, nb, k, chunks, chunk, start_pos, ratio, offset, stream);
  }
  if (plan.stripe) {
    launch_stripe<kStripeRows>(nb, grid.x, scores, out, n, nb, k, start_pos, ratio, offset, 1, nb, nullptr, nullptr,
                               nullptr, nullptr, 0, stream);
    return check_launch(what);
  }
  if (nb <= 4 * kSelThreads)
    hipLaunchKernelGGL(topk_reg_kernel<4>, grid, block, 0, stream, scores, out, n, nb, k, start_pos, ratio, offset, vec);
  else if (nb <= 8 * kSelThreads)
    hipLaunchKernelGGL(topk_reg_kernel<8>, grid, block, 0, stream, scores, out, n, nb, k, start_pos, ratio, offset, vec);
  else if (nb <= 16 * kSelThreads)
    hipLaunchKernelGGL(topk_reg_kernel<16>, grid, block, 0, stream, scores, out, n, nb, k, start_pos, ratio, offset,
                       vec);
  else if (nb <= 32 * kSelThreads)
    hipLaunchKernelGGL(topk_reg_kernel<32>, grid, block, 0, stream, scores, out, n, nb, k, start_pos, ratio, offset,
                       vec);
  else
    hipLaunchKernelGGL(topk_kernel, grid, block, 0, stream, scores, out, n, nb, k, start_pos, ratio, offset);
  return check_launch(what);
}

extern "C" int dsv41_topk_select(const float* scores, int32_t* out, int64_t rows, int32_t n, int32_t nb,
                                 int32_t topk, int32_t start_pos, int32_t ratio, int32_t offset, hipStream_t stream) {
  return topk_launch("dsv41_topk_select", scores, out, rows, n, nb, topk, start_pos, ratio, offset, nullptr, 0, false,
                     stream);
}

extern "C" size_t dsv41_topk_workspace_bytes(int64_t rows, int32_t nb, int32_t topk) {
  if (rows <= 0 || nb <= 0 || topk <= 0) return 0;
  const int k = topk < nb ? topk : nb;
  // At least what any smaller number of rows takes (few rows need more than many: from stripe_from on the
  // chunks are fewer, or none), so that a workspace sized for the largest batch serves every batch.
  auto bytes = [&](int64_t r) {
    const TopkPlan p = topk_plan(r, nb, k, true);
    return p.chunks ? topk_ws_bytes(r, p.chunks, k) : (size_t)0;
  };
  const int64_t few = stripe_from(nb, k) - 1;
  const size_t own = bytes(rows), less = rows > few ? bytes(few) : 0;
  return own > less ? own : less;
}

extern "C" int dsv41_topk_select_ws(const float* scores, int32_t* out, int64_t rows, int32_t n, int32_t nb,
                                    int32_t topk, int32_t start_pos, int32_t ratio, int32_t offset, void* workspace,
                                    size_t workspace_bytes, hipStream_t stream) {
  return topk_launch("dsv41_topk_select_ws", scores, out, rows, n, nb, topk, start_pos, ratio, offset, workspace,
                     workspace_bytes, true, stream);
}

extern "C" int dsv41_candidate_blocks(const float* scores, uint8_t* keep, int64_t rows, int32_t n, int32_t nb,
                                      int32_t topk_blocks, int32_t block_size, const int32_t* lens,
                                      int32_t start_pos, int32_t ratio, hipStream_t stream) {
  const char* what = "dsv41_candidate_blocks";
  DSV41_REQUIRE(scores && keep, DSV41_E_ARG, "%s: null tensor", what);
  DSV41_REQUIRE(rows >= 0 && n > 0 && nb >= 0 && topk_blocks >= 0 && block_size > 0 && start_pos >= 0 && ratio > 0,
                DSV41_E_ARG, "%s: bad sizes", what);
  DSV41_REQUIRE((nb + block_size - 1) / block_size <= kMaxCandBlocks, DSV41_E_SHAPE, "%s: more than %d blocks",
                what, kMaxCandBlocks);
  DSV41_REQUIRE(rows < (1ll << 31), DSV41_E_ARG, "%s: too many rows", what);
  if (rows == 0 || nb == 0) return 0;
  const int nblk = (nb + block_size - 1) / block_size;
  // a whole block of NaNs counts as NaN where the rows are 16-byte pieces, else as -inf
  const int nan_blocks = nb % 8 == 0 && aligned16(scores) && (reinterpret_cast<uintptr_t>(keep) & 7u) == 0 ? 1 : 0;
  if (block_size == 8 && rows >= cand_stripe_from(nblk) && topk_blocks > 0 && topk_blocks < nblk) {
    launch_stripe<kStripeBlocks>(nblk, (unsigned)rows, scores, nullptr, n, nb, topk_blocks, start_pos, ratio, 0, 1, nb,
                                 nullptr, nullptr, keep, lens, nan_blocks, stream);
    return check_launch(what);
  }
  if (nblk <= 4 * kSelThreads)
    hipLaunchKernelGGL(candidate_kernel<4>, dim3((unsigned)rows), dim3(kSelThreads), 0, stream, scores, keep, n, nb,
                       topk_blocks, block_size, lens, start_pos, ratio, nan_blocks);
  else
    hipLaunchKernelGGL(candidate_kernel<8>, dim3((unsigned)rows), dim3(kSelThreads), 0, stream, scores, keep, n, nb,
                       topk_blocks, block_size, lens, start_pos, ratio, nan_blocks);
  return check_launch(what);
}
