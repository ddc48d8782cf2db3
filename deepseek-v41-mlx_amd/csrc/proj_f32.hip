// The compressor's two projections, deepseek_v41_mlx/compressor.py:59-61: kv = x wkv^T and
// score = x wgate^T with float32 weights, in float32, for bf16 activations x.
//
//   y0[m, j] = sum_k x[m, k] * w0[j, k],  y1[m, j] = sum_k x[m, k] * w1[j, k]
//
// On the bf16 matrix cores without giving up any of the 24 bits of a weight: a float32 w is cut, by
// truncation, into three bf16 numbers of 8 significand bits each, w = h + m + l exactly, and the
// three products with the (already bf16) activation are exact in the MFMA, which adds them up in
// float32. Relative error (2-norm) against the float64 result, k = 5120, library float32 GEMM and this
// one: 64 rows 6.4e-7 and 2.0e-7, 1,024 rows 1.28e-6 and 5.5e-7, 8,192 rows 1.28e-6 and 7.9e-7.
//
// Bound by the matrix cores at chunk row counts (3 x 2 rows k n multiply-adds on the bf16 rate, a
// sixteenth of which is what float32 MFMAs reach) and by the weight stream (4 bytes each) at decode
// row counts. Both projections, k = 5120, n = 512 + 512, against the library (x widened to float32,
// then two float32 GEMMs), us: 8,191 rows 616 -> 216, 2,000 rows 173 -> 68, 64 rows 28.6 -> 15.5,
// 1 row 26.5 -> 13.1 (1,190 TFLOP/s of bf16 products at 8,191 rows).
//
// A workgroup owns TR weight rows (of the two weights stacked) x TM activation rows and walks 64
// channels per step, double-buffered. The activations arrive by LDS copies; the weights pass through
// registers, where each is cut once per workgroup, and lie in LDS as three bf16 planes, all in the
// XOR-swizzled rows that the fragment reads take without bank conflicts. The contraction is cut into
// `splits` ranges where the tiles alone would not fill the chip; then each range's float32 partial
// goes to the workspace and a second kernel adds them in range order.
#include "mfma.h"

namespace dsv41 {

struct ProjArgs {
  const bf16_t* x;                       // [rows, k]
  const float *w0, *w1;                  // [n0, k], [n - n0, k]
  float *y0, *y1;                        // [rows, n0], [rows, n - n0]
  float* part;                           // [splits, rows, n] partial sums (splits > 1)
  int rows, k, n, n0, splits;
};

// 16-byte chunk c of a 128-byte tile row (64 bf16) sits at slot c ^ proj_swz(row): a fragment read
// takes one chunk of 16 consecutive rows and no two of its lanes share a bank.
__device__ __forceinline__ int proj_swz(int row) { return (row & 7) ^ ((row >> 3) & 1); }

// The three bf16 planes of four weights, as packed pairs (even channel low): the upper 16 bits of
// what is left after each plane. Every difference is exact (at most 16, then 8 bits remain).
struct Planes {
  uint2 p[3];
};
__device__ __forceinline__ Planes cut_weights(const float4 w) {
  float r[4] = {w.x, w.y, w.z, w.w};
  Planes o;
#pragma unroll
  for (int s = 0; s < 3; ++s) {
    uint32_t u[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      u[i] = __float_as_uint(r[i]);
      r[i] = r[i] - __uint_as_float(u[i] & 0xFFFF0000u);
    }
    o.p[s] = make_uint2(__builtin_amdgcn_perm(u[1], u[0], 0x07060302u), __builtin_amdgcn_perm(u[3], u[2], 0x07060302u));
  }
  return o;
}

// Infinities: an infinite weight leaves NaN behind its first plane, and an infinite activation meets
// planes that are 0, so a sum that should be infinite comes out NaN. NaN sums are therefore formed again
// from what decides them alone: a weight counts as NaN, as an infinity, as 0 or as 2^-40 with its sign (so
// that no finite sum overflows). Infinite there, the result is that infinity; else it stays NaN. Per wave
// and 16 weight rows, from memory and on the matrix cores, so that rows full of NaN stay within a few times
// the finite ones' time (one output at a time by one lane, each a serial loop over k, took thousands of
// times as long).
__device__ __forceinline__ uint32_t weight_class(uint32_t w) {   // bf16 bits
  const uint32_t m = w & 0x7FFFFFFFu, s = (w >> 16) & 0x8000u;
  return m > 0x7F800000u ? 0x7FC0u : (m == 0x7F800000u ? s | 0x7F80u : (m ? s | 0x2B80u : 0u));
}
__device__ __forceinline__ void store_proj(const ProjArgs& a, int m, int j, f32x4 v) {   // columns j .. j + 3 of row m
  float* y = j >= a.n0 ? a.y1 + (int64_t)m * (a.n - a.n0) + (j - a.n0) : a.y0 + (int64_t)m * a.n0 + j;
  *reinterpret_cast<f32x4*>(y) = v;
}

// A GR x GM grid of waves, each 16 WR weight rows x 16 WM activation rows.
template <int WR, int WM, int GR, int GM>
struct ProjCfg {
  static constexpr int NWV = GR * GM, NT = 64 * NWV;
  static constexpr int TR = 16 * WR * GR, TM = 16 * WM * GM;
  static constexpr int BK = 64, RB = BK * 2;
  static constexpr int PLANE = TR * RB, STAGE = 3 * PLANE + TM * RB, LDS = 2 * STAGE;
  static constexpr int WL = TR / (4 * NWV);           // 1 KB weight loads per wave and step (4 rows of 256 bytes)
  static constexpr int XL = TM / (8 * NWV);           // 1 KB activation copies per wave and step (8 rows of 128 bytes)
  static_assert(WL * 4 * NWV == TR && XL * 8 * NWV == TM, "whole load instructions per wave");
  static_assert(LDS <= 160 * 1024, "LDS budget");
};

template <int WR, int WM, int GR, int GM>
__global__ __launch_bounds__(64 * GR * GM, (ProjCfg<WR, WM, GR, GM>::LDS <= 80 * 1024) ? 4 : 2) void proj_f32_kernel(
    ProjArgs a) {
  using C = ProjCfg<WR, WM, GR, GM>;
  __shared__ __align__(16) uint8_t lds[C::LDS];       // 2 x [h plane][m plane][l plane][activations]
  const int rtiles = a.n / C::TR;
  // consecutive tiles on one XCD, the weight tile fastest: the workgroups that read one activation
  // tile share that XCD's L2
  const int total = (int)gridDim.x;
  const int tile = total % 8 ? (int)blockIdx.x : ((int)blockIdx.x % 8) * (total / 8) + (int)blockIdx.x / 8;
  const int rt = tile % rtiles, sp = (tile / rtiles) % a.splits, mt = tile / (rtiles * a.splits);
  const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = (wave % GR) * 16 * WR, wm = (wave / GR) * 16 * WM;   // this wave's block
  const int steps = a.k / C::BK, first = sp * steps / a.splits;
  const int nk = (sp + 1) * steps / a.splits - first; // 64-channel steps of this range
  // weights: wave w loads tile rows w TR/NWV + 4 j + g, lane l16 the channels 4 l16 .. + 3 of a step
  const float* wsrc[C::WL];
  int wdst[C::WL];
#pragma unroll
  for (int j = 0; j < C::WL; ++j) {
    const int row = wave * (C::TR / C::NWV) + 4 * j + g;
    const int all = rt * C::TR + row;
    const float* base = all < a.n0 ? a.w0 + (int64_t)all * a.k : a.w1 + (int64_t)(all - a.n0) * a.k;
    wsrc[j] = base + (int64_t)first * C::BK + 4 * l16;
    wdst[j] = row * C::RB + (((l16 >> 1) ^ proj_swz(row)) << 4) + 8 * (l16 & 1);
  }
  uint64_t xsrc[C::XL];
#pragma unroll
  for (int j = 0; j < C::XL; ++j) {
    const int row = wave * (C::TM / C::NWV) + 8 * j + (lane >> 3);
    const int64_t m = min(mt * C::TM + row, a.rows - 1);              // rows past the end: not stored
    xsrc[j] = reinterpret_cast<uint64_t>(a.x + m * a.k + (int64_t)first * C::BK + 8 * ((lane & 7) ^ proj_swz(row)));
  }
  const uint32_t lds0 = lds_offset(lds);
  auto issue_x = [&](int buf, int kt) {
    const uint32_t dst = (uint32_t)__builtin_amdgcn_readfirstlane(
        (int)(lds0 + (uint32_t)(buf * C::STAGE + 3 * C::PLANE) + (uint32_t)(wave * (C::TM / C::NWV) * C::RB)));
#pragma unroll
    for (int j = 0; j < C::XL; ++j) dma16_vaddr(xsrc[j] + (uint64_t)kt * C::RB, dst + j * 1024);
  };
  float4 wreg[C::WL];
  auto load_w = [&](int kt) {
#pragma unroll
    for (int j = 0; j < C::WL; ++j) wreg[j] = *reinterpret_cast<const float4*>(wsrc[j] + kt * C::BK);
  };
  auto store_w = [&](int buf) {
#pragma unroll
    for (int j = 0; j < C::WL; ++j) {
      const Planes p = cut_weights(wreg[j]);
#pragma unroll
      for (int s = 0; s < 3; ++s) *reinterpret_cast<uint2*>(lds + buf * C::STAGE + s * C::PLANE + wdst[j]) = p.p[s];
    }
  };
  auto frag = [&](const uint8_t* t, int row, int chunk) {
    return ld_bf16x8(t + row * C::RB + ((chunk ^ proj_swz(row)) << 4));
  };

  f32x4 acc[WR][WM];
#pragma unroll
  for (int i = 0; i < WR; ++i)
#pragma unroll
    for (int j = 0; j < WM; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  issue_x(0, 0);
  load_w(0);
  store_w(0);
  for (int kt = 0; kt < nk; ++kt) {
    const int buf = kt & 1;
    wait_vmcnt<0>();                                  // this wave's activation copies of step kt
    __syncthreads();                                  // step kt is in LDS; step kt - 1's buffer is free
    const bool more = kt + 1 < nk;
    if (more) {
      issue_x(buf ^ 1, kt + 1);                       // copies first: the wait for the weights covers them
      load_w(kt + 1);
    }
    const uint8_t* wt = lds + buf * C::STAGE;
    const uint8_t* xt = wt + 3 * C::PLANE;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      bf16x8 bx[WM];
#pragma unroll
      for (int j = 0; j < WM; ++j) bx[j] = frag(xt, wm + 16 * j + l16, 4 * ks + g);
#pragma unroll
      for (int s = 2; s >= 0; --s) {                  // the smallest plane first
        bf16x8 af[WR];
#pragma unroll
        for (int i = 0; i < WR; ++i) af[i] = frag(wt + s * C::PLANE, wr + 16 * i + l16, 4 * ks + g);
#pragma unroll
        for (int i = 0; i < WR; ++i)
#pragma unroll
          for (int j = 0; j < WM; ++j) acc[i][j] = mfma16x16x32(af[i], bx[j], acc[i][j]);
      }
    }
    if (more) store_w(buf ^ 1);                       // the next step's weights, cut, while the MFMAs drain
  }

#pragma unroll
  for (int i = 0; i < WR; ++i) {
    bool nan = false;
#pragma unroll
    for (int j = 0; j < WM; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) nan = nan || acc[i][j][e] != acc[i][j][e];
    if (!__any(nan)) continue;                        // always, unless an input is infinite or NaN or a sum overflows
    const int all = rt * C::TR + wr + 16 * i + l16;
    const float* wrow = (all < a.n0 ? a.w0 + (int64_t)all * a.k : a.w1 + (int64_t)(all - a.n0) * a.k) +
                        (int64_t)first * C::BK + 8 * g;
    f32x4 dec[WM];
#pragma unroll
    for (int j = 0; j < WM; ++j) dec[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int c = 0; c < nk * C::BK; c += 32) {
      union {
        uint32_t u[4];
        bf16x8 v;
      } af;
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const uint4 w = *reinterpret_cast<const uint4*>(wrow + c + 4 * e);
        af.u[2 * e] = weight_class(w.x) | weight_class(w.y) << 16;
        af.u[2 * e + 1] = weight_class(w.z) | weight_class(w.w) << 16;
      }
#pragma unroll
      for (int j = 0; j < WM; ++j) {
        const int64_t m = min(mt * C::TM + wm + 16 * j + l16, a.rows - 1);
        dec[j] = mfma16x16x32(af.v, ld_bf16x8(a.x + m * a.k + (int64_t)first * C::BK + c + 8 * g), dec[j]);
      }
    }
#pragma unroll
    for (int j = 0; j < WM; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (acc[i][j][e] != acc[i][j][e] && fabsf(dec[j][e]) == INFINITY) acc[i][j][e] = dec[j][e];
  }

#pragma unroll
  for (int j = 0; j < WM; ++j) {
    const int m = mt * C::TM + wm + 16 * j + l16;
    if (m >= a.rows) continue;
#pragma unroll
    for (int i = 0; i < WR; ++i) {
      const int col = rt * C::TR + wr + 16 * i + 4 * g;
      if (a.splits > 1) *reinterpret_cast<f32x4*>(a.part + ((int64_t)sp * a.rows + m) * a.n + col) = acc[i][j];
      else store_proj(a, m, col, acc[i][j]);
    }
  }
}

// y[m, j] = sum over the ranges, in order, of part[s][m][j]; four outputs per thread.
__global__ __launch_bounds__(256) void proj_reduce_kernel(ProjArgs a) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  const int64_t total = (int64_t)a.rows * a.n;
  if (i >= total) return;
  f32x4 acc = *reinterpret_cast<const f32x4*>(a.part + i);
  for (int s = 1; s < a.splits; ++s) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(a.part + s * total + i);
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] += v[e];
  }
  const int m = (int)(i / a.n);
  store_proj(a, m, (int)(i - (int64_t)m * a.n), acc);
}

// The pooling of compress_pool_kernel (compress.hip: the same sums in the same order, the same state
// update) straight from the projections, for 512 channels and ratio 2 or 4: a contraction cut into
// ranges is summed here, range by range as proj_reduce_kernel does, so that kernel and its 4 bytes per
// value out and back are gone, and a group's rows are read once, all at the same time, into registers
// instead of three times one after another. Bound by the projections' bytes at chunk row counts and by
// launches and load latency at decode ones. Against the two calls (us, k = 5120): 1 token 16.0 -> 13.1,
// one of 32 sequences 19.6 -> 15.4, 300 tokens 34.8 -> 30.1, 1,000 66.0 -> 58.2, 8,191 228 -> 221.
constexpr int kChunkDim = 512;

struct ChunkArgs {
  ProjArgs p;                            // splits > 1: the rows lie as parts, else in y0 and y1
  float *kv_state, *score_state;         // [bsz, ratio, 512]
  bf16_t* latents;                       // [bsz, g, 512]
  const float* norm_w;
  int n, m, g, rem;                      // tokens, carried rows, complete groups, rows left open
  float eps;
};

// Channels tid + 256 u of NR projected rows: v[i][0] kv, v[i][1] score. Every load of up to four ranges
// goes out before the first sum: a row at a time, each sum waited for its own loads (a token of 64
// sequences 22.3 us against 14.6).
constexpr int kChunkU = kChunkDim / 256;
template <int NR>
__device__ __forceinline__ void proj_values(const ProjArgs& a, const int (&row)[NR], int tid, float (&v)[NR][2][kChunkU]) {
  const bool parts = a.splits > 1;
  const int64_t total = (int64_t)a.rows * a.n;
  const float* p[NR][2];
#pragma unroll
  for (int i = 0; i < NR; ++i)
#pragma unroll
    for (int z = 0; z < 2; ++z) {
      p[i][z] = parts ? a.part + (int64_t)row[i] * a.n + z * kChunkDim
                      : (z ? a.y1 : a.y0) + (int64_t)row[i] * kChunkDim;
#pragma unroll
      for (int u = 0; u < kChunkU; ++u) v[i][z][u] = p[i][z][tid + 256 * u];
    }
  if (!parts) return;
#pragma unroll 4
  for (int s = 1; s < a.splits; ++s)
#pragma unroll
    for (int i = 0; i < NR; ++i)
#pragma unroll
      for (int z = 0; z < 2; ++z)
#pragma unroll
        for (int u = 0; u < kChunkU; ++u) v[i][z][u] += (p[i][z] + s * total)[tid + 256 * u];
}

template <int R>
__global__ __launch_bounds__(256) void compress_chunk_kernel(ChunkArgs a) {
  constexpr int U = kChunkU;
  __shared__ float red[4];
  const int b = blockIdx.y, j = blockIdx.x, tid = threadIdx.x;
  float* kst = a.kv_state + (int64_t)b * R * kChunkDim;
  float* sst = a.score_state + (int64_t)b * R * kChunkDim;
  if (a.g > 0) {
    // rows j R .. of concat(state[:m], chunk); a carried one reads the chunk's first row and drops it
    int row[R];
    float v[R][2][U], carried[R][2][U];
    const int held = max(a.m - j * R, 0);          // uniform: only group 0 meets carried rows
#pragma unroll
    for (int q = 0; q < R; ++q) row[q] = b * a.n + max(j * R + q - a.m, 0);
    if (held > 0) {
#pragma unroll
      for (int q = 0; q < R; ++q)
#pragma unroll
        for (int u = 0; u < U; ++u) {
          carried[q][0][u] = kst[q * kChunkDim + tid + 256 * u];
          carried[q][1][u] = sst[q * kChunkDim + tid + 256 * u];
        }
    }
    proj_values<R>(a.p, row, tid, v);
    if (held > 0) {
#pragma unroll
      for (int q = 0; q < R; ++q)
#pragma unroll
        for (int z = 0; z < 2; ++z)
#pragma unroll
          for (int u = 0; u < U; ++u) v[q][z][u] = q < held ? carried[q][z][u] : v[q][z][u];
    }
    float pooled[U], ss = 0.0f;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      float mx = -INFINITY;
#pragma unroll
      for (int q = 0; q < R; ++q) mx = fmaxf(mx, v[q][1][u]);
      float w[R], den = 0.0f;
#pragma unroll
      for (int q = 0; q < R; ++q) den += w[q] = expf(v[q][1][u] - mx);
      float acc = 0.0f;
#pragma unroll
      for (int q = 0; q < R; ++q) acc += v[q][0][u] * (w[q] / den);
      pooled[u] = io<bf16_t>::rnd(acc);  // rounded to the latents' type before the norm
      ss += pooled[u] * pooled[u];
    }
    ss = group_sum(ss, 64);
    if ((tid & 63) == 0) red[tid >> 6] = ss;
    __syncthreads();
    float tot = 0.0f;
#pragma unroll
    for (int w = 0; w < 4; ++w) tot += red[w];
    const float inv = 1.0f / sqrtf(tot / (float)kChunkDim + a.eps);
    bf16_t* out = a.latents + ((int64_t)b * a.g + j) * kChunkDim;
#pragma unroll
    for (int u = 0; u < U; ++u) io<bf16_t>::st(out + tid + 256 * u, a.norm_w[tid + 256 * u] * (pooled[u] * inv));
  }
  // the open group's rows, by the workgroup that has read the carried ones (each thread its channels)
  if (j == 0) {
    for (int r = 0; r < a.rem; ++r) {
      const int t = a.m + a.n - a.rem + r;
      if (t < a.m) continue;             // a carried row, already in place
      const int row[1] = {b * a.n + t - a.m};
      float v[1][2][U];
      proj_values<1>(a.p, row, tid, v);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        kst[r * kChunkDim + tid + 256 * u] = v[0][0][u];
        sst[r * kChunkDim + tid + 256 * u] = v[0][1][u];
      }
    }
  }
}

template <int WR, int WM, int GR, int GM>
static void launch_proj(const ProjArgs& a, hipStream_t stream) {
  using C = ProjCfg<WR, WM, GR, GM>;
  const int64_t tiles = (int64_t)(a.n / C::TR) * a.splits * ((a.rows + C::TM - 1) / C::TM);
  hipLaunchKernelGGL((proj_f32_kernel<WR, WM, GR, GM>), dim3((unsigned)tiles), dim3(C::NT), 0, stream, a);
}

struct ProjPlan {
  int tr, tm, splits;
};

// Decode row counts: small tiles and as many contraction ranges as fit one round of 256 workgroups
// (one per CU). Chunks: of three activation tiles and up to 40 ranges the pair with the least time as
// measured per part (k = 5120, n = 1024): a round of workgroups takes 1.25, 1.66 or 2.56 us per
// 64-channel step with 64, 128 or 256 activation rows, and 3 us to start and end; each range's partial
// sums cost a write and a read at 5 TB/s. Within a few us of every size timed: 300 rows 29.4 -> 25.5 us,
// 1,000 rows 58.5 -> 42.0, 2,500 rows 137.6 -> 83.4, 4,096 rows 140.9 -> 117.4, 5,000 rows 207 -> 157.7 (before: the
// tile by row count alone, ranges of equal length only).
static ProjPlan proj_plan(int rows, int k, int n) {
  const int steps = k / 64;
  if (rows <= 128) {
    const int t = rows <= 32 ? 32 : 64;
    ProjPlan p{t, t, 1};
    const int64_t tiles = (int64_t)(n / p.tr) * ((rows + p.tm - 1) / p.tm);
    for (int s = 2; s <= 40; ++s)
      if (steps % s == 0 && tiles * s <= 256) p.splits = s;
    return p;
  }
  static const int kRows[3] = {64, 128, 256};
  static const double kStepUs[3] = {1.25, 1.66, 2.56};
  ProjPlan p{128, 256, 1};
  double best = 1e30;
  for (int t = 0; t < 3; ++t) {
    const int64_t tiles = (int64_t)(n / 128) * ((rows + kRows[t] - 1) / kRows[t]);
    for (int s = 1; s <= 40 && s <= steps; ++s) {
      const double us = (double)((tiles * s + 255) / 256) * ((steps + s - 1) / s * kStepUs[t] + 3.0) +
                        (s > 1 ? (double)s * rows * n * 8.0 / 5e6 : 0.0);
      if (us < best) {
        best = us;
        p.tm = kRows[t];
        p.splits = s;
      }
    }
  }
  return p;
}

}  // namespace dsv41

using namespace dsv41;

extern "C" size_t dsv41_linear_f32_pair_workspace_bytes(int32_t rows, int32_t k, int32_t n0, int32_t n1) {
  if (rows <= 0 || k <= 0 || n0 <= 0 || n1 < 0) return 0;
  const int n = n0 + n1;
  if (k % 64 || n0 % 128 || n1 % 128) return 0;
  const ProjPlan p = proj_plan(rows, k, n);
  return p.splits > 1 ? (size_t)p.splits * (size_t)rows * (size_t)n * sizeof(float) : 0;
}

// The checks of both entries below, then the projections: into y0 and y1, or into the workspace's parts.
static int run_proj(const char* what, ProjArgs& a, const ProjPlan& p, size_t workspace_bytes, hipStream_t stream) {
  DSV41_REQUIRE(a.k % 64 == 0 && a.n0 % 128 == 0 && (a.n - a.n0) % 128 == 0, DSV41_E_SHAPE,
                "%s: k = %d must be a multiple of 64, n0 = %d and n1 = %d of 128", what, a.k, a.n0, a.n - a.n0);
  DSV41_REQUIRE(aligned16(a.x) && aligned16(a.w0) && aligned16(a.w1) && aligned16(a.y0) && aligned16(a.y1), DSV41_E_ARG,
                "%s: tensors must be 16-byte aligned", what);
  DSV41_REQUIRE((int64_t)(a.n / p.tr) * p.splits * (((int64_t)a.rows + p.tm - 1) / p.tm) < (1ll << 31), DSV41_E_ARG,
                "%s: too many tiles", what);
  const size_t need = p.splits > 1 ? (size_t)p.splits * (size_t)a.rows * (size_t)a.n * sizeof(float) : 0;
  DSV41_REQUIRE(workspace_bytes >= need && (need == 0 || (a.part && aligned16(a.part))), DSV41_E_WORKSPACE,
                "%s: workspace of %zu bytes needed, %zu given", what, need, workspace_bytes);
  a.splits = p.splits;
  if (p.tr == 32) launch_proj<1, 1, 2, 2>(a, stream);
  else if (p.tr == 64) launch_proj<1, 2, 4, 2>(a, stream);
  else if (p.tm == 64) launch_proj<2, 2, 4, 2>(a, stream);
  else if (p.tm == 128) launch_proj<2, 4, 4, 2>(a, stream);
  else launch_proj<4, 4, 2, 4>(a, stream);
  return check_launch(what);
}

extern "C" int dsv41_linear_f32_pair(const void* x, const float* w0, const float* w1, float* y0, float* y1,
                                     void* workspace, size_t workspace_bytes, int32_t rows, int32_t k, int32_t n0,
                                     int32_t n1, int32_t dtype, hipStream_t stream) {
  const char* what = "dsv41_linear_f32_pair";
  DSV41_REQUIRE(x && w0 && w1 && y0 && y1, DSV41_E_ARG, "%s: null tensor", what);
  DSV41_REQUIRE(dtype == DSV41_BF16, DSV41_E_DTYPE, "%s: bf16 activations only (dtype %d)", what, dtype);
  DSV41_REQUIRE(rows >= 0 && k > 0 && n0 > 0 && n1 > 0 && (int64_t)n0 + n1 < (1 << 24), DSV41_E_ARG, "%s: bad sizes", what);
  if (rows == 0) return 0;
  const ProjPlan p = proj_plan(rows, k, n0 + n1);
  ProjArgs a{static_cast<const bf16_t*>(x), w0, w1, y0, y1, static_cast<float*>(workspace), rows, k, n0 + n1, n0, 1};
  const int rc = run_proj(what, a, p, workspace_bytes, stream);
  if (rc || p.splits <= 1) return rc;
  const int64_t quads = (int64_t)rows * a.n / 4;
  hipLaunchKernelGGL(proj_reduce_kernel, dim3((unsigned)((quads + 255) / 256)), dim3(256), 0, stream, a);
  return check_launch(what);
}

extern "C" size_t dsv41_compress_chunk_workspace_bytes(int32_t rows, int32_t k, int32_t dim) {
  const size_t parts = dsv41_linear_f32_pair_workspace_bytes(rows, k, dim, dim);
  return parts ? parts : (rows > 0 && dim > 0 ? 2 * (size_t)rows * (size_t)dim * sizeof(float) : 0);
}

extern "C" int dsv41_compress_chunk(const void* x, const float* w0, const float* w1, float* kv_state, float* score_state,
                                    void* latents, const float* norm_w, void* workspace, size_t workspace_bytes,
                                    int32_t bsz, int32_t n, int32_t k, int32_t dim, int32_t ratio, int32_t start_pos,
                                    float eps, int32_t dtype, hipStream_t stream) {
  const char* what = "dsv41_compress_chunk";
  DSV41_REQUIRE(x && w0 && w1 && kv_state && score_state && norm_w, DSV41_E_ARG, "%s: null tensor", what);
  DSV41_REQUIRE(dtype == DSV41_BF16, DSV41_E_DTYPE, "%s: bf16 activations only (dtype %d)", what, dtype);
  DSV41_REQUIRE(bsz >= 0 && bsz < 65536 && n >= 0 && k > 0 && start_pos >= 0 && (int64_t)bsz * n < (1ll << 31), DSV41_E_ARG,
                "%s: bad sizes", what);
  DSV41_REQUIRE(dim == kChunkDim && (ratio == 2 || ratio == 4), DSV41_E_SHAPE,
                "%s: dim %d and ratio %d (%d channels, ratio 2 or 4)", what, dim, ratio, kChunkDim);
  const int rows = bsz * n;
  if (rows == 0) return 0;
  const int m = start_pos % ratio, total = m + n, g = total / ratio;
  DSV41_REQUIRE(g == 0 || latents, DSV41_E_ARG, "%s: latents is null but %d groups complete", what, g);
  const size_t need = dsv41_compress_chunk_workspace_bytes(rows, k, dim);
  DSV41_REQUIRE(workspace && aligned16(workspace) && workspace_bytes >= need, DSV41_E_WORKSPACE,
                "%s: workspace of %zu bytes needed, %zu given", what, need, workspace_bytes);
  const ProjPlan p = proj_plan(rows, k, 2 * dim);
  float* ws = static_cast<float*>(workspace);
  ChunkArgs c{{static_cast<const bf16_t*>(x), w0, w1, ws, ws + (size_t)rows * dim, ws, rows, k, 2 * dim, dim, 1},
              kv_state, score_state, static_cast<bf16_t*>(latents), norm_w, n, m, g, total % ratio, eps};
  const int rc = run_proj(what, c.p, p, workspace_bytes, stream);
  if (rc) return rc;
  const dim3 grid((unsigned)(g > 0 ? g : 1), (unsigned)bsz);
  if (ratio == 2) hipLaunchKernelGGL(compress_chunk_kernel<2>, grid, dim3(256), 0, stream, c);
  else hipLaunchKernelGGL(compress_chunk_kernel<4>, grid, dim3(256), 0, stream, c);
  return check_launch(what);
}
