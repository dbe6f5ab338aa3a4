// Token-batch projections on the matrix cores: fp32-accurate products of
// many token rows with bf16 weight matrices (the input and output projections
// of the DeltaNet and attention mixers over more than a few tokens).
//
// A token value v (fp32) enters as three bf16 terms, hi = bf16(v),
// mid = bf16(v - hi), lo = bf16(v - hi - mid): together the 24 bits of v, so
// every product with a bf16 weight is the fp32 one.  Two terms (16 bits)
// would lose precision against the fp32 VALU products these kernels replace.
// The MFMAs of one 64-wide K step start from zero and their sum is added to
// the tile's fp32 accumulator by the VALU, in the smaller tiles four steps at
// a time: K / 64 roundings of the full sum or fewer instead of 3 K / 32 (error
// against 64 bits 1.0e-7 of the result, 1.3e-7 with the largest tile; the VALU
// kernels' 1.3e-7; accumulating in the MFMA throughout, 4.9e-7).
//
// Tile: BN weight rows x BM tokens per workgroup, K in steps of 64.  Both
// operands go through LDS in 128-byte rows whose 16-byte chunks are
// XOR-swizzled by the row (chunk ^ (row & 7)): the row-wise staging writes and
// the operand reads (16 rows x 16 B) show no bank conflicts in the counters.  Weight and
// token loads are one to four steps ahead of the step that computes.
//
// An infinite weight makes its row NaN (an infinity times the terms' signs and
// zeros), a token's infinity its own products infinite or NaN as fp32 ones.
//
// What bounds it: at a few dozen tokens the latency of a step (LDS write,
// barrier, LDS read, a chain of six MFMAs: ~0.7 us with one workgroup on a
// CU), which double-buffered LDS, eight wavefronts and small tiles shorten; at
// hundreds of tokens the MFMAs with the fp32 -> bf16 split beside them, which
// large tiles amortise (770 of the 1206 TFLOP/s a library bf16 GEMM reaches,
// three MFMAs per product counted; under a profiler 40 to 46% of the busy CUs'
// matrix cycles).  The DeltaNet input projections (12,352 rows, K 2048), VALU
// kernel (whole rows per wavefront) / here, us: 8 tokens 38 / 25.5, 32 105 / 26,
// 64 197 / 31, 128 385 / 41, 256 796 / 64, 512 2056 / 101, 1000 4006 / 198.
#include "fk_common.h"
#include "fk_host.h"

namespace fk {

struct GemmArgs {
  const void* w[4];  // bf16 [rows[i], K], rows a multiple of 16 (0: unused)
  float* out[4];     // f32 [T, rows[i]]
  int rows[4];
  int R;             // sum of rows
  int T, K;
  // XM 0: token rows x [T, K] with RMSNorm and norm weight
  const void* x;
  const void* nw;
  float eps, off;
  // XM 1: token planes [3][T][K] (hi, mid, lo)
  const uint16_t* planes;
  const void* residual;  // [T, R] (nullable), with residual_out = residual + out[0]
  int residual_dt;
  float* residual_out;
  float* part;  // split K: partial sums [splits][T][R] instead of out
  int splits;
  int nrb, ntb;  // row and token tiles
  int vec;       // every output (and residual) is 16-byte aligned: 16-byte stores
};

constexpr int kGemmBK = 64;

__device__ __forceinline__ void store4(float* p, const float (&v)[4], bool vec) {
  if (vec) {
    *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
  } else {
#pragma unroll
    for (int q = 0; q < 4; ++q) p[q] = v[q];
  }
}

// XM: 0 = token rows normalised here (bf16 norm weight), 1 = token planes;
// BFX: dtype of x (XM 0); WN x WM wavefronts over the tile; DB: two LDS
// buffers, the next step staged beside this step's MFMAs (SF: issued before
// them); PW, PX: steps that the weight and token loads are ahead.
template <int BN, int BM, int WN, int WM, int OCC, bool DB, bool SF, int PW, int PX, int XM, bool BFX>
__global__ __launch_bounds__(64 * WN * WM, OCC) void token_gemm_kernel(GemmArgs a) {
  constexpr int RP = 8 * WN * WM;                  // rows staged per pass: 8 threads (16 B each) a row
  constexpr int WPT = BN / RP;                     // weight chunks per thread and step
  constexpr int XPT = BM / RP > 0 ? BM / RP : 1;   // token rows per thread and step (8 values each)
  constexpr int TN = BN / WN / 16, TM = BM / WM / 16, NBUF = DB ? 2 : 1;
  static_assert(BN % RP == 0 && TN >= 1 && TM >= 1, "tile and wavefronts");
  __shared__ u32x4 s_w[NBUF][BN * 8];
  __shared__ u32x4 s_x[NBUF][3 * BM * 8];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // Consecutive workgroups go to the 8 XCDs in turn: an XCD takes every
  // eighth row tile with all its token tiles, so a weight tile is read into
  // one L2.
  const int xcd = blockIdx.x & 7, loc = blockIdx.x >> 3;
  const int rb = (loc / a.ntb) * 8 + xcd, tb = loc % a.ntb;
  if (rb >= a.nrb) return;
  const int r0 = rb * BN, t0 = tb * BM;
  const int K = a.K, T = a.T, steps = K / kGemmBK;
  const int k_lo = (int)((long long)steps * blockIdx.y / a.splits) * kGemmBK;
  const int k_hi = (int)((long long)steps * (blockIdx.y + 1) / a.splits) * kGemmBK;

  const int srow = tid >> 3, chunk = tid & 7;
  const uint16_t* wp[WPT];
#pragma unroll
  for (int p = 0; p < WPT; ++p) {
    int row = min(r0 + p * RP + srow, a.R - 1), m = 0;
    if (row >= a.rows[0]) { row -= a.rows[0]; m = 1; }
    if (m == 1 && row >= a.rows[1]) { row -= a.rows[1]; m = 2; }
    if (m == 2 && row >= a.rows[2]) { row -= a.rows[2]; m = 3; }
    const void* base = m == 0 ? a.w[0] : m == 1 ? a.w[1] : m == 2 ? a.w[2] : a.w[3];
    wp[p] = reinterpret_cast<const uint16_t*>(base) + (size_t)row * K + chunk * 8;
  }
  const bool xrow_ok = BM >= RP || srow < BM;  // (a tile of fewer tokens than a pass stages: the spare threads repeat)
  size_t xo[XPT];
#pragma unroll
  for (int p = 0; p < XPT; ++p) xo[p] = (size_t)min(t0 + p * RP + (BM >= RP ? srow : srow % BM), T - 1) * K + chunk * 8;

  // Loads past the last step repeat it: straight-line, so that the waits
  // count exactly (a load under a condition waits for all before it).
  u32x4 wr[PW][WPT];
  Raw8<BFX> xr[PX][XPT];
  u32x4 pr[PX][XPT][3];
  Raw8<true> nwr[PX];
  auto load_w = [&](int k, int u) {
    k = min(k, k_hi - kGemmBK);
#pragma unroll
    for (int p = 0; p < WPT; ++p) wr[u][p] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wp[p] + k));
  };
  auto load_x = [&](int k, int u) {
    k = min(k, k_hi - kGemmBK);
    if constexpr (XM == 0) {
#pragma unroll
      for (int p = 0; p < XPT; ++p) xr[u][p] = load_raw8<BFX>(a.x, xo[p] + k);
      nwr[u] = load_raw8<true>(a.nw, (size_t)k + chunk * 8);
    } else {
      const size_t plane = (size_t)T * K;
#pragma unroll
      for (int p = 0; p < XPT; ++p)
#pragma unroll
        for (int q = 0; q < 3; ++q) pr[u][p][q] = *reinterpret_cast<const u32x4*>(a.planes + q * plane + xo[p] + k);
    }
  };
  float ss[XPT];
#pragma unroll
  for (int p = 0; p < XPT; ++p) ss[p] = 0.f;
  int staged = k_lo;  // the next step to stage (squares are added for real steps only)
  auto stage = [&](int b, int uw, int ux) {
    if constexpr (XM == 0) {
      float g[8];
      raw8_to_f32<true>(nwr[ux], g);
      const bool real = staged < k_hi;
#pragma unroll
      for (int p = 0; p < XPT; ++p) {
        float v[8], sq = 0.f;
        raw8_to_f32<BFX>(xr[ux][p], v);
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          sq = fmaf(v[q], v[q], sq);
          v[q] *= a.off + g[q];
        }
        ss[p] = real ? ss[p] + sq : ss[p];
        // (an infinity makes its row's scale 0 and the row NaN either way)
        split3_8<false>(v, pr[ux][p][0], pr[ux][p][1], pr[ux][p][2]);
      }
      staged += kGemmBK;
    }
    if (xrow_ok) {
#pragma unroll
      for (int p = 0; p < XPT; ++p) {
        const int r = p * RP + srow;
#pragma unroll
        for (int q = 0; q < 3; ++q) s_x[b][q * BM * 8 + r * 8 + (chunk ^ (r & 7))] = pr[ux][p][q];
      }
    }
#pragma unroll
    for (int p = 0; p < WPT; ++p) {
      const int r = p * RP + srow;
      s_w[b][r * 8 + (chunk ^ (r & 7))] = wr[uw][p];
    }
  };

  const int wn = wave / WM, wm = wave % WM;
  const int n = lane & 15, g4 = lane >> 4;
  // Sums of four steps at a time where the registers allow (TWO), then of
  // those: half the rounding error of one running sum of K / 64 terms.
  constexpr bool TWO = TN * TM <= 4;
  f32x4_t acc[TN][TM], sum[TWO ? TN : 1][TWO ? TM : 1];
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) {
      acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      if constexpr (TWO) sum[i][j] = acc[i][j];
    }
  auto flush = [&]() {
    if constexpr (TWO)
#pragma unroll
      for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j) {
          sum[i][j] += acc[i][j];
          acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
  };
  int nstep = 0;
  auto compute = [&](int b) {
    bf16x8_t av[TN][2];
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const int r = (wn * TN + i) * 16 + n;
        av[i][s] = __builtin_bit_cast(bf16x8_t, s_w[b][r * 8 + ((s * 4 + g4) ^ (r & 7))]);
      }
#pragma unroll
    for (int j = 0; j < TM; ++j) {
      const int r = (wm * TM + j) * 16 + n;
      bf16x8_t bv[3][2];
#pragma unroll
      for (int q = 0; q < 3; ++q)
#pragma unroll
        for (int s = 0; s < 2; ++s)
          bv[q][s] = __builtin_bit_cast(bf16x8_t, s_x[b][q * BM * 8 + r * 8 + ((s * 4 + g4) ^ (r & 7))]);
      f32x4_t c[TN];
#pragma unroll
      for (int i = 0; i < TN; ++i) c[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int q = 2; q >= 0; --q)  // the small terms first
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
          for (int i = 0; i < TN; ++i) c[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[i][s], bv[q][s], c[i], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < TN; ++i) acc[i][j] += c[i];
    }
    if ((++nstep & 3) == 0) flush();
  };

  constexpr int U0 = PW > PX ? PW : PX, U = DB && U0 < 2 ? 2 : U0;
#pragma unroll
  for (int u = 0; u < PX; ++u) load_x(k_lo + u * kGemmBK, u);
#pragma unroll
  for (int u = 0; u < PW; ++u) load_w(k_lo + u * kGemmBK, u);
  if constexpr (DB) {
    stage(0, 0, 0);
    load_x(k_lo + PX * kGemmBK, 0);
    load_w(k_lo + PW * kGemmBK, 0);
    __syncthreads();
    for (int k0 = k_lo; k0 < k_hi; k0 += U * kGemmBK) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = k0 + u * kGemmBK;
        if (k >= k_hi) break;
        // step k computes from buffer u & 1 while step k + 1 is staged into
        // the other (past the last step: the repeated loads, never read)
        if constexpr (SF) {
          stage((u & 1) ^ 1, (u + 1) % PW, (u + 1) % PX);
          compute(u & 1);
        } else {
          compute(u & 1);
          stage((u & 1) ^ 1, (u + 1) % PW, (u + 1) % PX);
        }
        load_x(k + (PX + 1) * kGemmBK, (u + 1) % PX);
        load_w(k + (PW + 1) * kGemmBK, (u + 1) % PW);
        __syncthreads();
      }
    }
  } else {
    for (int k0 = k_lo; k0 < k_hi; k0 += U * kGemmBK) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = k0 + u * kGemmBK;
        if (k >= k_hi) break;
        if (k > k_lo) __syncthreads();  // the previous step's operands are read
        stage(0, u % PW, u % PX);
        __syncthreads();
        load_x(k + PX * kGemmBK, u % PX);
        load_w(k + PW * kGemmBK, u % PW);
        compute(0);
      }
    }
    __syncthreads();
  }

  if constexpr (TWO) {
    flush();
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j) acc[i][j] = sum[i][j];
  }
  float* s_rs = reinterpret_cast<float*>(&s_x[0][0]);  // (every operand is read)
  if constexpr (XM == 0) {
    // 1 / rms of the tile's tokens: the 8 threads of a row add their squares
#pragma unroll
    for (int p = 0; p < XPT; ++p) {
      float v = ss[p];
      v += __uint_as_float(dpp_u32<kDppQuadXor1>(__float_as_uint(v)));
      v += __uint_as_float(dpp_u32<kDppQuadXor2>(__float_as_uint(v)));
      v += __uint_as_float(dpp_u32<kDppRowHalfMirror>(__float_as_uint(v)));
      if (chunk == 0 && xrow_ok) s_rs[p * RP + srow] = rsqrtf(v / (float)K + a.eps);
    }
    __syncthreads();
  }

  // lane: rows 4 g4 .. + 4 of a row tile (in one matrix: its rows are a
  // multiple of 16), token n of a token tile
#pragma unroll
  for (int i = 0; i < TN; ++i) {
    int row = r0 + (wn * TN + i) * 16;
    if (row >= a.R) continue;
    int m = 0;
    if (!a.part) {
      if (row >= a.rows[0]) { row -= a.rows[0]; m = 1; }
      if (m == 1 && row >= a.rows[1]) { row -= a.rows[1]; m = 2; }
      if (m == 2 && row >= a.rows[2]) { row -= a.rows[2]; m = 3; }
    }
    float* out = a.part ? a.part + (size_t)blockIdx.y * T * a.R : m == 0 ? a.out[0] : m == 1 ? a.out[1] : m == 2 ? a.out[2] : a.out[3];
    const int ld = a.part ? a.R : m == 0 ? a.rows[0] : m == 1 ? a.rows[1] : m == 2 ? a.rows[2] : a.rows[3];
#pragma unroll
    for (int j = 0; j < TM; ++j) {
      const int tl = (wm * TM + j) * 16 + n, t = t0 + tl;
      if (t >= T) continue;
      const float rs = XM == 0 ? s_rs[tl] : 1.f;
      const size_t o = (size_t)t * ld + row + g4 * 4;
      const float v[4] = {acc[i][j][0] * rs, acc[i][j][1] * rs, acc[i][j][2] * rs, acc[i][j][3] * rs};
      store4(out + o, v, a.vec);
      if (XM == 1 && !a.part && a.residual_out) {
        float r[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) r[q] = load_scalar(a.residual, a.residual_dt, o + q) + v[q];
        store4(a.residual_out + o, r, a.vec);
      }
    }
  }
}

// out = the sum of the K splits' partials (in split order), residual_out =
// residual + out.
struct GemmReduceArgs {
  const float* part;
  int splits;
  size_t n;  // T * R, a multiple of 16
  float* out;
  const void* residual;
  int residual_dt;
  float* residual_out;
  int vec;
};
__global__ __launch_bounds__(256) void token_gemm_reduce_kernel(GemmReduceArgs a) {
  const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= a.n) return;
  float4 v = *reinterpret_cast<const float4*>(a.part + i);
  for (int s = 1; s < a.splits; ++s) {
    const float4 p = *reinterpret_cast<const float4*>(a.part + (size_t)s * a.n + i);
    v.x += p.x;
    v.y += p.y;
    v.z += p.z;
    v.w += p.w;
  }
  const float o[4] = {v.x, v.y, v.z, v.w};
  store4(a.out + i, o, a.vec);
  if (a.residual_out) {
    float r[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) r[q] = load_scalar(a.residual, a.residual_dt, i + q) + o[q];
    store4(a.residual_out + i, r, a.vec);
  }
}

// Tiles, in the order of kGemmTiles.
template <int XM, bool BFX>
static void launch_tile(int tile, const GemmArgs& a, hipStream_t s) {
  const dim3 grid((unsigned)(((a.nrb + 7) / 8) * 8 * a.ntb), (unsigned)a.splits);
  switch (tile) {
#define FK_TILE(I, BN, BM, WN, WM, OCC, DB, SF, PW, PX)                                                             \
  case I:                                                                                                           \
    hipLaunchKernelGGL((token_gemm_kernel<BN, BM, WN, WM, OCC, DB, SF, PW, PX, XM, BFX>), grid, dim3(64 * WN * WM), \
                       0, s, a);                                                                                    \
    break;
    FK_TILE(0, 64, 32, 4, 2, 2, true, true, 4, 2)
    FK_TILE(1, 64, 64, 4, 2, 2, true, false, 2, 2)
    FK_TILE(2, 128, 64, 4, 2, 2, true, false, 2, 2)
    FK_TILE(3, 128, 128, 4, 4, 4, true, true, 1, 1)
    FK_TILE(4, 256, 128, 4, 4, 4, false, false, 1, 1)
#undef FK_TILE
  }
}

// Measured time of a tile's workgroups over K = 2048, us: one round of at
// most one workgroup per CU, and each further round (12,352 and 9,216 rows, 16
// to 1024 tokens, every tile at every size; further rounds of the small tiles
// share CUs).  The tile with the smallest estimate is taken: small tiles while
// one round of them holds the batch, large ones where the split of the tokens
// would be redone often (within 2% of the best tile on average, 11% at worst:
// 105 for 93 at 257 to 320 tokens of 12,352 rows).
struct GemmTile {
  int bn, bm;
  float first, next;
};
constexpr GemmTile kGemmTiles[] = {{64, 32, 26.f, 13.f}, {64, 64, 31.5f, 19.f}, {128, 64, 39.f, 34.f}, {128, 128, 57.f, 58.f}, {256, 128, 90.f, 97.f}};

static int pick_tile(int T, int R, int splits) {
  const int cus = device_cus() > 0 ? device_cus() : 256;
  int best = 0;
  float best_us = 0.f;
  for (int i = 0; i < (int)(sizeof(kGemmTiles) / sizeof(kGemmTiles[0])); ++i) {
    const GemmTile& t = kGemmTiles[i];
    const long long wgs = (long long)((R + t.bn - 1) / t.bn) * ((T + t.bm - 1) / t.bm) * splits;
    const float us = t.first + t.next * (float)((wgs + cus - 1) / cus - 1);
    if (i == 0 || us < best_us) {
      best = i;
      best_us = us;
    }
  }
  return best;
}

bool norm_gemm_ok(const int (&rows)[4], int K, int weight_dt, int nw_dt) {
  for (int r : rows)
    if (r % 16) return false;
  return weight_dt == FK_DTYPE_BF16 && nw_dt == FK_DTYPE_BF16 && K >= kGemmBK && K % kGemmBK == 0;
}

int launch_norm_gemm(const void* x, int x_dt, const void* nw, const void* const (&w)[4],
                     const int (&rows)[4], float* const (&out)[4], int T, int K, float eps, float off,
                     hipStream_t s) {
  GemmArgs a = {};
  a.R = 0;
  for (int i = 0; i < 4; ++i) {
    a.w[i] = w[i];
    a.rows[i] = rows[i];
    a.out[i] = out[i];
    a.R += rows[i];
  }
  a.T = T;
  a.K = K;
  a.x = x;
  a.nw = nw;
  a.eps = eps;
  a.off = off;
  a.splits = 1;
  a.vec = 1;
  for (int i = 0; i < 4; ++i)
    if (rows[i] && !aligned16(out[i])) a.vec = 0;
  const int tile = pick_tile(T, a.R, 1);
  a.nrb = (a.R + kGemmTiles[tile].bn - 1) / kGemmTiles[tile].bn;
  a.ntb = (T + kGemmTiles[tile].bm - 1) / kGemmTiles[tile].bm;
  if (x_dt == FK_DTYPE_BF16) launch_tile<0, true>(tile, a, s);
  else launch_tile<0, false>(tile, a, s);
  return check_launch("token_gemm_kernel");
}

// Tile and K splits of launch_plane_gemm.  A split is one more round of
// partial sums through memory, but a quarter of the K steps on four times the
// CUs where a batch has few tiles.  Estimate, us (measured at 2,048 rows, K
// 4096, 4 to 1000 tokens; splits up to 8): the tile's time over its share of K
// + the launch, and the reduction's launch and traffic.  us with the best
// split and without: 32 tokens 13 / 36, 64 16 / 35, 128 20 / 35, 256 25 / 36,
// 512 38 / 43, 1000 57.
static void plane_tiles(int T, int R, int K, size_t part_bytes, int& tile, int& splits) {
  constexpr float kFirst[] = {17.f, 20.5f, 25.5f, 44.f, 80.f};
  const int cus = device_cus() > 0 ? device_cus() : 256;
  float best = 0.f;
  tile = -1;
  for (int i = 0; i < (int)(sizeof(kGemmTiles) / sizeof(kGemmTiles[0])); ++i) {
    const GemmTile& t = kGemmTiles[i];
    const long long tiles = (long long)((R + t.bn - 1) / t.bn) * ((T + t.bm - 1) / t.bm);
    for (int s = 1; s <= 8; s *= 2) {
      if (s > 1 && (tiles * s > cus || K / kGemmBK < 4 * s || (size_t)s * T * R * 4 > part_bytes)) break;
      float us = 5.f + (kFirst[i] + t.next * (float)((tiles * s + cus - 1) / cus - 1)) * (float)K / (2048.f * s);
      if (s > 1) us += 3.f + (float)s * T * R * 8.f / 3.0e6f;
      if (tile < 0 || us < best) {
        best = us;
        tile = i;
        splits = s;
      }
    }
  }
}

bool plane_gemm_ok(int R, int K, int weight_dt) {
  return weight_dt == FK_DTYPE_BF16 && R % 16 == 0 && K >= kGemmBK && K % kGemmBK == 0;
}

int launch_plane_gemm(const uint16_t* planes, const void* w, int R, int T, int K, const void* residual,
                      int residual_dt, float* out, float* residual_out, float* part, size_t part_bytes,
                      hipStream_t s) {
  GemmArgs a = {};
  int tile;
  plane_tiles(T, R, K, part_bytes, tile, a.splits);
  a.w[0] = w;
  a.rows[0] = R;
  a.out[0] = out;
  a.R = R;
  a.T = T;
  a.K = K;
  a.planes = planes;
  a.residual = residual;
  a.residual_dt = residual_dt;
  a.residual_out = residual_out;
  a.part = a.splits > 1 ? part : nullptr;
  const int vec = aligned16(out) && (!residual_out || aligned16(residual_out));
  a.vec = a.part || vec;
  a.nrb = (R + kGemmTiles[tile].bn - 1) / kGemmTiles[tile].bn;
  a.ntb = (T + kGemmTiles[tile].bm - 1) / kGemmTiles[tile].bm;
  launch_tile<1, false>(tile, a, s);
  int st = check_launch("token_gemm_kernel");
  if (st || a.splits == 1) return st;
  GemmReduceArgs r;
  r.part = part;
  r.splits = a.splits;
  r.n = (size_t)T * R;
  r.out = out;
  r.residual = residual;
  r.residual_dt = residual_dt;
  r.residual_out = residual_out;
  r.vec = vec;
  hipLaunchKernelGGL(token_gemm_reduce_kernel, dim3((unsigned)((r.n / 4 + 255) / 256)), dim3(256), 0, s, r);
  return check_launch("token_gemm_reduce_kernel");
}

}  // namespace fk
