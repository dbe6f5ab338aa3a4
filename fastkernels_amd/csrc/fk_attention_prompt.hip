// Gated attention over many rows of one sequence (a prompt, or a chunk of one
// behind a filled cache), on the matrix cores.  Semantics: fk_attention.hip.
//
//   launch_norm_gemm          [q | gate], k and v of every row (fk_gemm.hip)
//   attn_prompt_prep_kernel   head norms and RoPE: scaled queries, the rows'
//                             keys (fp32, and rounded into the cache with v)
//   attn_prompt_kernel        (chunk of positions, kv head, 64 query rows):
//                             online softmax over tiles of 16 positions,
//                             scores and weighted values as
//                             v_mfma_f32_16x16x4_f32: fp32 products and sums
//   attn_prompt_merge_kernel  chunk partials, output gate, the gated values as
//                             three bf16 terms
//   launch_plane_gemm         output projection and residual (fk_gemm.hip)
//
// Calls of 32 rows (four launches, each streaming every weight, with VALU
// dot products) took 1417 us for 200 rows behind 1,000 positions and 2650 for
// 256 behind 3,000; this takes 179 to 187 and 265.  The rows' own keys and
// values enter unrounded for every row of the call, whatever the cache's type.
#include "fk_common.h"
#include "fk_host.h"

namespace fk {

constexpr int kPromptHd = 256;    // head_dim
constexpr int kPromptRows = 64;   // query rows (token, head of one kv head) per workgroup, 16 per wavefront
constexpr int kPromptTile = 16;   // positions per tile
// Workgroups aimed at when the positions are split into chunks: two per CU.
// (384 / 512 / 1024, us a call: 256 rows behind 3,000 positions 302 / 266 /
// 276, 200 behind 1,000 174 / 186 / 174, 64 behind 3,000 122 / 118 / 135, 32
// behind 3,000 99 / 102 / 102: more chunks cost the merge.)
constexpr int kPromptWgs = 512;
constexpr int kPromptMaxChunks = 64;

struct PromptArgs {
  const float* qg;  // [T, heads, 2 hd] query and gate
  const float* k;   // [T, kvh, hd] before norm and RoPE
  const float* v;   // [T, kvh, hd]
  const void* qn_w;
  const void* kn_w;
  int qn_dt, kn_dt;
  void* kc;
  void* vc;
  const int* start_dev;
  int start, max_pos;
  int T, heads, kvh;
  int rope_dim, interleaved;
  float theta_log2, eps;
  float* q_rot;  // [T, heads, hd] normalised, rotated, times hd^-1/2
  float* k_rot;  // [T, kvh, hd]
  int* v_bad;    // [T, kvh] whether the row's values hold an infinity or NaN
  float* stat;   // [T, heads, nc, 2] chunk maximum and sum
  float* acc;    // [T, heads, nc, hd] chunk's weighted values
  int nc, chunk; // chunks of positions
  int ntb;       // row blocks
  uint16_t* planes;  // [3][T][heads * hd]
  uint32_t* err;
};

// The start position, or -1 when a device-held one leaves the cache.
__device__ __forceinline__ int prompt_start(const PromptArgs& a) {
  const int s = a.start_dev ? *a.start_dev : a.start;
  return positions_in_cache(s, a.T, a.max_pos) ? s : -1;
}

template <bool CBF>
__global__ __launch_bounds__(256) void attn_prompt_prep_kernel(PromptArgs a) {
  constexpr int hd = kPromptHd;
  __shared__ float s_row[4][hd];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int per = a.heads + a.kvh;
  const long long row = (long long)blockIdx.x * 4 + wave;  // (token, query head or kv head)
  const bool in = row < (long long)a.T * per;
  const int t = in ? (int)(row / per) : 0, h = in ? (int)(row - (long long)t * per) : 0;
  const bool key = h >= a.heads;
  const int j = h - a.heads;
  const int start = prompt_start(a);
  const float* src = key ? a.k + ((size_t)t * a.kvh + j) * hd : a.qg + ((size_t)t * a.heads + h) * 2 * hd;
  const float4 x4 = *reinterpret_cast<const float4*>(src + lane * 4);
  const float x[4] = {x4.x, x4.y, x4.z, x4.w};
  const float ss = wave_sum((x[0] * x[0] + x[1] * x[1]) + (x[2] * x[2] + x[3] * x[3]));
  const float r = rsqrtf(ss / (float)hd + a.eps);
  float y[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float w = load_scalar(key ? a.kn_w : a.qn_w, key ? a.kn_dt : a.qn_dt, lane * 4 + q);
    y[q] = x[q] * r * (1.f + w);
    s_row[wave][lane * 4 + q] = y[q];
  }
  __syncthreads();
  if (!in) return;
  const int rd = a.rope_dim, pos = (start < 0 ? 0 : start) + t;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int d = lane * 4 + q;
    if (d < rd) {
      int i, partner;
      float sign;
      if (a.interleaved) {
        i = d >> 1;
        partner = d ^ 1;
        sign = (d & 1) ? 1.f : -1.f;
      } else {
        const int hh = rd >> 1;
        i = d < hh ? d : d - hh;
        partner = d < hh ? d + hh : d - hh;
        sign = d < hh ? -1.f : 1.f;
      }
      const float inv_freq = exp2f(-(float)(2 * i) / (float)rd * a.theta_log2);
      float sn, cs;
      sincosf((float)pos * inv_freq, &sn, &cs);
      y[q] = y[q] * cs + sign * s_row[wave][partner] * sn;
    }
  }
  if (!key) {
    const float scale = rsqrtf((float)hd);
    *reinterpret_cast<float4*>(a.q_rot + ((size_t)t * a.heads + h) * hd + lane * 4) =
        make_float4(y[0] * scale, y[1] * scale, y[2] * scale, y[3] * scale);
    return;
  }
  *reinterpret_cast<float4*>(a.k_rot + ((size_t)t * a.kvh + j) * hd + lane * 4) = make_float4(y[0], y[1], y[2], y[3]);
  if (start < 0) return;  // no cache access
  const float4 v4 = *reinterpret_cast<const float4*>(a.v + ((size_t)t * a.kvh + j) * hd + lane * 4);
  const bool bad = __ballot(!(fabsf(v4.x) < INFINITY && fabsf(v4.y) < INFINITY && fabsf(v4.z) < INFINITY &&
                              fabsf(v4.w) < INFINITY)) != 0ull;
  if (lane == 0) a.v_bad[t * a.kvh + j] = bad;
  const size_t o = ((size_t)(start + t) * a.kvh + j) * hd + lane * 4;
  if constexpr (CBF) {
    // (the same rounding as store_scalar's, NaN kept)
    const float v[4] = {v4.x, v4.y, v4.z, v4.w};
    uint32_t kp[2], vp[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      kp[q] = (uint32_t)f32_to_bf16_bits(y[2 * q]) | ((uint32_t)f32_to_bf16_bits(y[2 * q + 1]) << 16);
      vp[q] = (uint32_t)f32_to_bf16_bits(v[2 * q]) | ((uint32_t)f32_to_bf16_bits(v[2 * q + 1]) << 16);
    }
    *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(a.kc) + o) = make_uint2(kp[0], kp[1]);
    *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(a.vc) + o) = make_uint2(vp[0], vp[1]);
  } else {
    *reinterpret_cast<float4*>(reinterpret_cast<float*>(a.kc) + o) = make_float4(y[0], y[1], y[2], y[3]);
    *reinterpret_cast<float4*>(reinterpret_cast<float*>(a.vc) + o) = v4;
  }
}

// Wavefront w: query rows 16 w .. + 16 of the block (row = token * G + head of
// kv head j), one per lane l % 16.  MFMA operands (16x16x4: lane l holds row
// or column l % 16 at k = l / 16) with the k order chosen so that lanes read
// 16 bytes at a time:
//   S^T = K Q^T: step (J, i) takes dim 16 J + 4 (l / 16) + i; result: lane's
//     query l % 16, positions 4 (l / 16) + q
//   O^T = V^T P^T: step q takes position 4 (l / 16) + q, which is where the
//     lane's probability already is; row r of value tile (g, i) is dim
//     64 g + 4 r + i
// Products of 16 dims (scores) and of a tile's 16 positions (values) start
// from zero and are added by the VALU, the scores' in pairs: summed inside the
// MFMAs throughout (chains of 128 products, and the running sum of the values)
// the calls' error against 64 bits was 6.3e-7 to 9.1e-7 at 300 to 3,000
// positions, where it is 3.1e-7 to 4.3e-7 (the VALU dot products that this
// replaced: 3.3e-7 to 4.4e-7), for 1 to 2% of a call's time.
// The 16-byte chunks of a tile row are XOR-swizzled by the row.  Bound by the
// fp32 MFMAs (128 of 32 cycles a wavefront and tile) and, between them, the
// tile's chain of sums, maximum, exponentials and barrier, which the second
// workgroup of the CU covers in part.
template <bool CBF>
__global__ __launch_bounds__(256, 2) void attn_prompt_kernel(PromptArgs a) {
  constexpr int hd = kPromptHd, CH = hd / 4;
  __shared__ f32x4_t s_k[2][kPromptTile][CH];
  __shared__ f32x4_t s_v[2][kPromptTile][CH];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int n = lane & 15, g4 = lane >> 4;
  // the row blocks of a (chunk, kv head) on one XCD: they read the same rows
  const int xcd = blockIdx.x & 7, loc = blockIdx.x >> 3;
  const int cj = (loc / a.ntb) * 8 + xcd, tb = loc % a.ntb;
  if (cj >= a.nc * a.kvh) return;
  const int c = cj / a.kvh, j = cj - c * a.kvh;
  const int G = a.heads / a.kvh, start = prompt_start(a);
  if (start < 0) return;
  const int tpb = kPromptRows / G;  // tokens per block (G divides 64)
  const int t0 = tb * tpb, t_last = min(t0 + tpb, a.T) - 1;
  const int p_lo = c * a.chunk, p_hi = min(p_lo + a.chunk, start + t_last + 1);
  if (p_lo >= p_hi) return;  // (the merge takes only the chunks a token reaches)
  const int row = wave * 16 + n, tq = t0 + row / G, hq = j * G + row % G;
  const bool live = tq <= t_last;
  const int t = live ? tq : t_last;  // (rows past the last token repeat it; not stored)
  const int pos = start + t;

  f32x4_t q[16];
  {
    const float* qp = a.q_rot + ((size_t)t * a.heads + hq) * hd + g4 * 4;
#pragma unroll
    for (int J = 0; J < 16; ++J) q[J] = *reinterpret_cast<const f32x4_t*>(qp + J * 16);
  }
  // tile rows: wavefront w stages positions w, w + 4, .. (a row is 64 lanes x
  // 4 values); positions from `start` on come from this call's own keys and
  // values
  f32x4_t rk[4], rv[4];
  auto fetch = [&](int p0) {  // (unconditional, clamped: positions past the chunk repeat its last)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int p = min(p0 + wave + 4 * i, p_hi - 1);
      const size_t own = ((size_t)(p < start ? 0 : p - start) * a.kvh + j) * hd + lane * 4;
      const size_t at = ((size_t)p * a.kvh + j) * hd + lane * 4;
      if constexpr (CBF) {
        if (p < start) {  // (uniform)
          const uint2 k2 = *reinterpret_cast<const uint2*>(reinterpret_cast<const uint16_t*>(a.kc) + at);
          const uint2 v2 = *reinterpret_cast<const uint2*>(reinterpret_cast<const uint16_t*>(a.vc) + at);
          rk[i] = f32x4_t{__uint_as_float(k2.x << 16), __uint_as_float(k2.x & 0xffff0000u), __uint_as_float(k2.y << 16),
                          __uint_as_float(k2.y & 0xffff0000u)};
          rv[i] = f32x4_t{__uint_as_float(v2.x << 16), __uint_as_float(v2.x & 0xffff0000u), __uint_as_float(v2.y << 16),
                          __uint_as_float(v2.y & 0xffff0000u)};
        } else {
          rk[i] = *reinterpret_cast<const f32x4_t*>(a.k_rot + own);
          rv[i] = *reinterpret_cast<const f32x4_t*>(a.v + own);
        }
      } else {
        const float* kp = p < start ? reinterpret_cast<const float*>(a.kc) + at : a.k_rot + own;
        const float* vp = p < start ? reinterpret_cast<const float*>(a.vc) + at : a.v + own;
        rk[i] = *reinterpret_cast<const f32x4_t*>(kp);
        rv[i] = *reinterpret_cast<const f32x4_t*>(vp);
      }
    }
  };
  // A tile may hold positions that some of its queries do not see: their
  // probabilities are 0, which an infinity or NaN among the values (a later
  // token's) would still turn into NaN.  Such values of the call's own rows
  // are staged as 0; attn_prompt_merge_kernel adds them for the queries that
  // see them.
  auto stage = [&](int b, int p0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = wave + 4 * i;
      f32x4_t v4 = rv[i];
      const bool own = min(p0 + r, p_hi - 1) >= start;  // (uniform)
#pragma unroll
      for (int e = 0; e < 4; ++e) v4[e] = own && !(fabsf(v4[e]) < INFINITY) ? 0.f : v4[e];
      s_k[b][r][lane ^ r] = rk[i];
      s_v[b][r][lane ^ r] = v4;
    }
  };
  // the swizzled chunks, up to multiples of 16 (four addresses each, not one per read)
  int kx[4], vx[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    kx[i] = (i * 4 + g4) ^ n;  // chunk 4 J + l / 16 of key l % 16: 16 (J / 4) + kx[J % 4]
    vx[i] = n ^ (g4 * 4 + i);  // chunk 16 g + l % 16 of key 4 (l / 16) + i: 16 g + vx[i]
  }
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  // four steps of a product, from zero
  auto product = [&](const f32x4_t& x, const f32x4_t& y) __attribute__((always_inline)) {
    f32x4_t c = zero;
#pragma unroll
    for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_16x16x4f32(x[e], y[e], c, 0, 0, 0);
    return c;
  };
  f32x4_t o[16];
#pragma unroll
  for (int d = 0; d < 16; ++d) o[d] = zero;
  float m = -INFINITY, l = 0.f;

  fetch(p_lo);
  stage(0, p_lo);
  __syncthreads();
  for (int p0 = p_lo, b = 0; p0 < p_hi; p0 += kPromptTile, b ^= 1) {
    fetch(p0 + kPromptTile);
    f32x4_t s4;  // (the products of 16 dims each, added in pairs)
    {
      auto dims16 = [&](int J) __attribute__((always_inline)) { return product(s_k[b][n][(J >> 2) * 16 + kx[J & 3]], q[J]); };
      auto dims64 = [&](int J) __attribute__((always_inline)) {
        const f32x4_t lo = dims16(J) + dims16(J + 1);
        return lo + (dims16(J + 2) + dims16(J + 3));
      };
      const f32x4_t lo = dims64(0) + dims64(4);
      s4 = lo + (dims64(8) + dims64(12));
    }
    f32x4_t p;
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int at = p0 + g4 * 4 + i;
      p[i] = at <= pos && at < p_hi ? s4[i] : -INFINITY;
      mx = fmaxf(mx, p[i]);
    }
    mx = fmaxf(mx, __uint_as_float(xor16_u32(__float_as_uint(mx))));
    mx = fmaxf(mx, __uint_as_float(xor32_u32(__float_as_uint(mx))));
    const float mn = fmaxf(m, mx);
    const float f = m == -INFINITY ? 0.f : __expf(m - mn);  // (nothing summed yet: 0)
#pragma unroll
    for (int i = 0; i < 4; ++i) p[i] = p[i] == -INFINITY ? 0.f : __expf(p[i] - mn);
    l = fmaf(l, f, (p[0] + p[1]) + (p[2] + p[3]));
    m = mn;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      f32x4_t v4[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) v4[i] = s_v[b][g4 * 4 + i][g * 16 + vx[i]];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const f32x4_t c = product(f32x4_t{v4[0][e], v4[1][e], v4[2][e], v4[3][e]}, p);
#pragma unroll
        for (int r = 0; r < 4; ++r) o[g * 4 + e][r] = fmaf(o[g * 4 + e][r], f, c[r]);
        asm volatile("" : "+v"(o[g * 4 + e]));  // (sunk into the loop's next block, the updates would keep every product)
      }
    }
    stage(b ^ 1, p0 + kPromptTile);  // (past the last tile: not read)
    __syncthreads();
  }
  l += __uint_as_float(xor16_u32(__float_as_uint(l)));
  l += __uint_as_float(xor32_u32(__float_as_uint(l)));
  if (!live) return;
  const size_t base = ((size_t)t * a.heads + hq) * a.nc + c;
  if (g4 == 0) *reinterpret_cast<float2*>(a.stat + base * 2) = make_float2(m, l);
  // o[4 g + i][q']: dim 64 g + 4 (4 g4 + q') + i
#pragma unroll
  for (int g = 0; g < 4; ++g)
#pragma unroll
    for (int e = 0; e < 4; ++e)
      *reinterpret_cast<float4*>(a.acc + base * hd + g * 64 + (g4 * 4 + e) * 4) =
          make_float4(o[g * 4][e], o[g * 4 + 1][e], o[g * 4 + 2][e], o[g * 4 + 3][e]);
}

// A wavefront per (token, head): the chunks that the token reaches, against
// the largest chunk maximum in chunk order, the own values that are not
// finite, the output gate, three bf16 terms.
__global__ __launch_bounds__(256) void attn_prompt_merge_kernel(PromptArgs a) {
  constexpr int hd = kPromptHd;
  const int lane = threadIdx.x & 63;
  const long long row = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int start = prompt_start(a);
  if (start < 0 && blockIdx.x == 0 && threadIdx.x == 0)
    __hip_atomic_fetch_or(a.err, FK_DEVICE_ERR_POSITION, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (row >= (long long)a.T * a.heads) return;
  const int t = (int)(row / a.heads);
  const int nc = start < 0 ? 0 : (start + t) / a.chunk + 1;  // chunks of positions 0 .. start + t
  const float* st = a.stat + (size_t)row * a.nc * 2;
  float M = -INFINITY;
  for (int c = lane; c < nc; c += kWave) M = fmaxf(M, st[c * 2]);
  M = wave_max(M);
  float L = 0.f;
  float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int c = 0; c < nc; ++c) {
    const float mc = st[c * 2], f = mc == -INFINITY ? 0.f : __expf(mc - M);
    const float4 v = *reinterpret_cast<const float4*>(a.acc + ((size_t)row * a.nc + c) * hd + lane * 4);
    L += st[c * 2 + 1] * f;
    o.x = fmaf(v.x, f, o.x);
    o.y = fmaf(v.y, f, o.y);
    o.z = fmaf(v.z, f, o.z);
    o.w = fmaf(v.w, f, o.w);
  }
  // the call's own values that are not finite, which the chunks summed as 0
  const int j = (int)(row - (long long)t * a.heads) / (a.heads / a.kvh);
  for (int u0 = 0; start >= 0 && u0 <= t; u0 += kWave) {
    uint64_t rows = __ballot(u0 + lane <= t && a.v_bad[(size_t)min(u0 + lane, t) * a.kvh + j] != 0);
    for (; rows; rows &= rows - 1) {
      const size_t at = ((size_t)(u0 + __builtin_ctzll(rows)) * a.kvh + j) * hd + lane * 4;
      const float4 q4 = *reinterpret_cast<const float4*>(a.q_rot + (size_t)row * hd + lane * 4);
      const float4 k4 = *reinterpret_cast<const float4*>(a.k_rot + at), v4 = *reinterpret_cast<const float4*>(a.v + at);
      const float p = __expf(wave_sum((q4.x * k4.x + q4.y * k4.y) + (q4.z * k4.z + q4.w * k4.w)) - M);
      o.x += fabsf(v4.x) < INFINITY ? 0.f : p * v4.x;
      o.y += fabsf(v4.y) < INFINITY ? 0.f : p * v4.y;
      o.z += fabsf(v4.z) < INFINITY ? 0.f : p * v4.z;
      o.w += fabsf(v4.w) < INFINITY ? 0.f : p * v4.w;
    }
  }
  const float4 gate = *reinterpret_cast<const float4*>(a.qg + (size_t)row * 2 * hd + hd + lane * 4);
  const float y[4] = {poison_if(start < 0, (o.x / L) * sigmoid(gate.x)), poison_if(start < 0, (o.y / L) * sigmoid(gate.y)),
                      poison_if(start < 0, (o.z / L) * sigmoid(gate.z)), poison_if(start < 0, (o.w / L) * sigmoid(gate.w))};
  const size_t plane = (size_t)a.T * a.heads * hd, i = (size_t)row * hd + lane * 4;
  uint32_t w[3][2];
#pragma unroll
  for (int q = 0; q < 2; ++q) split3_2(y[2 * q], y[2 * q + 1], w[0][q], w[1][q], w[2][q]);
#pragma unroll
  for (int q = 0; q < 3; ++q) *reinterpret_cast<uint2*>(a.planes + q * plane + i) = make_uint2(w[q][0], w[q][1]);
}

// The device-held position past the call's rows (every kernel of the call has
// read it).
__global__ void attn_prompt_advance_kernel(int* start, int T, int max_pos) {
  const int s = *start;
  if (positions_in_cache(s, T, max_pos)) *start = s + T;
}

struct PromptWs {
  float *qg, *k, *v, *q_rot, *k_rot, *stat, *acc, *part;
  int* v_bad;
  uint16_t* planes;
  size_t part_bytes;
};

static int prompt_max_chunks(int T, int heads, int kvh) {
  const long long ntb = ((long long)T * (heads / kvh) + kPromptRows - 1) / kPromptRows;
  const long long nc = kPromptWgs / (ntb * kvh);
  return nc < 1 ? 1 : nc > kPromptMaxChunks ? kPromptMaxChunks : (int)nc;
}

static size_t prompt_ws_layout(int T, int heads, int kvh, char* base, PromptWs* ws) {
  size_t off = 0;
  auto take = [&](size_t bytes) {
    const size_t at = off;
    off = align_up(off + bytes, 256);
    return base ? base + at : nullptr;
  };
  auto floats = [&](size_t n) { return reinterpret_cast<float*>(take(n * 4)); };
  const size_t q = (size_t)T * heads * kPromptHd, kv = (size_t)T * kvh * kPromptHd;
  // rows of chunk partials: at most kPromptWgs * kPromptRows from two chunks on,
  // whatever T (as a bound that never falls, so that a size that is enough for
  // T rows is enough for fewer)
  const size_t th = (size_t)T * heads, most = (size_t)kPromptWgs * kPromptRows;
  const size_t parts = th > most ? th : th * kPromptMaxChunks < most ? th * kPromptMaxChunks : most;
  ws->qg = floats(2 * q);
  ws->k = floats(kv);
  ws->v = floats(kv);
  ws->q_rot = floats(q);
  ws->k_rot = floats(kv);
  ws->v_bad = reinterpret_cast<int*>(take((size_t)T * kvh * 4));
  ws->stat = floats(parts * 2);
  ws->acc = floats(parts * kPromptHd);
  ws->planes = reinterpret_cast<uint16_t*>(take(q * 6));
  ws->part_bytes = token_part_bytes(T);
  ws->part = reinterpret_cast<float*>(take(token_part_reserve(T)));
  return off;
}

bool attn_prompt_ok(int T, int hidden, int heads, int kvh, int hd, int weight_dt, int norm_dt) {
  if (T < 1 || hd != kPromptHd || heads < 1 || kvh < 1 || heads % kvh) return false;
  const int G = heads / kvh;
  if (G > 8 || (G & (G - 1)) || kvh > 64 || heads > 4096 / hd) return false;
  const int rows[4] = {2 * heads * hd, kvh * hd, kvh * hd, 0};
  return norm_gemm_ok(rows, hidden, weight_dt, norm_dt) && plane_gemm_ok(hidden, heads * hd, weight_dt);
}

size_t attn_prompt_ws_bytes(int T, int heads, int kvh) {
  PromptWs ws;
  return prompt_ws_layout(T, heads, kvh, nullptr, &ws);
}

int launch_attn_prompt(const AttnPromptCall& p, void* workspace, hipStream_t s) {
  PromptWs ws;
  prompt_ws_layout(p.T, p.heads, p.kvh, reinterpret_cast<char*>(workspace), &ws);
  const void* const w[4] = {p.wq, p.wk, p.wv, nullptr};
  const int rows[4] = {2 * p.heads * kPromptHd, p.kvh * kPromptHd, p.kvh * kPromptHd, 0};
  float* const out[4] = {ws.qg, ws.k, ws.v, nullptr};
  int st = launch_norm_gemm(p.x, p.x_dt, p.nw, w, rows, out, p.T, p.hidden, p.eps, 1.0f, s);
  if (st) return st;
  PromptArgs a = {};
  a.qg = ws.qg;
  a.k = ws.k;
  a.v = ws.v;
  a.qn_w = p.qn_w;
  a.kn_w = p.kn_w;
  a.qn_dt = a.kn_dt = p.qk_dt;
  a.kc = p.kc;
  a.vc = p.vc;
  a.start_dev = p.start_dev;
  a.start = p.start;
  a.max_pos = p.max_pos;
  a.T = p.T;
  a.heads = p.heads;
  a.kvh = p.kvh;
  a.rope_dim = p.rope_dim;
  a.interleaved = p.interleaved;
  a.theta_log2 = log2f(p.theta);
  a.eps = p.qk_eps;
  a.q_rot = ws.q_rot;
  a.k_rot = ws.k_rot;
  a.v_bad = ws.v_bad;
  a.stat = ws.stat;
  a.acc = ws.acc;
  a.planes = ws.planes;
  a.err = p.err;
  a.ntb = (p.T * (p.heads / p.kvh) + kPromptRows - 1) / kPromptRows;
  // chunks of at least two tiles over the positions the call can reach (the
  // cache length when the position is known on the device only)
  const int reach = p.start_dev ? p.max_pos : p.start + p.T;
  int nc = prompt_max_chunks(p.T, p.heads, p.kvh);
  a.chunk = (reach + nc - 1) / nc;
  if (a.chunk < 2 * kPromptTile) a.chunk = 2 * kPromptTile;
  a.chunk = (a.chunk + kPromptTile - 1) / kPromptTile * kPromptTile;
  a.nc = (reach + a.chunk - 1) / a.chunk;
  const bool cbf = p.cache_dt == FK_DTYPE_BF16;
  const dim3 pgrid((unsigned)(((size_t)p.T * (p.heads + p.kvh) + 3) / 4));
  if (cbf) hipLaunchKernelGGL(attn_prompt_prep_kernel<true>, pgrid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL(attn_prompt_prep_kernel<false>, pgrid, dim3(256), 0, s, a);
  st = check_launch("attn_prompt_prep_kernel");
  if (st) return st;
  const dim3 grid((unsigned)((a.nc * a.kvh + 7) / 8 * 8 * a.ntb));
  if (cbf) hipLaunchKernelGGL(attn_prompt_kernel<true>, grid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL(attn_prompt_kernel<false>, grid, dim3(256), 0, s, a);
  st = check_launch("attn_prompt_kernel");
  if (st) return st;
  hipLaunchKernelGGL(attn_prompt_merge_kernel, dim3((unsigned)(((size_t)p.T * p.heads + 3) / 4)), dim3(256), 0, s, a);
  st = check_launch("attn_prompt_merge_kernel");
  if (st) return st;
  st = launch_plane_gemm(ws.planes, p.wo, p.hidden, p.T, p.heads * kPromptHd, p.hidden_out ? p.x : nullptr, p.x_dt,
                         p.update, p.hidden_out, ws.part, ws.part_bytes, s);
  if (st || !p.start_dev) return st;
  hipLaunchKernelGGL(attn_prompt_advance_kernel, dim3(1), dim3(1), 0, s, const_cast<int*>(p.start_dev), p.T, p.max_pos);
  return check_launch("attn_prompt_advance_kernel");
}

}  // namespace fk
