// Row RMS norm and the one-token attention step of the packed Pollux decoder
// (pollux.py:566-626 evaluated for one new position per sequence).
//
// rmsnorm_kernel: y = x * rsqrt(mean(x^2) + eps) * w over rows of d fp32
//   values (RMSNorm.forward, pollux.py:580-582); one wave per row, float4
//   loads (all of a row's issued at once up to 2,048 values), the sum of
//   squares reduced across the wave with shuffles.
//
// decode_attention_kernel: one block per (sequence, head).  For the new token
//   it RMS-normalises q and k over the head's 24 values (q_ln / k_ln,
//   pollux.py:615-620), writes k and v into the caches at the position read
//   from device memory, then computes softmax_j<=pos(q . K_j / sqrt 24) V_j
//   over the cached positions (the causal scaled_dot_product_attention of
//   pollux.py:624 for the last query): an online softmax per group of four
//   lanes over its positions, combined across the block at the end.
//   Reading the position from device memory lets a captured graph replay the
//   step while the position advances on the device; a position outside the
//   cache writes nothing and yields NaN outputs.
//
// prefill_attention_kernel: the same for t new positions p .. p+t-1 of every
//   sequence (the prompt of a prefill, pollux.py:615-626 with is_causal over
//   the cached prefix) on fp32 MFMA, in one launch: a block takes 64 queries of
//   one (head, sequence) and walks the keys up to its last query 64 at a time.

#include "plx_device.h"

namespace plx {
namespace {

constexpr int kNormRowsPerBlock = 4;  // one wave per row
constexpr int kNormRegVec = 8;        // float4 per lane held in registers (rows of <= 2,048 values)
constexpr int kAttnThreads = 256;
constexpr int kArgThreads = 1024;
constexpr int kArgRegs = 16;  // float4 per thread held in registers (rows of <= 65,536 values)

__device__ __forceinline__ float wave_sum(float v) { return wave_reduce_sum(v); }

// REG: rows of up to kNormRegVec float4 per lane (d <= 2,048) are held in
// registers, so every load of the row is in flight before the reduction (a
// loop of dependent trips through memory costs ~1 us per trip at one row).
template <bool REG>
__global__ __launch_bounds__(64 * kNormRowsPerBlock) void rmsnorm_kernel(const float *__restrict__ x,
                                                                        const float *__restrict__ w,
                                                                        float *__restrict__ y, int64_t rows, int d,
                                                                        float eps) {
  const int lane = threadIdx.x & 63;
  const int64_t row = static_cast<int64_t>(blockIdx.x) * kNormRowsPerBlock + (threadIdx.x >> 6);
  if (row >= rows) return;
  const float4 *xr = reinterpret_cast<const float4 *>(x + row * d);
  const float4 *wr = reinterpret_cast<const float4 *>(w);
  float4 *yr = reinterpret_cast<float4 *>(y + row * d);
  const int n4 = d >> 2;
  float ss = 0.f;
  if constexpr (REG) {
    float4 v[kNormRegVec], g[kNormRegVec];
#pragma unroll
    for (int k = 0; k < kNormRegVec; ++k) {
      const int i = lane + 64 * k;
      v[k] = i < n4 ? xr[i] : make_float4(0.f, 0.f, 0.f, 0.f);
      g[k] = i < n4 ? wr[i] : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int k = 0; k < kNormRegVec; ++k) {
      ss = fmaf(v[k].x, v[k].x, ss);
      ss = fmaf(v[k].y, v[k].y, ss);
      ss = fmaf(v[k].z, v[k].z, ss);
      ss = fmaf(v[k].w, v[k].w, ss);
    }
    ss = wave_sum(ss);
    const float r = 1.0f / sqrtf(ss / static_cast<float>(d) + eps);
#pragma unroll
    for (int k = 0; k < kNormRegVec; ++k) {
      const int i = lane + 64 * k;
      if (i < n4)
        yr[i] = make_float4(v[k].x * r * g[k].x, v[k].y * r * g[k].y, v[k].z * r * g[k].z, v[k].w * r * g[k].w);
    }
  } else {
    for (int i = lane; i < n4; i += 64) {
      const float4 v = xr[i];
      ss = fmaf(v.x, v.x, ss);
      ss = fmaf(v.y, v.y, ss);
      ss = fmaf(v.z, v.z, ss);
      ss = fmaf(v.w, v.w, ss);
    }
    ss = wave_sum(ss);
    const float r = 1.0f / sqrtf(ss / static_cast<float>(d) + eps);
    for (int i = lane; i < n4; i += 64) {
      const float4 v = xr[i], g = wr[i];
      yr[i] = make_float4(v.x * r * g.x, v.y * r * g.y, v.z * r * g.z, v.w * r * g.w);
    }
  }
}

// q, k, v: [b, H, 24] projections of the new token; caches [b, H, max_len, 24];
// out [b, H, 24].  Four lanes share a position: lane l of wave w holds dims
// 6(l & 3) .. +6 of the K and V rows of positions 64r + 16w + (l >> 2),
// r = 0, 1, ..., so one wave load covers 16 consecutive rows (1.5 KB) where a
// row per lane touched 64 cache lines per instruction.  Each group of four
// runs an online softmax over its positions (the score: its partial dot
// products summed over the four lanes, the same bits in each); the groups
// combine within the wave by DPP / shuffles over lanes of equal dims, the
// waves through LDS.  The positions' K / V rows are loaded kAttnRounds rounds
// of 64 at a time, from clamped addresses (no branch holds a load); round 0
// before the position is read (rows clamped to the cache), so those loads
// and the position's are in flight together.  The new position's normalised
// k and its v stand in for its (not yet written) cache rows.  3 rounds per
// trip (90 VGPRs; 5 waves per SIMD: 16 sequences x 80 heads are resident at
// once) measured 1% faster than 4 at batch 16 and 0.3% at batch 1.
constexpr int kAttnRounds = 3;
__global__ __launch_bounds__(kAttnThreads, 5) void decode_attention_kernel(
    const float *__restrict__ q, const float *__restrict__ k, const float *__restrict__ v, int64_t heads,
    int64_t in_stride, const float *__restrict__ q_w, const float *__restrict__ k_w, float eps,
    float *__restrict__ k_cache, float *__restrict__ v_cache, const int64_t *__restrict__ pos_ptr, int64_t max_len,
    float scale, float *__restrict__ out) {
  constexpr int kSub = kDim / 4;  // dims per lane
  __shared__ float red[kAttnThreads / 64][kDim + 2];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int d0 = (lane & 3) * kSub;
  const int grp = wave * 16 + (lane >> 2);  // position within a round of 64
  const int64_t bh = blockIdx.x;            // sequence * H + head
  float *kc = k_cache + bh * max_len * kDim + d0;
  float *vc = v_cache + bh * max_len * kDim + d0;
  float kr[kAttnRounds][kSub], vr[kAttnRounds][kSub];
  auto load_row = [&](int r, int64_t j) {
    const float2 *a = reinterpret_cast<const float2 *>(kc + j * kDim);
    const float2 *b = reinterpret_cast<const float2 *>(vc + j * kDim);
#pragma unroll
    for (int i = 0; i < kSub / 2; ++i) {
      const float2 x = a[i], y = b[i];
      kr[r][2 * i] = x.x; kr[r][2 * i + 1] = x.y;
      vr[r][2 * i] = y.x; vr[r][2 * i + 1] = y.y;
    }
  };
  load_row(0, grp < max_len ? grp : max_len - 1);
  // q, k, v rows of `heads` heads, in_stride floats apart per sequence
  const int64_t in = (bh / heads) * in_stride + (bh % heads) * kDim + d0;
  float qv[kSub], kv[kSub], vn[kSub], qw[kSub], kw[kSub];
#pragma unroll
  for (int i = 0; i < kSub / 2; ++i) {
    const float2 a = reinterpret_cast<const float2 *>(q + in)[i], b = reinterpret_cast<const float2 *>(k + in)[i];
    const float2 c = reinterpret_cast<const float2 *>(v + in)[i];
    const float2 e = reinterpret_cast<const float2 *>(q_w + d0)[i], f = reinterpret_cast<const float2 *>(k_w + d0)[i];
    qv[2 * i] = a.x; qv[2 * i + 1] = a.y; kv[2 * i] = b.x; kv[2 * i + 1] = b.y;
    vn[2 * i] = c.x; vn[2 * i + 1] = c.y; qw[2 * i] = e.x; qw[2 * i + 1] = e.y;
    kw[2 * i] = f.x; kw[2 * i + 1] = f.y;
  }
  const int64_t pos = *pos_ptr;
  if (pos < 0 || pos >= max_len) {  // the caller's position is outside the cache: write nothing
    if (tid < kDim) out[bh * kDim + tid] = __builtin_nanf("");
    return;
  }
#pragma unroll
  for (int r = 1; r < kAttnRounds; ++r) {
    const int64_t j = 64 * r + grp;
    load_row(r, j < pos ? j : pos);
  }

  // per-head RMS norms of q and k: 6 squares per lane, summed over the four lanes
  float sq[2] = {0.f, 0.f};
#pragma unroll
  for (int i = 0; i < kSub; ++i) {
    sq[0] = fmaf(qv[i], qv[i], sq[0]);
    sq[1] = fmaf(kv[i], kv[i], sq[1]);
  }
#pragma unroll
  for (int u = 0; u < 2; ++u) sq[u] += dpp_f32<0xB1>(sq[u]);
#pragma unroll
  for (int u = 0; u < 2; ++u) sq[u] += dpp_f32<0x4E>(sq[u]);
  const float rq = 1.0f / sqrtf(sq[0] / static_cast<float>(kDim) + eps);
  const float rk = 1.0f / sqrtf(sq[1] / static_cast<float>(kDim) + eps);
  float qn[kSub], kn[kSub];
#pragma unroll
  for (int i = 0; i < kSub; ++i) {
    qn[i] = qv[i] * rq * qw[i];
    kn[i] = kv[i] * rk * kw[i];
  }
  if (tid < 4) {  // the new row into the caches
#pragma unroll
    for (int i = 0; i < kSub / 2; ++i) {
      reinterpret_cast<float2 *>(kc + pos * kDim)[i] = make_float2(kn[2 * i], kn[2 * i + 1]);
      reinterpret_cast<float2 *>(vc + pos * kDim)[i] = make_float2(vn[2 * i], vn[2 * i + 1]);
    }
  }

  float m = -INFINITY, l = 0.f, acc[kSub];
#pragma unroll
  for (int i = 0; i < kSub; ++i) acc[i] = 0.f;
  // online softmax step of this group with key row kk and value row vv (all four lanes take it)
  auto step = [&](const float *kk, const float *vv) {
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < kSub; ++i) s = fmaf(qn[i], kk[i], s);
    s += dpp_f32<0xB1>(s);
    s += dpp_f32<0x4E>(s);
    s *= scale;
    const float mn = fmaxf(m, s);
    const float a = expf(m - mn), p = expf(s - mn);  // m = -inf at the first step: a = 0
    l = fmaf(l, a, p);
#pragma unroll
    for (int i = 0; i < kSub; ++i) acc[i] = fmaf(acc[i], a, p * vv[i]);
    m = mn;
  };
  const int64_t n_rounds = pos / 64 + 1;  // positions 0 .. pos
  for (int64_t r0 = 0; r0 < n_rounds; r0 += kAttnRounds) {
    if (r0 > 0) {
#pragma unroll
      for (int r = 0; r < kAttnRounds; ++r) {
        const int64_t j = 64 * (r0 + r) + grp;
        load_row(r, j < pos ? j : pos);
      }
    }
#pragma unroll
    for (int r = 0; r < kAttnRounds; ++r) {
      if (r0 + r >= n_rounds) break;
      const int64_t j = 64 * (r0 + r) + grp;
      if (j < pos) {
        step(kr[r], vr[r]);
      } else if (j == pos) {
        step(kn, vn);
      }
    }
  }

  // the wave's maximum, every group's state rescaled to it and summed over the
  // groups (lanes of equal dims: DPP row rotations by 4 and 8, then shuffles)
  float bmv[1] = {m};
  group_reduce<64, true>(bmv);
  const float bm = bmv[0];
  const float f = m == -INFINITY ? 0.f : expf(m - bm);
  float part[kSub + 1];
#pragma unroll
  for (int i = 0; i < kSub; ++i) part[i] = acc[i] * f;
  part[kSub] = l * f;
#pragma unroll
  for (int i = 0; i <= kSub; ++i) part[i] += dpp_f32<0x124>(part[i]);
#pragma unroll
  for (int i = 0; i <= kSub; ++i) part[i] += dpp_f32<0x128>(part[i]);
#pragma unroll
  for (int i = 0; i <= kSub; ++i) part[i] += __shfl_xor(part[i], 16, 64);
#pragma unroll
  for (int i = 0; i <= kSub; ++i) part[i] += __shfl_xor(part[i], 32, 64);
  if (lane < 4) {
#pragma unroll
    for (int i = 0; i < kSub; ++i) red[wave][d0 + i] = part[i];
    if (lane == 0) {
      red[wave][kDim] = part[kSub];
      red[wave][kDim + 1] = bm;
    }
  }
  __syncthreads();
  if (tid < kDim) {
    float gm = red[0][kDim + 1];
#pragma unroll
    for (int w = 1; w < kAttnThreads / 64; ++w) gm = fmaxf(gm, red[w][kDim + 1]);
    float sacc = 0.f, sl = 0.f;
#pragma unroll
    for (int w = 0; w < kAttnThreads / 64; ++w) {
      const float mw = red[w][kDim + 1];
      const float g = mw == -INFINITY ? 0.f : expf(mw - gm);
      sacc = fmaf(red[w][tid], g, sacc);
      sl = fmaf(red[w][kDim], g, sl);
    }
    out[bh * kDim + tid] = sacc / sl;
  }
}

// q, k, v, out: [b, t, H, 24] (rows of the prompt, at cache positions p0 .. p0+t-1); caches
// [b, H, max_len, 24].  One block of 4 waves per 64 queries (16 a wave) of one (head, sequence), the blocks
// with the most keys first.  Keys come in tiles of 64: the cached prefix from the caches, the prompt's from
// k and v, their norm (k_ln) taken here by every block that needs them (4 lanes a key; a few percent of the
// tile's products), so no block waits for another; the block whose queries are the tile's positions writes
// its rows into the caches.
//   Contractions: v_mfma_f32_16x16x4_f32, fp32 throughout.  S^T = K Q^T per 16 keys: lane l holds query l % 16
// and keys 4 (l / 16) + r, r = 0..3; the contraction index is dim 6 g + c for lane group g and step c, so a
// lane reads its 6 dims of a key as 3 8-byte pieces.  P^T is then, register r, the B operand of a step over
// keys 4 g + r without any exchange between lanes; its A operand is V^T from LDS (one 16-byte read per lane
// for 4 steps), in two tiles of dims (0-15; 16-23, then a row of ones that sums the probabilities).
// Online softmax per query: the maximum over the tile's 64 keys, exchanged between the four lanes of a query
// once per tile; the accumulators are rescaled only in tiles where some maximum of the wave rose.  The maximum is
// taken off before the scale: a rounded product of it would be common to a tile's keys, and beside scores of 2^31 (norm
// weights of 1e4 and more) larger than the exponents that 2^x has.
//   Error: scores in two chains of three MFMAs, a tile's sums from zero and then added: 1.9e-7 from float64 at 1,024
// positions (one chain through the running sums 3.4e-7; the VALU form 1.9e-7).
//   A V row that is not finite must not reach the queries before it (0 * inf): the tile that holds both
// (the block's own) then adds its keys one by one, each to the queries at or after it.
//   What bounds it: the chain within a tile (barrier, LDS, dependent MFMAs, exchanges, exponentials), which four waves
// per SIMD do not cover.  Counters at 1,024 tokens x 80 heads: matrix cores 24% busy (56 MFMAs of 32 cycles per 16
// queries x 64 keys; 25% of the second dims tile is padding), VALU issue 18%, bank conflicts 4%.  There 889 -> 119 us
// against a thread row of 16 lanes per query on the VALU in four launches of 256 positions.
constexpr int kPfTile = 64;               // queries per block, keys per tile
constexpr int kPfK = 26;                  // floats between keys in LDS (K)
constexpr int kPfV = 68;                  // floats between dims in LDS (V^T)
typedef float f32x4 __attribute__((ext_vector_type(4)));

__global__ __launch_bounds__(kAttnThreads, 4) void prefill_attention_kernel(
    const float *__restrict__ q, const float *__restrict__ k, const float *__restrict__ v,
    const float *__restrict__ q_w, const float *__restrict__ k_w, float eps, float *__restrict__ k_cache,
    float *__restrict__ v_cache, int64_t heads, int64_t in_stride, int t_total, int p0, int64_t max_len,
    float scale_log2, float *__restrict__ out) {
  constexpr int kSub = kDim / 4;  // dims per lane
  __shared__ __align__(16) float ks[2][kPfTile * kPfK];
  __shared__ __align__(16) float vt[2][(kDim + 1) * kPfV];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, n = lane & 15, g = lane >> 4;
  const int64_t bh = blockIdx.y;  // sequence * heads + head
  const int64_t bb = bh / heads, h = bh % heads;
  const int qt = static_cast<int>(gridDim.x - 1 - blockIdx.x);  // query tile: the longest first
  const float *kin = k + bb * t_total * in_stride + h * kDim, *vin = v + bb * t_total * in_stride + h * kDim;
  float *kc = k_cache + bh * max_len * kDim, *vc = v_cache + bh * max_len * kDim;
  const int n_pre = (p0 + kPfTile - 1) / kPfTile;  // tiles of the cached prefix
  const int n_tiles = n_pre + qt + 1;

  // a tile's rows: 4 lanes a key, 6 dims each; rows past the prefix / the prompt: zeros
  const int key = tid >> 2, d0 = (tid & 3) * kSub;
  float kr[kSub], vr[kSub];
  auto load = [&](int tile) {
    const bool pre = tile < n_pre;
    const int r = (pre ? tile : tile - n_pre) * kPfTile + key, lim = pre ? p0 : t_total;
    const int64_t rc = r < lim ? r : lim - 1;
    const float2 *a = reinterpret_cast<const float2 *>((pre ? kc + rc * kDim : kin + rc * in_stride) + d0);
    const float2 *b = reinterpret_cast<const float2 *>((pre ? vc + rc * kDim : vin + rc * in_stride) + d0);
#pragma unroll
    for (int i = 0; i < kSub / 2; ++i) {
      const float2 x = a[i], y = b[i];
      kr[2 * i] = x.x; kr[2 * i + 1] = x.y;
      vr[2 * i] = y.x; vr[2 * i + 1] = y.y;
    }
  };
  // the loaded rows into LDS (the prompt's keys normalised; the block's own also into the caches); returns
  // whether this thread's part of V is finite
  float kw[kSub];
#pragma unroll
  for (int i = 0; i < kSub; ++i) kw[i] = k_w[d0 + i];
  auto store = [&](int tile, int buf) {
    const bool pre = tile < n_pre;
    const int r = (pre ? tile : tile - n_pre) * kPfTile + key;
    const bool valid = r < (pre ? p0 : t_total);
    if (!pre) {
      float sq = 0.f;
#pragma unroll
      for (int i = 0; i < kSub; ++i) sq = fmaf(kr[i], kr[i], sq);
      sq += dpp_f32<0xB1>(sq);
      sq += dpp_f32<0x4E>(sq);
      const float rk = 1.0f / sqrtf(sq / static_cast<float>(kDim) + eps);
#pragma unroll
      for (int i = 0; i < kSub; ++i) kr[i] = kr[i] * rk * kw[i];
      if (tile == n_tiles - 1 && valid) {
#pragma unroll
        for (int i = 0; i < kSub / 2; ++i) {
          reinterpret_cast<float2 *>(kc + static_cast<int64_t>(p0 + r) * kDim + d0)[i] = make_float2(kr[2 * i], kr[2 * i + 1]);
          reinterpret_cast<float2 *>(vc + static_cast<int64_t>(p0 + r) * kDim + d0)[i] = make_float2(vr[2 * i], vr[2 * i + 1]);
        }
      }
    }
    bool finite = true;
#pragma unroll
    for (int i = 0; i < kSub; ++i) {
      if (!valid) kr[i] = vr[i] = 0.f;
      finite &= (__float_as_uint(vr[i]) & 0x7F800000u) != 0x7F800000u;
      vt[buf][(d0 + i) * kPfV + key] = vr[i];
    }
#pragma unroll
    for (int i = 0; i < kSub / 2; ++i)
      *reinterpret_cast<float2 *>(&ks[buf][key * kPfK + d0 + 2 * i]) = make_float2(kr[2 * i], kr[2 * i + 1]);
    return finite;
  };
  load(0);
  if (tid < 2 * kPfTile) vt[tid >> 6][kDim * kPfV + (tid & 63)] = 1.f;  // the probabilities' sum

  // this wave's 16 queries: lane (n, g) holds dims 6g .. 6g+5 of query n, normalised (q_ln)
  const int qrow = qt * kPfTile + wave * 16 + n;
  float qv[kSub];
  {
    const int64_t rc = qrow < t_total ? qrow : t_total - 1;
    const float2 *a = reinterpret_cast<const float2 *>(q + (bb * t_total + rc) * in_stride + h * kDim + g * kSub);
    float sq = 0.f;
#pragma unroll
    for (int i = 0; i < kSub / 2; ++i) {
      const float2 x = a[i];
      qv[2 * i] = x.x; qv[2 * i + 1] = x.y;
      sq = fmaf(x.y, x.y, fmaf(x.x, x.x, sq));
    }
    sq += __shfl_xor(sq, 16, 64);
    sq += __shfl_xor(sq, 32, 64);
    const float rq = 1.0f / sqrtf(sq / static_cast<float>(kDim) + eps);
#pragma unroll
    for (int i = 0; i < kSub; ++i) qv[i] = qv[i] * rq * q_w[g * kSub + i];
  }

  f32x4 o0 = {0.f, 0.f, 0.f, 0.f}, o1 = {0.f, 0.f, 0.f, 0.f};  // dims 4g + r; 16 + 4g + r (24: the sum)
  float m = -INFINITY;
  const int vrow0 = n * kPfV + 4 * g, vrow1 = min(16 + n, kDim) * kPfV + 4 * g;
  bool finite = store(0, 0);
  for (int tile = 0; tile < n_tiles; ++tile) {
    const int buf = tile & 1;
    const bool own = tile == n_tiles - 1;
    const bool all_finite = __syncthreads_and(finite) != 0;  // (tile's rows are in LDS; the other buffer is free)
    if (!own) load(tile + 1);
    const int live = own ? wave + 1 : kPfTile / 16;  // 16-key parts with a key at or before some query of the wave
    f32x4 sc[4];
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) {
      sc[kt] = f32x4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
      if (kt >= live) continue;  // (wave-uniform)
      const float2 *a = reinterpret_cast<const float2 *>(&ks[buf][(16 * kt + n) * kPfK + g * kSub]);
      f32x4 c = {0.f, 0.f, 0.f, 0.f}, d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < kSub / 2; ++i) {
        const float2 x = a[i];
        c = __builtin_amdgcn_mfma_f32_16x16x4f32(x.x, qv[2 * i], c, 0, 0, 0);
        d = __builtin_amdgcn_mfma_f32_16x16x4f32(x.y, qv[2 * i + 1], d, 0, 0, 0);
      }
      sc[kt] = c + d;
    }
    // keys past the query (own tile) or past the prefix (its last tile)
    if (own || tile == n_pre - 1) {
      const int last = own ? wave * 16 + n : p0 - 1 - tile * kPfTile;
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (16 * kt + 4 * g + r > last) sc[kt][r] = -INFINITY;
    }
    float mx = sc[0][0];
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
      for (int r = 0; r < 4; ++r) mx = fmaxf(mx, sc[kt][r]);
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    if (__any(mx > m)) {
      const float mn = fmaxf(m, mx);
      const float f = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m - mn) * scale_log2);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        o0[r] *= f;
        o1[r] *= f;
      }
      m = mn;
    }
    // the tile's sums from zero, added to the running ones on the VALU: one rounding of those per tile
    f32x4 t0 = {0.f, 0.f, 0.f, 0.f}, t1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) {
      if (kt >= live) continue;  // (wave-uniform)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        sc[kt][r] = __builtin_amdgcn_exp2f((sc[kt][r] - m) * scale_log2);  // (a masked key: 2^-inf = 0)
      if (!own || all_finite) {
        const float4 a = *reinterpret_cast<const float4 *>(&vt[buf][vrow0 + 16 * kt]);
        const float4 b = *reinterpret_cast<const float4 *>(&vt[buf][vrow1 + 16 * kt]);
        t0 = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, sc[kt][0], t0, 0, 0, 0);
        t1 = __builtin_amdgcn_mfma_f32_16x16x4f32(b.x, sc[kt][0], t1, 0, 0, 0);
        t0 = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, sc[kt][1], t0, 0, 0, 0);
        t1 = __builtin_amdgcn_mfma_f32_16x16x4f32(b.y, sc[kt][1], t1, 0, 0, 0);
        t0 = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, sc[kt][2], t0, 0, 0, 0);
        t1 = __builtin_amdgcn_mfma_f32_16x16x4f32(b.z, sc[kt][2], t1, 0, 0, 0);
        t0 = __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, sc[kt][3], t0, 0, 0, 0);
        t1 = __builtin_amdgcn_mfma_f32_16x16x4f32(b.w, sc[kt][3], t1, 0, 0, 0);
      } else {
        float *ps = &ks[buf ^ 1][wave * 256];  // (the last tile: the other buffer is done with)
#pragma unroll
        for (int r = 0; r < 4; ++r) ps[(4 * g + r) * 16 + n] = sc[kt][r];
#pragma unroll 1
        for (int kk = 0; kk < 16; ++kk) {
          const float pr = ps[kk * 16 + n];
          if (16 * kt + kk > wave * 16 + n) continue;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            t0[e] = fmaf(pr, vt[buf][(4 * g + e) * kPfV + 16 * kt + kk], t0[e]);
            t1[e] = fmaf(pr, vt[buf][min(16 + 4 * g + e, kDim) * kPfV + 16 * kt + kk], t1[e]);
          }
        }
      }
    }
    o0 += t0;
    o1 += t1;
    if (!own) finite = store(tile + 1, buf ^ 1);
  }
  const float sum = __shfl(o1[0], 32 + n, 64);  // dim 24: lanes of g = 2, register 0
  if (qrow < t_total) {
    float *o = out + (bb * t_total + qrow) * heads * kDim + h * kDim + 4 * g;
    *reinterpret_cast<float4 *>(o) = make_float4(o0[0] / sum, o0[1] / sum, o0[2] / sum, o0[3] / sum);
    if (g < 2)
      *reinterpret_cast<float4 *>(o + 16) = make_float4(o1[0] / sum, o1[1] / sum, o1[2] / sum, o1[3] / sum);
  }
}

// torch.argmax's order: a NaN beats every number; among equal values (or
// NaNs) the lowest index wins.
__device__ __forceinline__ bool arg_better(float v, int i, float bv, int bi) {
  const bool vn = v != v, bn = bv != bv;
  if (vn || bn) return vn && (!bn || i < bi);
  return v > bv || (v == bv && i < bi);
}

// One block per row of cols values; each thread scans its strided share
// (increasing indices), then the block reduces (value, index) pairs.
template <bool VEC>
__global__ __launch_bounds__(kArgThreads) void argmax_rows_kernel(const float *__restrict__ x, int cols,
                                                                  int64_t *__restrict__ out) {
  __shared__ float sv[kArgThreads / 64];
  __shared__ int si[kArgThreads / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const float *r = x + static_cast<int64_t>(blockIdx.x) * cols;
  float bv = -INFINITY;
  int bi = cols;  // beyond every index: the first -inf wins when all are -inf
  if constexpr (VEC) {
    const float4 *r4 = reinterpret_cast<const float4 *>(r);
    const int n4 = cols / 4;
    auto take = [&](const float4 &v, int i) {
      if (arg_better(v.x, 4 * i, bv, bi)) { bv = v.x; bi = 4 * i; }
      if (arg_better(v.y, 4 * i + 1, bv, bi)) { bv = v.y; bi = 4 * i + 1; }
      if (arg_better(v.z, 4 * i + 2, bv, bi)) { bv = v.z; bi = 4 * i + 2; }
      if (arg_better(v.w, 4 * i + 3, bv, bi)) { bv = v.w; bi = 4 * i + 3; }
    };
    if (n4 <= kArgThreads * kArgRegs) {
      // the whole row in flight at once (clamped indices: no branch holds a load)
      float4 v[kArgRegs];
#pragma unroll
      for (int k = 0; k < kArgRegs; ++k) {
        const int i = tid + kArgThreads * k;
        v[k] = r4[i < n4 ? i : 0];
      }
#pragma unroll
      for (int k = 0; k < kArgRegs; ++k)
        if (tid + kArgThreads * k < n4) take(v[k], tid + kArgThreads * k);
    } else {
#pragma unroll 4
      for (int i = tid; i < n4; i += kArgThreads) take(r4[i], i);
    }
  } else {
#pragma unroll 4
    for (int i = tid; i < cols; i += kArgThreads) {
      const float v = r[i];
      if (arg_better(v, i, bv, bi)) { bv = v; bi = i; }
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const float ov = __shfl_xor(bv, off, 64);
    const int oi = __shfl_xor(bi, off, 64);
    if (arg_better(ov, oi, bv, bi)) { bv = ov; bi = oi; }
  }
  if (lane == 0) {
    sv[wave] = bv;
    si[wave] = bi;
  }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < kArgThreads / 64; ++w)
      if (arg_better(sv[w], si[w], bv, bi)) { bv = sv[w]; bi = si[w]; }
    out[blockIdx.x] = bi < cols ? bi : 0;
  }
}

}  // namespace

int launch_argmax_rows(const float *x, int64_t rows, int64_t cols, int64_t *out, hipStream_t s) {
  if (rows <= 0) return PLX_OK;
  if (cols <= 0 || cols > 0x7FFFFFFFll || rows > 0x7FFFFFFFll)
    return fail(PLX_EINVAL, "argmax_rows: shape (%lld, %lld)", static_cast<long long>(rows), static_cast<long long>(cols));
  const bool vec = cols % 4 == 0 && (reinterpret_cast<uintptr_t>(x) & 15u) == 0;
  if (vec)
    hipLaunchKernelGGL((argmax_rows_kernel<true>), dim3(static_cast<unsigned>(rows)), dim3(kArgThreads), 0, s, x,
                       static_cast<int>(cols), out);
  else
    hipLaunchKernelGGL((argmax_rows_kernel<false>), dim3(static_cast<unsigned>(rows)), dim3(kArgThreads), 0, s, x,
                       static_cast<int>(cols), out);
  return check_launch("argmax_rows_kernel");
}

int launch_rms_norm(const float *x, const float *w, float *y, int64_t rows, int64_t d, float eps, hipStream_t s) {
  if (rows <= 0) return PLX_OK;
  if (d <= 0 || d % 4 != 0 || d > (1 << 24))
    return fail(PLX_EINVAL, "rms_norm: row length %lld must be a positive multiple of 4", static_cast<long long>(d));
  const uintptr_t al = reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(y);
  if ((al & 15u) != 0) return fail(PLX_EINVAL, "rms_norm: x, w and y must be 16-byte aligned");
  const int64_t blocks = (rows + kNormRowsPerBlock - 1) / kNormRowsPerBlock;
  if (blocks > 0x7FFFFFFFll) return fail(PLX_EINVAL, "rms_norm: too many rows");
  if (d <= 64 * 4 * kNormRegVec)
    hipLaunchKernelGGL((rmsnorm_kernel<true>), dim3(static_cast<unsigned>(blocks)), dim3(64 * kNormRowsPerBlock), 0, s,
                       x, w, y, rows, static_cast<int>(d), eps);
  else
    hipLaunchKernelGGL((rmsnorm_kernel<false>), dim3(static_cast<unsigned>(blocks)), dim3(64 * kNormRowsPerBlock), 0, s,
                       x, w, y, rows, static_cast<int>(d), eps);
  return check_launch("rmsnorm_kernel");
}

int launch_decode_attention(const float *q, const float *k, const float *v, int64_t qkv_stride, int64_t heads,
                            const float *q_w, const float *k_w, float eps, float *k_cache, float *v_cache,
                            const int64_t *pos, int64_t seqs_heads, int64_t max_len, float *out, hipStream_t s) {
  if (seqs_heads <= 0) return PLX_OK;
  if (max_len <= 0 || max_len > (1 << 24))
    return fail(PLX_EINVAL, "decode_attention: cache length %lld outside 1..2^24", static_cast<long long>(max_len));
  if (seqs_heads > 0x7FFFFFFFll) return fail(PLX_EINVAL, "decode_attention: too many heads");
  const uintptr_t al = reinterpret_cast<uintptr_t>(k_cache) | reinterpret_cast<uintptr_t>(v_cache);
  if ((al & 15u) != 0) return fail(PLX_EINVAL, "decode_attention: caches must be 16-byte aligned");
  if (qkv_stride == 0) {  // contiguous [seqs_heads, 24]
    heads = 1;
    qkv_stride = kDim;
  }
  if (heads <= 0 || seqs_heads % heads != 0 || qkv_stride < heads * kDim)
    return fail(PLX_EINVAL, "decode_attention: rows of %lld heads %lld floats apart do not tile %lld head rows",
                static_cast<long long>(heads), static_cast<long long>(qkv_stride), static_cast<long long>(seqs_heads));
  // the kernel reads q, k, v and the norm weights as float2
  const uintptr_t al8 = reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) |
                        reinterpret_cast<uintptr_t>(v) | reinterpret_cast<uintptr_t>(q_w) |
                        reinterpret_cast<uintptr_t>(k_w);
  if ((al8 & 7u) != 0 || (qkv_stride & 1) != 0)
    return fail(PLX_EINVAL, "decode_attention: q, k, v and the norm weights must be 8-byte aligned, the row stride even");
  hipLaunchKernelGGL(decode_attention_kernel, dim3(static_cast<unsigned>(seqs_heads)), dim3(kAttnThreads), 0, s, q, k,
                     v, heads, qkv_stride, q_w, k_w, eps, k_cache, v_cache, pos, max_len,
                     1.0f / sqrtf(static_cast<float>(kDim)), out);
  return check_launch("decode_attention_kernel");
}

int launch_prefill_attention(const float *q, const float *k, const float *v, int64_t qkv_stride, const float *q_w,
                             const float *k_w, float eps, float *k_cache, float *v_cache, int64_t b, int64_t heads,
                             int64_t t, int64_t p0, int64_t max_len, float *out, hipStream_t s) {
  if (b <= 0 || heads <= 0 || t <= 0) return PLX_OK;
  if (max_len <= 0 || max_len > (1 << 24))
    return fail(PLX_EINVAL, "prefill_attention: cache length %lld outside 1..2^24", static_cast<long long>(max_len));
  if (p0 < 0 || p0 + t > max_len)
    return fail(PLX_EINVAL, "prefill_attention: positions %lld..%lld outside the cache of %lld", static_cast<long long>(p0),
                static_cast<long long>(p0 + t - 1), static_cast<long long>(max_len));
  if (heads > 0xFFFFll || b > 0xFFFFll) return fail(PLX_EINVAL, "prefill_attention: too many heads or sequences");
  const uintptr_t al = reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(v) |
                       reinterpret_cast<uintptr_t>(k_cache) | reinterpret_cast<uintptr_t>(v_cache) |
                       reinterpret_cast<uintptr_t>(out);
  if ((al & 15u) != 0) return fail(PLX_EINVAL, "prefill_attention: q, k, v, caches and out must be 16-byte aligned");
  if (qkv_stride == 0) qkv_stride = heads * kDim;  // contiguous rows
  if (qkv_stride < heads * kDim || qkv_stride % 4 != 0)
    return fail(PLX_EINVAL, "prefill_attention: q, k, v rows %lld floats apart (at least %lld, a multiple of 4)",
                static_cast<long long>(qkv_stride), static_cast<long long>(heads * kDim));
  const int64_t q_tiles = (t + kPfTile - 1) / kPfTile;
  // the softmax takes powers of two
  const float scale_log2 = static_cast<float>(1.4426950408889634 / sqrt(static_cast<double>(kDim)));
  // the grid's y dimension holds 65,535 (sequence, head) pairs: more go in several launches
  const int64_t seqs = 0xFFFFll / heads;
  for (int64_t s0 = 0; s0 < b; s0 += seqs) {
    const int64_t nb = b - s0 < seqs ? b - s0 : seqs;
    const int64_t in = s0 * t * qkv_stride, cache = s0 * heads * max_len * kDim;
    hipLaunchKernelGGL(prefill_attention_kernel, dim3(static_cast<unsigned>(q_tiles), static_cast<unsigned>(nb * heads)),
                       dim3(kAttnThreads), 0, s, q + in, k + in, v + in, q_w, k_w, eps, k_cache + cache, v_cache + cache,
                       heads, qkv_stride, static_cast<int>(t), static_cast<int>(p0), max_len, scale_log2, out + s0 * t * heads * kDim);
    const int st = check_launch("prefill_attention_kernel");
    if (st != PLX_OK) return st;
  }
  return PLX_OK;
}

}  // namespace plx
