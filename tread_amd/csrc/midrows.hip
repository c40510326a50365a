// Decoder layers for 3 to 128 token rows (a query, a follow-up turn, a short system prompt): every
// projection streams its weights once from HBM, so the layer is priced by the weights' bytes and by
// the launches between them. One call queues every kernel of every layer.
//
// y[M, N] = x[M, K] . W[N, K]^T is cut into units of 64 features x 128 K (16 KB of weights). The units
// are dealt in tile-major order to work groups of 4 waves, `upg` consecutive units each, so that
// every work group streams the same number of bytes whatever N and K are: a tile-per-group grid of a
// 3 584 x 18 944 projection has 56 tiles for 256 CUs, one of 37 888 x 3 584 a second round of 80.
// Weights and x rows go from global memory straight into LDS, NST stages deep (swizzled 16-byte
// chunks as in the attention kernel), and each wave multiplies 16 features by all rows with
// v_mfma_f32_16x16x32_bf16. A work group's fp32 sums of one tile are one partial: they go to slot
// (work group + tile) of the workspace, and the kernel that consumes the projection (RoPE + splice,
// residual add + RMSNorm, SiLU gating) adds a tile's partials in work group order, adds the bias and
// rounds once to bf16 itself, so the split costs no launch.
#include <mutex>

#include "common.h"
#include "../../include/tread_hip.h"
#include "lds.h"

namespace tread {

constexpr int MID_TN = 64;        // features per tile
constexpr int MID_BK = 128;       // K per unit
constexpr int MID_THREADS = 256;  // 4 waves of 16 features
constexpr int MID_CH = MID_BK / 8;
constexpr int MID_MAX_ROWS = 128;
constexpr int MID_MAX_HIDDEN = 16384;

// How a projection's units are dealt: work group g takes units [g upg, (g + 1) upg).
struct MidPlan {
  int tiles, ku;  // feature tiles, units per tile
  int upg, groups;
};

struct MidGemmArgs {
  const bf16_t* x;
  const bf16_t* w;
  float* part;  // [groups + tiles][M][MID_TN]
  int M, K;
  MidPlan p;
};

template <int MB>
struct MidStage {
  static constexpr int W_ELEMS = MID_TN * MID_BK;
  static constexpr int ELEMS = W_ELEMS + MB * 16 * MID_BK;
  static constexpr int LPT = 4 + MB;  // 16-byte loads per lane and stage
};

template <int MB, int NST>
__global__ __launch_bounds__(MID_THREADS) void mid_gemm_kernel(const MidGemmArgs a) {
  using ST = MidStage<MB>;
  constexpr int LPT = ST::LPT;
  extern __shared__ __align__(16) bf16_t smem[];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int l15 = lane & 15, kg = lane >> 4;
  const int u0 = blockIdx.x * a.p.upg, u1 = min(u0 + a.p.upg, a.p.tiles * a.p.ku);
  const int n = u1 - u0;

  // Load q of a stage fills the 64 chunk positions from (q * 4 + wave) * 64 on, lane l position + l:
  // row pos / 16, slot pos % 16, holding chunk slot ^ (row % 16) of that row, so that the 16 rows of a
  // fragment read (the same chunk of each) spread over every bank.
  int woff[4], xoff[MB];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int pos = (q * 4 + wv) * 64 + lane, row = pos / MID_CH;
    woff[q] = row * a.K + ((pos % MID_CH) ^ (row & 15)) * 8;
  }
#pragma unroll
  for (int q = 0; q < MB; ++q) {
    const int pos = (q * 4 + wv) * 64 + lane, row = pos / MID_CH;
    // rows past M repeat the last one: their products are never stored
    xoff[q] = min(row, a.M - 1) * a.K + ((pos % MID_CH) ^ (row & 15)) * 8;
  }
  int it = u0 / a.p.ku, ik = u0 % a.p.ku;  // tile and K unit of the next load
  auto issue = [&](int buf) {
    const bf16_t* wp = a.w + (int64_t)it * MID_TN * a.K + ik * MID_BK;
    const bf16_t* xp = a.x + ik * MID_BK;
    bf16_t* dst = smem + buf * ST::ELEMS;
#pragma unroll
    for (int q = 0; q < 4; ++q) lds_load16_nt(wp + woff[q], dst + (q * 4 + wv) * 64 * 8);
#pragma unroll
    for (int q = 0; q < MB; ++q) lds_load16(xp + xoff[q], dst + ST::W_ELEMS + (q * 4 + wv) * 64 * 8);
    if (++ik == a.p.ku) {
      ik = 0;
      ++it;
    }
  };
  // fragment addresses in stage 0, one per 32-K step: weight row wv * 16 + l % 16 (and, at fixed
  // offsets, x row l % 16 of each 16-row block), chunk step * 4 + lane / 16
  uint32_t addr[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) addr[s] = lds_addr(smem + l15 * MID_BK + (((s * 4 + kg) ^ l15) * 8));
  const uint32_t wrow = (uint32_t)(wv * 16 * MID_BK * 2);

  f32x4_t acc[MB];
#pragma unroll
  for (int b = 0; b < MB; ++b) acc[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < NST - 1; ++s)
    if (s < n) issue(s);
  int tile = u0 / a.p.ku, k = u0 % a.p.ku, buf = 0;
  for (int i = 0; i < n; ++i) {
    // this unit's loads landed (the later stages' may fly); vmcnt counts loads and stores in issue order
    if (i + NST - 1 <= n) vm_wait<LPT * (NST - 2)>();
    else vm_wait<0>();
    tile_barrier();
    if (i + NST - 1 < n) issue(buf == 0 ? NST - 1 : buf - 1);  // the buffer of unit i - 1, read by every wave
    const uint32_t so = (uint32_t)(buf * ST::ELEMS * 2);
    bf16x8_t wf[4], xf[4][MB];
    auto read = [&](auto S) {
      constexpr int s = decltype(S)::value;
      wf[s] = lds_read128<0>(addr[s] + so + wrow);
      static_for<MB>([&](auto B) {
        constexpr int b = decltype(B)::value;
        xf[s][b] = lds_read128<(ST::W_ELEMS + b * 16 * MID_BK) * 2>(addr[s] + so);
      });
    };
    // reads of AHEAD steps in flight (the wait counter holds 15)
    constexpr int AHEAD = 2 * (1 + MB) <= 15 ? 2 : 1;
    static_for<AHEAD>([&](auto S) { read(S); });
    static_for<4>([&](auto S) {
      constexpr int s = decltype(S)::value;
      if constexpr (s + AHEAD < 4) read(std::integral_constant<int, s + AHEAD>{});
      constexpr int after = (s + AHEAD < 4 ? AHEAD : 3 - s) * (1 + MB);
      lgkm_wait<after>(wf[s]);
#pragma unroll
      for (int b = 0; b < MB; ++b) {
        asm volatile("" : "+v"(xf[s][b]));  // waited for with wf[s]
        acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[s], xf[s][b], acc[b], 0, 0, 0);
      }
    });
    buf = buf == NST - 1 ? 0 : buf + 1;
    if (++k == a.p.ku || i + 1 == n) {
      // lane l: row b * 16 + l % 16, features wv * 16 + (l / 16) * 4 .. + 3
      float* pp = a.part + ((int64_t)(blockIdx.x + tile) * a.M + l15) * MID_TN + wv * 16 + kg * 4;
#pragma unroll
      for (int b = 0; b < MB; ++b) {
        if (b * 16 + l15 < a.M) *reinterpret_cast<f32x4_t*>(pp + b * 16 * MID_TN) = acc[b];
        acc[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
      k = 0;
      ++tile;
    }
  }
}

// What a consumer needs to add up a projection's partials.
struct MidSrc {
  const float* part;
  int M, ku, upg;
};

// fp32 sums of features n .. n + 7 (n a multiple of 8) of row m, in work group order.
__device__ __forceinline__ void mid_sum8(const MidSrc& s, int m, int n, float (&v)[8]) {
  const int t = n / MID_TN;
  const int g0 = t * s.ku / s.upg, g1 = ((t + 1) * s.ku - 1) / s.upg;
  const float* p = s.part + ((int64_t)(g0 + t) * s.M + m) * MID_TN + n % MID_TN;
  const int64_t st = (int64_t)s.M * MID_TN;
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = 0.f;
#pragma unroll 4
  for (int g = g0; g <= g1; ++g, p += st) {
    const f32x4_t a = *reinterpret_cast<const f32x4_t*>(p), b = *reinterpret_cast<const f32x4_t*>(p + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[e] += a[e];
      v[4 + e] += b[e];
    }
  }
}
__device__ __forceinline__ u32x4_t pack8(const float (&v)[8]) {
  return u32x4_t{pack_bf(v[0], v[1]), pack_bf(v[2], v[3]), pack_bf(v[4], v[5]), pack_bf(v[6], v[7])};
}

// s = h + d, d = delta (bf16) or the partials of `src` rounded to bf16 (or nothing); s to h_out, the
// row's RMSNorm to x_out, rounded as add_rmsnorm_row does. One work group per row.
constexpr int MID_NORM_THREADS = 512;
template <int CPT>
__global__ __launch_bounds__(MID_NORM_THREADS) void mid_norm_kernel(const bf16_t* h, const bf16_t* delta, MidSrc src,
                                                                    const bf16_t* __restrict__ w, float eps, int hidden,
                                                                    bf16_t* h_out, bf16_t* __restrict__ x_out) {
  __shared__ float red[MID_NORM_THREADS / 64];
  const int m = blockIdx.x, nch = hidden / 8;
  const int64_t row = (int64_t)m * hidden;
  u32x4_t v[CPT], ww[CPT];
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < CPT; ++j) {
    const int c = threadIdx.x + j * MID_NORM_THREADS;
    if (c >= nch) continue;
    ww[j] = *reinterpret_cast<const u32x4_t*>(w + c * 8);
    u32x4_t a = *reinterpret_cast<const u32x4_t*>(h + row + c * 8);
    if (src.part || delta) {
      u32x4_t d;
      if (src.part) {
        float f[8];
        mid_sum8(src, m, c * 8, f);
        d = pack8(f);
      } else {
        d = *reinterpret_cast<const u32x4_t*>(delta + row + c * 8);
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) a[q] = pack_bf(lo_bf(a[q]) + lo_bf(d[q]), hi_bf(a[q]) + hi_bf(d[q]));
    }
    *reinterpret_cast<u32x4_t*>(h_out + row + c * 8) = a;
    v[j] = a;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float l = lo_bf(a[q]), hh = hi_bf(a[q]);
      ss = fmaf(l, l, ss);
      ss = fmaf(hh, hh, ss);
    }
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) ss += __shfl_xor(ss, o);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
  __syncthreads();
  float t = 0.f;
#pragma unroll
  for (int q = 0; q < MID_NORM_THREADS / 64; ++q) t += red[q];
  const float r = 1.0f / sqrtf(t / (float)hidden + eps);
#pragma unroll
  for (int j = 0; j < CPT; ++j) {
    const int c = threadIdx.x + j * MID_NORM_THREADS;
    if (c >= nch) continue;
    u32x4_t o;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      o[q] = pack_bf(bf2f(f2bf(lo_bf(v[j][q]) * r)) * lo_bf(ww[j][q]), bf2f(f2bf(hi_bf(v[j][q]) * r)) * hi_bf(ww[j][q]));
    *reinterpret_cast<u32x4_t*>(x_out + row + c * 8) = o;
  }
}

// Partials (+ bias) rounded to bf16: y [M, N].
__global__ __launch_bounds__(256) void mid_reduce_kernel(MidSrc src, const bf16_t* __restrict__ bias, int N,
                                                         bf16_t* __restrict__ y) {
  const int t = blockIdx.x * 256 + threadIdx.x, per = N / 8;
  if (t >= src.M * per) return;
  const int m = t / per, n = (t % per) * 8;
  float v[8];
  mid_sum8(src, m, n, v);
  if (bias)
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] += bf2f(bias[n + e]);
  *reinterpret_cast<u32x4_t*>(y + (int64_t)m * N + n) = pack8(v);
}

// act [M, inter] = bf16(bf16(silu(g)) * u) from the gate|up projection's partials (silu_mul's roundings).
__global__ __launch_bounds__(256) void mid_swiglu_kernel(MidSrc src, int inter, bf16_t* __restrict__ act) {
  const int t = blockIdx.x * 256 + threadIdx.x, per = inter / 8;
  if (t >= src.M * per) return;
  const int m = t / per, n = (t % per) * 8;
  float g[8], u[8];
  mid_sum8(src, m, n, g);
  mid_sum8(src, m, inter + n, u);
#pragma unroll
  for (int e = 0; e < 8; ++e) g[e] = silu_bf16(bf2f(f2bf(g[e]))) * bf2f(f2bf(u[e]));
  *reinterpret_cast<u32x4_t*>(act + (int64_t)m * inter + n) = pack8(g);
}

// q|k|v partials (+ bias) -> rotated q, rotated k and v in the cache, with the rounding points of
// qkv_rope_splice_kernel. One thread per 8 pairs of a q or k head, or 8 elements of a v head.
__global__ __launch_bounds__(64) void mid_rope_kernel(MidSrc src, const bf16_t* __restrict__ bias,
                                                      const bf16_t* __restrict__ cosb, const bf16_t* __restrict__ sinb,
                                                      const int64_t* __restrict__ rows, int hq, int hkv, int hd,
                                                      bf16_t* __restrict__ q_out, bf16_t* __restrict__ kc,
                                                      bf16_t* __restrict__ vc, int64_t t_cap) {
  const int half = hd / 2, pg = half / 8, rot = (hq + hkv) * pg, per = rot + hkv * (hd / 8);
  const int t = blockIdx.x * 64 + threadIdx.x;
  if (t >= src.M * per) return;
  const int m = t / per, task = t % per;
  const int64_t row = rows[m];
  const bool row_ok = row >= 0 && row < t_cap;  // out-of-range rows splice nothing
  auto load = [&](int n, float (&v)[8]) {
    mid_sum8(src, m, n, v);
    if (bias)
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] += bf2f(bias[n + e]);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = bf2f(f2bf(v[e]));
  };
  float a[8], b[8];
  if (task >= rot) {
    const int vt = task - rot, h = vt / (hd / 8), c = (vt % (hd / 8)) * 8;
    if (!row_ok) return;
    load((hq + hkv + h) * hd + c, a);
    *reinterpret_cast<u32x4_t*>(vc + ((int64_t)h * t_cap + row) * hd + c) = pack8(a);
    return;
  }
  const int h = task / pg, c = (task % pg) * 8;
  bf16_t* dst;
  if (h < hq) {
    dst = q_out + ((int64_t)m * hq + h) * hd;
  } else {
    if (!row_ok) return;
    dst = kc + ((int64_t)(h - hq) * t_cap + row) * hd;
  }
  load(h * hd + c, a);
  load(h * hd + c + half, b);
  const u32x4_t cw = *reinterpret_cast<const u32x4_t*>(cosb + (int64_t)m * half + c);
  const u32x4_t sw = *reinterpret_cast<const u32x4_t*>(sinb + (int64_t)m * half + c);
  float o1[8], o2[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float co = e & 1 ? hi_bf(cw[e / 2]) : lo_bf(cw[e / 2]), si = e & 1 ? hi_bf(sw[e / 2]) : lo_bf(sw[e / 2]);
    o1[e] = bf2f(f2bf(a[e] * co)) + bf2f(f2bf(-b[e] * si));
    o2[e] = bf2f(f2bf(b[e] * co)) + bf2f(f2bf(a[e] * si));
  }
  *reinterpret_cast<u32x4_t*>(dst + c) = pack8(o1);
  *reinterpret_cast<u32x4_t*>(dst + c + half) = pack8(o2);
}

static bool mid_shape_ok(int64_t m, int64_t n, int64_t k) {
  return m > 0 && m <= MID_MAX_ROWS && n > 0 && k > 0 && n % MID_TN == 0 && k % MID_BK == 0 && n <= (1 << 24) &&
         k <= (1 << 20) && (n / MID_TN) * (k / MID_BK) <= (1 << 28);
}

// Pipeline stages by blocks of 16 rows, and (mid_plan) work groups per CU: what 160 KB of LDS holds.
constexpr int mid_stages(int mb) { return mb <= 2 ? 3 : mb <= 6 ? 4 : 3; }
static MidPlan mid_plan(int64_t m, int64_t n, int64_t k) {
  MidPlan p;
  p.tiles = (int)(n / MID_TN);
  p.ku = (int)(k / MID_BK);
  const int units = p.tiles * p.ku;
  const int most = cu_count() * (m <= 32 ? 2 : 1);
  p.upg = (units + most - 1) / most;
  p.groups = (units + p.upg - 1) / p.upg;
  return p;
}
static size_t mid_part_bytes(const MidPlan& p, int64_t m) { return (size_t)(p.groups + p.tiles) * m * MID_TN * 4; }

template <int MB>
static void mid_launch(const MidGemmArgs& a, hipStream_t s) {
  constexpr int NST = mid_stages(MB);
  static_assert(NST * MidStage<MB>::ELEMS * 2 * (MB <= 2 ? 2 : 1) <= 160 * 1024, "stages fit in LDS");
  hipLaunchKernelGGL((mid_gemm_kernel<MB, NST>), dim3(a.p.groups), dim3(MID_THREADS),
                     NST * MidStage<MB>::ELEMS * sizeof(bf16_t), s, a);
}

static int mid_gemm(const bf16_t* x, const bf16_t* w, int64_t m, int64_t n, int64_t k, float* part, MidSrc* src,
                    hipStream_t s) {
  MidGemmArgs a;
  a.x = x;
  a.w = w;
  a.part = part;
  a.M = (int)m;
  a.K = (int)k;
  a.p = mid_plan(m, n, k);
  *src = MidSrc{part, (int)m, a.p.ku, a.p.upg};
  switch ((m + 15) / 16) {
    case 1: mid_launch<1>(a, s); break;
    case 2: mid_launch<2>(a, s); break;
    case 3: mid_launch<3>(a, s); break;
    case 4: mid_launch<4>(a, s); break;
    case 5: mid_launch<5>(a, s); break;
    case 6: mid_launch<6>(a, s); break;
    case 7: mid_launch<7>(a, s); break;
    default: mid_launch<8>(a, s); break;
  }
  return check_launch("mid gemm");
}

static int mid_norm(const bf16_t* h, const bf16_t* delta, const MidSrc& src, const bf16_t* w, float eps, int64_t m,
                    int hidden, bf16_t* h_out, bf16_t* x, hipStream_t s) {
  const dim3 g((unsigned)m), b(MID_NORM_THREADS);
  const int cpt = (hidden / 8 + MID_NORM_THREADS - 1) / MID_NORM_THREADS;
  if (cpt <= 1) hipLaunchKernelGGL(mid_norm_kernel<1>, g, b, 0, s, h, delta, src, w, eps, hidden, h_out, x);
  else if (cpt <= 2) hipLaunchKernelGGL(mid_norm_kernel<2>, g, b, 0, s, h, delta, src, w, eps, hidden, h_out, x);
  else hipLaunchKernelGGL(mid_norm_kernel<4>, g, b, 0, s, h, delta, src, w, eps, hidden, h_out, x);
  return check_launch("mid norm");
}

static int mid_reduce(const MidSrc& src, const bf16_t* bias, int64_t n, bf16_t* y, hipStream_t s) {
  const int64_t t = src.M * (n / 8);
  hipLaunchKernelGGL(mid_reduce_kernel, dim3((unsigned)((t + 255) / 256)), dim3(256), 0, s, src, bias, (int)n, y);
  return check_launch("mid reduce");
}

static size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

struct MidShape {
  int64_t m, t_cap;
  int hidden, hq, hkv, hd, inter;
};

static bool mid_layers_shape_ok(const MidShape& d) {
  if (d.hq <= 0 || d.hkv <= 0 || d.hq % d.hkv || (d.hd != 64 && d.hd != 128) || d.hidden <= 0 || d.inter <= 0 ||
      d.hidden > MID_MAX_HIDDEN || d.inter > (1 << 22) || d.hq > 4096 || d.t_cap <= 0)
    return false;
  return mid_shape_ok(d.m, (int64_t)(d.hq + 2 * d.hkv) * d.hd, d.hidden) &&
         mid_shape_ok(d.m, d.hidden, (int64_t)d.hq * d.hd) && mid_shape_ok(d.m, 2 * (int64_t)d.inter, d.hidden) &&
         mid_shape_ok(d.m, d.hidden, d.inter) && d.inter % MID_TN == 0;
}

// Workspace of a layer: x, q, attention output, gated rows, partials, attention partials.
struct MidWs {
  size_t x, q, o, act, part, attn, total;
};
static MidWs mid_ws(const MidShape& d) {
  const int64_t qd = (int64_t)d.hq * d.hd;
  MidWs w;
  size_t at = 0;
  auto take = [&](size_t b) {
    const size_t p = at;
    at += align256(b);
    return p;
  };
  w.x = take((size_t)d.m * d.hidden * 2);
  w.q = take((size_t)d.m * qd * 2);
  w.o = take((size_t)d.m * qd * 2);
  w.act = take((size_t)d.m * d.inter * 2);
  size_t part = 0;
  auto most = [&](int64_t n, int64_t k) {
    const size_t b = mid_part_bytes(mid_plan(d.m, n, k), d.m);
    if (b > part) part = b;
  };
  most((int64_t)(d.hq + 2 * d.hkv) * d.hd, d.hidden);
  most(d.hidden, qd);
  most(2 * (int64_t)d.inter, d.hidden);
  most(d.hidden, d.inter);
  w.part = take(part);
  w.attn = take(tread_subset_attn_workspace_bytes(d.m, d.hq, d.hkv, d.hd, d.t_cap));
  w.total = at + 256;
  return w;
}

}  // namespace tread

using namespace tread;

extern "C" size_t tread_mid_linear_workspace_bytes(int64_t m, int64_t n, int64_t k) {
  return mid_shape_ok(m, n, k) ? mid_part_bytes(mid_plan(m, n, k), m) : 0;
}

extern "C" int tread_mid_linear_bf16(const void* x, const void* weight, const void* bias, int64_t m, int64_t n,
                                     int64_t k, void* y, void* ws, size_t ws_bytes, tread_stream_t stream) {
  if (m == 0 || n == 0) return 0;
  if (!mid_shape_ok(m, n, k))
    return fail(TREAD_EINVAL, "mid_linear: unsupported shape (m=%lld n=%lld k=%lld)", (long long)m, (long long)n, (long long)k);
  if (!x || !weight || !y || !ws) return fail(TREAD_EINVAL, "mid_linear: null pointer");
  if (((uintptr_t)x | (uintptr_t)weight | (uintptr_t)y | (uintptr_t)ws) & 15)
    return fail(TREAD_EINVAL, "mid_linear: operands not 16-byte aligned");
  if (ws_bytes < mid_part_bytes(mid_plan(m, n, k), m)) return fail(TREAD_EINVAL, "mid_linear: workspace too small");
  MidSrc src;
  int rc = mid_gemm((const bf16_t*)x, (const bf16_t*)weight, m, n, k, (float*)ws, &src, (hipStream_t)stream);
  return rc ? rc : mid_reduce(src, (const bf16_t*)bias, n, (bf16_t*)y, (hipStream_t)stream);
}

extern "C" size_t tread_mid_layers_workspace_bytes(int64_t m, int hidden, int hq, int hkv, int head_dim, int inter,
                                                   int64_t t_cap) {
  const MidShape d = {m, t_cap, hidden, hq, hkv, head_dim, inter};
  return mid_layers_shape_ok(d) ? mid_ws(d).total : 0;
}

extern "C" int tread_mid_layers_bf16(const tread_layer_t* layers, int n_layers, const void* h, const void* delta,
                                     int64_t m, int hidden, int hq, int hkv, int head_dim, int inter, float eps,
                                     const void* cos, const void* sin, const int64_t* rows, const int64_t* kend,
                                     const int64_t* kseg, int64_t n_shared, int64_t t_cap, float scale, void* h_out,
                                     void* delta_out, void* ws, size_t ws_bytes, tread_stream_t stream) {
  if (m == 0 || n_layers == 0) return 0;
  const MidShape d = {m, t_cap, hidden, hq, hkv, head_dim, inter};
  if (n_layers < 0 || !mid_layers_shape_ok(d))
    return fail(TREAD_EINVAL, "mid_layers: unsupported shape (m=%lld hidden=%d hq=%d hkv=%d head_dim=%d inter=%d)",
                (long long)m, hidden, hq, hkv, head_dim, inter);
  if (!layers || !h || !cos || !sin || !rows || !kend || !h_out || !delta_out || !ws)
    return fail(TREAD_EINVAL, "mid_layers: null pointer");
  uintptr_t align = (uintptr_t)h | (uintptr_t)delta | (uintptr_t)cos | (uintptr_t)sin | (uintptr_t)h_out | (uintptr_t)delta_out;
  for (int l = 0; l < n_layers; ++l) {
    const tread_layer_t& w = layers[l];
    if (!w.ln1 || !w.wqkv || !w.wo || !w.ln2 || !w.wgu || !w.wd || !w.k_cache || !w.v_cache)
      return fail(TREAD_EINVAL, "mid_layers: layer %d has a null pointer", l);
    align |= (uintptr_t)w.ln1 | (uintptr_t)w.wqkv | (uintptr_t)w.wo | (uintptr_t)w.ln2 | (uintptr_t)w.wgu |
             (uintptr_t)w.wd | (uintptr_t)w.k_cache | (uintptr_t)w.v_cache;
  }
  if (align & 15) return fail(TREAD_EINVAL, "mid_layers: operands not 16-byte aligned");
  const MidWs wl = mid_ws(d);
  if (ws_bytes < wl.total) return fail(TREAD_EINVAL, "mid_layers: workspace of %zu bytes, needs %zu", ws_bytes, wl.total);
  char* base = (char*)(((uintptr_t)ws + 255) & ~(uintptr_t)255);
  bf16_t *x = (bf16_t*)(base + wl.x), *q = (bf16_t*)(base + wl.q), *o = (bf16_t*)(base + wl.o);
  bf16_t *act = (bf16_t*)(base + wl.act), *ho = (bf16_t*)h_out;
  float* part = (float*)(base + wl.part);
  void* attn_ws = base + wl.attn;
  const size_t attn_bytes = tread_subset_attn_workspace_bytes(m, hq, hkv, head_dim, t_cap);
  hipStream_t s = (hipStream_t)stream;
  const int64_t qd = (int64_t)hq * head_dim, nqkv = (int64_t)(hq + 2 * hkv) * head_dim;
  const MidSrc none = {nullptr, 0, 1, 1};
  MidSrc src = none;
  int rc = 0;
  for (int l = 0; l < n_layers; ++l) {
    const tread_layer_t& w = layers[l];
    // src: the previous layer's down projection (none before the first, whose residual is delta)
    if ((rc = mid_norm(l ? ho : (const bf16_t*)h, l ? nullptr : (const bf16_t*)delta, src, (const bf16_t*)w.ln1, eps, m,
                       hidden, ho, x, s)))
      return rc;
    if ((rc = mid_gemm(x, (const bf16_t*)w.wqkv, m, nqkv, hidden, part, &src, s))) return rc;
    const int64_t tasks = m * ((int64_t)(hq + hkv) * (head_dim / 16) + (int64_t)hkv * (head_dim / 8));
    hipLaunchKernelGGL(mid_rope_kernel, dim3((unsigned)((tasks + 63) / 64)), dim3(64), 0, s, src, (const bf16_t*)w.bqkv,
                       (const bf16_t*)cos, (const bf16_t*)sin, rows, hq, hkv, head_dim, q, (bf16_t*)w.k_cache,
                       (bf16_t*)w.v_cache, t_cap);
    if ((rc = check_launch("mid rope"))) return rc;
    if ((rc = tread_subset_attn_bf16(q, w.k_cache, w.v_cache, kend, kseg, n_shared, m, hq, hkv, head_dim, t_cap, scale, o,
                                     attn_ws, attn_bytes, stream)))
      return rc;
    if ((rc = mid_gemm(o, (const bf16_t*)w.wo, m, hidden, qd, part, &src, s))) return rc;
    if ((rc = mid_norm(ho, nullptr, src, (const bf16_t*)w.ln2, eps, m, hidden, ho, x, s))) return rc;
    if ((rc = mid_gemm(x, (const bf16_t*)w.wgu, m, 2 * (int64_t)inter, hidden, part, &src, s))) return rc;
    const int64_t at = m * (inter / 8);
    hipLaunchKernelGGL(mid_swiglu_kernel, dim3((unsigned)((at + 255) / 256)), dim3(256), 0, s, src, inter, act);
    if ((rc = check_launch("mid swiglu"))) return rc;
    if ((rc = mid_gemm(act, (const bf16_t*)w.wd, m, hidden, inter, part, &src, s))) return rc;
  }
  return mid_reduce(src, nullptr, hidden, (bf16_t*)delta_out, s);
}
