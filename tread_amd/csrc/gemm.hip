// Projections of many token rows: y[M, N] = x[M, K] . W[N, K]^T in bf16 with fp32 sums, plain or with the
// MLP's SiLU gating in the epilogue (W = [gate; up], y = bf16(bf16(silu(g)) * u)), so that gate|up is
// never written or read back.
//
// A work group of 8 waves owns 256 features x 256 rows of y, one work group per CU; wave (w % 4, w / 4)
// computes 64 features x 128 rows with v_mfma_f32_32x32x16_bf16 (A = weights, B = rows: a lane holds
// one row's features, four consecutive ones per register group). K goes by in tiles of 64, each
// operand's from global memory straight into one of five 32 KB LDS slots (XOR-swizzled 16-byte chunks, no
// bank conflicts by counter); a wave reads the fragments of its next 16 K while it multiplies these, also
// across tiles, so that one barrier per tile is all it waits for. The work groups are persistent: their K
// tiles form one stream over all the y tiles they own, and the next y tile's loads fly during an epilogue.
//
// Matrix cores busy 60 % of the cycles at the 1.8 GHz that the power limit leaves (1.05-1.13 PFLOP/s on
// large shapes; a library kernel with 128 x 128 features and rows per wave, one wave per SIMD, reaches
// 73 % there). Measured without effect: two 64 KB buffers or K tiles of 32, loads spread over the
// products, waves half a step apart, lines touched ahead of the loads, K order staggered over the row
// tiles; raised wave priority costs 2-3 %.
//
// y tiles are dealt in rounds of one per CU; a round's tiles on one XCD form a block 8 tiles of rows
// wide, so that its L2 serves each panel several times. The last, partial round would leave CUs idle
// for up to a whole tile's K: its tiles are cut along K into `split` items, whose fp32 sums a second
// kernel adds in order.
#include "common.h"
#include "../../include/tread_hip.h"
#include "lds.h"

namespace tread {

constexpr int GEMM_BM = 256;  // rows (tokens) per tile
constexpr int GEMM_BN = 256;  // weight rows per tile
constexpr int GEMM_BK = 64;  // K per tile
constexpr int GEMM_SLOTS = 5;  // LDS slots of one operand's K tile (32 KB each)
constexpr int GEMM_WAVES = 8;
constexpr int GEMM_THREADS = GEMM_WAVES * 64;
constexpr int GEMM_CH = GEMM_BK / 8;            // 16-byte chunks per tile row
constexpr int GEMM_KS = GEMM_BK / 16;           // MFMA steps per K tile
constexpr int GEMM_TILE = GEMM_BN * GEMM_BK;    // elements of the weight (or row) tile
constexpr int GEMM_LPU = GEMM_TILE / 8 / GEMM_THREADS;  // 16-byte loads per lane and operand tile
constexpr int GEMM_GM = 8;                      // row tiles per block of the tile order
constexpr int GEMM_XCD = 8;

struct GemmArgs {
  const bf16_t* x;
  const bf16_t* w;
  const bf16_t* bias;
  bf16_t* y;
  float* part;  // [rem * split][8 waves][32 register quads][64 lanes][4] fp32 sums of the split tiles
  int64_t M, N, K;  // N: weight rows (gate and up rows with SWIGLU)
  int tm, tn;       // tiles of rows, of features
  int rounds;       // whole rounds of gridDim.x tiles
  int rem, split;   // tiles of the last round, K slices of each
};

// Tile L of the order: blocks of GEMM_GM row tiles, walked feature tile by feature tile.
__device__ __forceinline__ void gemm_tile(const GemmArgs& a, int L, int& im, int& in) {
  const int per = GEMM_GM * a.tn, g = L / per, r = L - g * per;
  const int gm = min(GEMM_GM, a.tm - g * GEMM_GM);
  in = r / gm;
  im = g * GEMM_GM + r - in * gm;
}

// Item j of work group position p: its tile, K tiles [k0, k1) and partial slot (-1: a whole tile).
struct GemmItem {
  int L, k0, k1, slot;
};
__device__ __forceinline__ bool gemm_item(const GemmArgs& a, int p, int j, GemmItem& it) {
  const int kt = (int)(a.K / GEMM_BK), G = gridDim.x;
  if (j < a.rounds) {
    it = GemmItem{j * G + p, 0, kt, -1};
    return true;
  }
  const int q = (j - a.rounds) * G + p;
  if (q >= a.rem * a.split) return false;
  const int s = q / a.rem;
  it.L = a.rounds * G + q - s * a.rem;
  it.k0 = (int)((int64_t)kt * s / a.split);
  it.k1 = (int)((int64_t)kt * (s + 1) / a.split);
  it.slot = a.split > 1 ? q : -1;
  return true;
}

// Writes one 32-feature x 32-row block: v[r] is feature f0 + (r / 4) * 8 + (lane / 32) * 4 + r % 4 of row
// `row`. Lanes l and l ^ 32 trade halves so that each stores 8 consecutive features of its row.
__device__ __forceinline__ void gemm_store(bf16_t* yr, bool row_ok, int64_t f0, int64_t nf, const float (&v)[16]) {
  const int half = (threadIdx.x & 63) >> 5;
#pragma unroll
  for (int g = 0; g < 4; g += 2) {
    u32x4_t o;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const uint32_t lo = pack_bf(v[g * 4 + 2 * q], v[g * 4 + 2 * q + 1]);
      const uint32_t hi = pack_bf(v[g * 4 + 4 + 2 * q], v[g * 4 + 4 + 2 * q + 1]);
      const auto s = __builtin_amdgcn_permlane32_swap(lo, hi, false, false);
      o[q] = s[0];
      o[2 + q] = s[1];
    }
    const int64_t f = f0 + (g + half) * 8;
    if (row_ok && f < nf) *reinterpret_cast<u32x4_t*>(yr + f) = o;
  }
}

// The epilogue of a wave's 64 x 128 sums (quad(b, c, g): registers 4 g .. 4 g + 3 of feature block b, row block c).
template <bool SWIGLU, typename Q>
__device__ __forceinline__ void gemm_epilogue(const GemmArgs& a, int im, int in, int wv, int c0, int c1, Q&& quad) {
  const int lane = threadIdx.x & 63, c31 = lane & 31, half = lane >> 5;
  const int wn = wv & 3, wm = wv >> 2;
  const int64_t nf = SWIGLU ? a.N / 2 : a.N;
#pragma unroll
  for (int c = c0; c < c1; ++c) {
    const int64_t row = (int64_t)im * GEMM_BM + wm * 128 + c * 32 + c31;
    const bool ok = row < a.M;
    bf16_t* yr = a.y + row * nf;
    float v[2][16];
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4_t s = quad(b, c, g);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[b][g * 4 + e] = s[e];
      }
    if constexpr (SWIGLU) {
#pragma unroll
      for (int r = 0; r < 16; ++r) v[0][r] = silu_bf16(bf2f(f2bf(v[0][r]))) * bf2f(f2bf(v[1][r]));
      gemm_store(yr, ok, (int64_t)in * (GEMM_BN / 2) + wn * 32, nf, v[0]);
    } else {
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const int64_t f0 = (int64_t)in * GEMM_BN + wn * 64 + b * 32;
        if (a.bias)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const int64_t f = f0 + g * 8 + half * 4;
            const u32x2_t w = f < nf ? *reinterpret_cast<const u32x2_t*>(a.bias + f) : u32x2_t{0u, 0u};
#pragma unroll
            for (int e = 0; e < 4; ++e) v[b][g * 4 + e] += e & 1 ? hi_bf(w[e / 2]) : lo_bf(w[e / 2]);
          }
        gemm_store(yr, ok, f0, nf, v[b]);
      }
    }
  }
}

template <bool SWIGLU>
__global__ __launch_bounds__(GEMM_THREADS) void gemm_kernel(const GemmArgs a) {
  constexpr int RP = 256 / (GEMM_BK * 2);  // tile rows per 256 bytes of LDS (all banks)
  extern __shared__ __align__(16) bf16_t smem[];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int c31 = lane & 31, half = lane >> 5;
  const int wn = wv & 3, wm = wv >> 2;
  const int p = (blockIdx.x % GEMM_XCD) * (gridDim.x / GEMM_XCD) + blockIdx.x / GEMM_XCD;  // an XCD's groups in a row

  int total = 0;  // K tiles of this work group's stream
  {
    GemmItem t;
    for (int j = a.rounds; gemm_item(a, p, j, t); ++j) total += t.k1 - t.k0;
    total += a.rounds * (int)(a.K / GEMM_BK);
  }
  if (total == 0) return;

  // The stream's operand tiles go through LDS slots in the order rows 0, weights 0, rows 1, ... (unit u in
  // slot u % GEMM_SLOTS). Load q of a unit fills the 64 chunk positions from (q * 8 + wave) * 64 on, lane l
  // position + l: tile row pos / CH, slot pos % CH, holding chunk slot ^ ((row / RP) % CH), so that 16 rows'
  // reads of one chunk cover every bank.
  const int lrow = wv * (64 / GEMM_CH) + lane / GEMM_CH;                    // tile row of load 0
  constexpr int LSTEP = GEMM_THREADS / GEMM_CH;                            // rows between a lane's loads
  const int lch = ((lane % GEMM_CH) ^ ((lrow / RP) % GEMM_CH)) * 8;  // LSTEP is a multiple of RP * CH
  static_assert(LSTEP % (RP * GEMM_CH) == 0, "every load of a lane takes the same chunk");
  struct Cursor {
    int j = 0, left = 0;           // next item, K tiles left of this one
    int64_t at = 0;                // K offset
    int64_t row[GEMM_LPU];         // element offsets of this lane's rows
  };
  Cursor cx, cw;
  auto advance = [&](Cursor& c, bool weights) {
    if (c.left == 0) {
      GemmItem t;
      if (!gemm_item(a, p, c.j, t)) return;  // past the stream's end: the last K tile again, into free slots
      ++c.j;
      c.left = t.k1 - t.k0;
      int im, in;
      gemm_tile(a, t.L, im, in);
#pragma unroll
      for (int q = 0; q < GEMM_LPU; ++q) {
        const int row = lrow + q * LSTEP;
        int64_t g;
        if (!weights) {
          g = min((int64_t)im * GEMM_BM + row, a.M - 1);
        } else if constexpr (SWIGLU) {  // 32 gate rows, then the up rows of the same features, and so on
          const int64_t f = min((int64_t)in * (GEMM_BN / 2) + (row >> 6) * 32 + (row & 31), a.N / 2 - 1);
          g = (row & 32) ? a.N / 2 + f : f;
        } else {
          g = min((int64_t)in * GEMM_BN + row, a.N - 1);
        }
        c.row[q] = g * a.K + lch;
      }
      c.at = (int64_t)t.k0 * GEMM_BK;
    } else {
      c.at += GEMM_BK;
    }
    --c.left;
  };
  auto load = [&](const Cursor& c, const bf16_t* base, int q, int slot) {
    lds_load16(base + c.row[q] + c.at, smem + slot * GEMM_TILE + (q * GEMM_WAVES + wv) * 64 * 8);
  };

  // fragment addresses in slot 0: tile row (block) + lane % 32, chunk 2 step + lane / 32
  uint32_t waddr[GEMM_KS], xaddr[GEMM_KS];
#pragma unroll
  for (int s = 0; s < GEMM_KS; ++s) {
    const int ch = ((2 * s + half) ^ ((c31 / RP) % GEMM_CH)) * 8;
    waddr[s] = lds_addr(smem + (wn * 64 + c31) * GEMM_BK + ch);
    xaddr[s] = lds_addr(smem + (wm * 128 + c31) * GEMM_BK + ch);
  }
  constexpr int BLK = 32 * GEMM_BK * 2;  // bytes of a 32-row block
  struct Frags {
    bf16x8_t w[2], x[4];
  };
  auto read = [&](auto S, uint32_t ow, uint32_t ox, Frags& f) {
    constexpr int s = decltype(S)::value;
    f.w[0] = lds_read128<0>(waddr[s] + ow);
    f.x[0] = lds_read128<0>(xaddr[s] + ox);
    f.x[1] = lds_read128<BLK>(xaddr[s] + ox);
    f.w[1] = lds_read128<BLK>(waddr[s] + ow);
    f.x[2] = lds_read128<2 * BLK>(xaddr[s] + ox);
    f.x[3] = lds_read128<3 * BLK>(xaddr[s] + ox);
  };
  auto wait = [&](auto N, Frags& f) {  // f's six reads landed, N later ones may fly
    constexpr int n = decltype(N)::value;
    asm volatile("s_waitcnt lgkmcnt(%6)"
                 : "+v"(f.w[0]), "+v"(f.w[1]), "+v"(f.x[0]), "+v"(f.x[1]), "+v"(f.x[2]), "+v"(f.x[3])
                 : "n"(n));
  };
  f32x16_t acc[2][4];
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[b][c][r] = 0.f;
  auto mma = [&](const Frags& f) {
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int b = 0; b < 2; ++b) acc[b][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.w[b], f.x[c], acc[b][c], 0, 0, 0);
  };

  // units 0 .. 4: rows 0, weights 0, rows 1, weights 1, rows 2
#pragma unroll
  for (int u = 0; u < GEMM_SLOTS; ++u) {
    advance(u & 1 ? cw : cx, u & 1);
#pragma unroll
    for (int q = 0; q < GEMM_LPU; ++q) load(u & 1 ? cw : cx, u & 1 ? a.w : a.x, q, u);
  }
  vm_wait<3 * GEMM_LPU>();  // tile 0 landed
  tile_barrier();
  Frags f0, f1;
  read(std::integral_constant<int, 0>{}, GEMM_TILE * 2u, 0u, f0);
  wait(std::integral_constant<int, 0>{}, f0);
  int cj = 0, ck = 0, sx = 0;  // item and K tiles left of the products, slot of the tile's rows
  GemmItem cur{};
  auto slot_add = [](int s, int d) { return s + d >= GEMM_SLOTS ? s + d - GEMM_SLOTS : s + d; };
  for (int i = 0; i < total; ++i) {
    if (ck == 0) {
      gemm_item(a, p, cj++, cur);
      ck = cur.k1 - cur.k0;
    }
    const int sw = slot_add(sx, 1), nx = slot_add(sx, 2), nw = slot_add(sx, 3);
    const uint32_t ox = (uint32_t)(sx * GEMM_TILE * 2), ow = (uint32_t)(sw * GEMM_TILE * 2);
    static_for<GEMM_KS>([&](auto S) {
      constexpr int s = decltype(S)::value;
      Frags& now = (s & 1) ? f1 : f0;
      Frags& nxt = (s & 1) ? f0 : f1;
      if constexpr (s + 1 < GEMM_KS) {
        read(std::integral_constant<int, s + 1>{}, ow, ox, nxt);
        if constexpr (s > 0) wait(std::integral_constant<int, 6>{}, now);
        mma(now);
      } else {
        wait(std::integral_constant<int, 0>{}, now);  // this wave is done reading the tile
        // the next tile landed for this wave (the rows after it may fly), then for all; this tile's
        // slots are free for all: they take the weights of tile i + 2 and the rows of tile i + 3
        vm_wait<GEMM_LPU>();
        tile_barrier();
        read(std::integral_constant<int, 0>{}, (uint32_t)(nw * GEMM_TILE * 2), (uint32_t)(nx * GEMM_TILE * 2), nxt);
        advance(cw, true);
#pragma unroll
        for (int q = 0; q < GEMM_LPU; ++q) load(cw, a.w, q, sx);
        advance(cx, false);
#pragma unroll
        for (int q = 0; q < GEMM_LPU; ++q) load(cx, a.x, q, sw);
        mma(now);
        wait(std::integral_constant<int, 0>{}, nxt);  // no read is in flight where the loop closes
      }
    });
    sx = nx;
    if (--ck == 0) {
      if (cur.slot >= 0) {
        float* pp = a.part + ((int64_t)cur.slot * GEMM_WAVES + wv) * 32 * 256 + lane * 4;
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int g = 0; g < 4; ++g)
              *reinterpret_cast<f32x4_t*>(pp + ((b * 4 + c) * 4 + g) * 256) =
                  f32x4_t{acc[b][c][4 * g], acc[b][c][4 * g + 1], acc[b][c][4 * g + 2], acc[b][c][4 * g + 3]};
      } else {
        int im, in;
        gemm_tile(a, cur.L, im, in);
        gemm_epilogue<SWIGLU>(a, im, in, wv, 0, 4, [&](int b, int c, int g) {
          return f32x4_t{acc[b][c][4 * g], acc[b][c][4 * g + 1], acc[b][c][4 * g + 2], acc[b][c][4 * g + 3]};
        });
      }
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[b][c][r] = 0.f;
    }
  }
  vm_wait<0>();  // the loads past the stream's end
}

// Adds the K slices of the last round's tiles in order and finishes them: one wave per 64 features x 32 rows
// of a tile (a 32-row block of one of the tile's waves: tile, wave, block from blockIdx.x).
template <bool SWIGLU>
__global__ __launch_bounds__(64) void gemm_reduce_kernel(const GemmArgs a, int first) {
  const int c0 = blockIdx.x & 3, wv = (blockIdx.x >> 2) % GEMM_WAVES, t = (blockIdx.x >> 2) / GEMM_WAVES;
  int im, in;
  gemm_tile(a, first + t, im, in);
  const float* p0 = a.part + ((int64_t)t * GEMM_WAVES + wv) * 32 * 256 + (threadIdx.x & 63) * 4;
  const int64_t st = (int64_t)a.rem * GEMM_WAVES * 32 * 256;
  gemm_epilogue<SWIGLU>(a, im, in, wv, c0, c0 + 1, [&](int b, int c, int g) {
    const float* pp = p0 + ((b * 4 + c) * 4 + g) * 256;
    f32x4_t s = *reinterpret_cast<const f32x4_t*>(pp);
    for (int k = 1; k < a.split; ++k) s += *reinterpret_cast<const f32x4_t*>(pp + k * st);
    return s;
  });
}

struct GemmPlan {
  int tm, tn, groups, rounds, rem, split;
};

static bool gemm_shape_ok(int64_t m, int64_t n, int64_t k) {
  return m > 0 && n > 0 && k > 0 && n % 8 == 0 && k % GEMM_BK == 0 && m <= (1 << 24) && n <= (1 << 24) && k <= (1 << 20) &&
         ((m + GEMM_BM - 1) / GEMM_BM) * ((n + GEMM_BN - 1) / GEMM_BN) <= (1 << 24);
}

static GemmPlan gemm_plan(int64_t m, int64_t n, int64_t k) {
  GemmPlan p;
  p.tm = (int)((m + GEMM_BM - 1) / GEMM_BM);
  p.tn = (int)((n + GEMM_BN - 1) / GEMM_BN);
  const int tiles = p.tm * p.tn, cus = cu_count();
  p.groups = cus >= GEMM_XCD ? cus / GEMM_XCD * GEMM_XCD : GEMM_XCD;
  p.rounds = tiles / p.groups;
  p.rem = tiles % p.groups;
  p.split = 1;
  // Cost of the last round in K tiles (about 1 us each): its rounds of 1 / split tiles, and for cut
  // tiles the reduction's launch and the 256 KB of sums that each slice writes and the reduction reads.
  if (p.rem) {
    const int kt = (int)(k / GEMM_BK);
    double best = kt;
    for (int s = 2; s <= 8 && kt / s >= 8; ++s) {
      const double items = (double)p.rem * s / p.groups;
      const double cost = (double)((p.rem * s + p.groups - 1) / p.groups) * kt / s + 3 + 24 * items;
      if (cost < best) best = cost, p.split = s;
    }
  }
  return p;
}

static size_t gemm_ws_bytes(const GemmPlan& p) {
  return p.rem && p.split > 1 ? (size_t)p.rem * p.split * GEMM_BM * GEMM_BN * sizeof(float) : 0;
}

template <bool SWIGLU>
static int gemm_launch(const GemmArgs& a, const GemmPlan& p, hipStream_t s) {
  hipLaunchKernelGGL(gemm_kernel<SWIGLU>, dim3(p.groups), dim3(GEMM_THREADS),
                     GEMM_SLOTS * GEMM_TILE * sizeof(bf16_t), s, a);
  int rc = check_launch("linear");
  if (rc || !p.rem || p.split <= 1) return rc;
  hipLaunchKernelGGL(gemm_reduce_kernel<SWIGLU>, dim3(p.rem * GEMM_WAVES * 4), dim3(64), 0, s, a, p.rounds * p.groups);
  return check_launch("linear reduce");
}

static int gemm_run(const char* what, const void* x, const void* w, const void* bias, int64_t m, int64_t n, int64_t k,
                    bool swiglu, void* y, void* ws, size_t ws_bytes, hipStream_t s) {
  if (m == 0 || n == 0) return 0;
  if (!gemm_shape_ok(m, n, k) || (swiglu && n % 16))
    return fail(TREAD_EINVAL, "%s: unsupported shape (m=%lld n=%lld k=%lld)", what, (long long)m, (long long)n, (long long)k);
  if (!x || !w || !y) return fail(TREAD_EINVAL, "%s: null pointer", what);
  if (((uintptr_t)x | (uintptr_t)w | (uintptr_t)y | (uintptr_t)bias) & 15) return fail(TREAD_EINVAL, "%s: operands not 16-byte aligned", what);
  GemmPlan p = gemm_plan(m, n, k);
  if (gemm_ws_bytes(p) && (!ws || ((uintptr_t)ws & 15) || ws_bytes < gemm_ws_bytes(p))) p.split = 1;
  GemmArgs a;
  a.x = (const bf16_t*)x;
  a.w = (const bf16_t*)w;
  a.bias = (const bf16_t*)bias;
  a.y = (bf16_t*)y;
  a.part = (float*)ws;
  a.M = m;
  a.N = n;
  a.K = k;
  a.tm = p.tm;
  a.tn = p.tn;
  a.rounds = p.rounds;
  a.rem = p.rem;
  a.split = p.split;
  return swiglu ? gemm_launch<true>(a, p, s) : gemm_launch<false>(a, p, s);
}

}  // namespace tread

using namespace tread;

extern "C" size_t tread_linear_workspace_bytes(int64_t m, int64_t n, int64_t k) {
  return gemm_shape_ok(m, n, k) ? gemm_ws_bytes(gemm_plan(m, n, k)) : 0;
}

extern "C" int tread_linear_bf16(const void* x, const void* weight, const void* bias, int64_t m, int64_t n, int64_t k,
                                 void* y, void* ws, size_t ws_bytes, tread_stream_t stream) {
  return gemm_run("linear", x, weight, bias, m, n, k, false, y, ws, ws_bytes, (hipStream_t)stream);
}

extern "C" int tread_linear_swiglu_bf16(const void* x, const void* wgu, int64_t m, int64_t inter, int64_t k, void* y,
                                        void* ws, size_t ws_bytes, tread_stream_t stream) {
  return gemm_run("linear_swiglu", x, wgu, nullptr, m, 2 * inter, k, true, y, ws, ws_bytes, (hipStream_t)stream);
}
