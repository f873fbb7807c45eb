// lbk_tile64.hip — Block-ELL products at B = 64 (forward: more tokens than the decode kernels take)
// (gfx950, bf16 MFMA): y = x W (+ bias), h = silu(x Wg) * (x Wu), out = h Wd (+ residual).
//
// t64_kernel<MODE, MT, ST>: a workgroup of four waves owns 64 MT tokens and one block row, wave w
// 16 MT of the tokens and all 64 output columns.  The row's live slots (gate's, then up's) are the
// steps of its main loop.  A step needs the slot's raw [64 in, 64 out] tile (8 KB) and the
// tokens' 128-byte pieces of the slot's column block (8 MT KB).  Both come to LDS by direct
// global -> LDS loads (16 bytes a lane, eight lanes a row, so every line is read whole), ST steps
// deep; one barrier a step.  The tile is the MFMA's A operand, read transposed
// (ds_read_b64_tr_b16), so weights need no packed copy, and the tokens are the B operand, so a lane
// ends with four consecutive columns of one token.
//
// Bound by the lines that miss the L2 (3.7 TB/s at 1.1 GB through it at the size below); each
// token's pieces are read once per block row that uses them.  4096 -> 14336 at 0.1, 2048 tokens:
// gate/up 243 -> 84 us (545 TFLOP/s), down 129 -> 37 us (630) against the row-block kernel.
//
// LDS layout: a token row's 16-byte chunk c is at chunk c ^ (row & 7): the eight lanes of a read
// phase fall on eight chunks.  A tile row's chunk c is at c ^ f(row), f = 2 bit1(row) + 4 bit3(row):
// the transposed reads of a half-wave (rows t .. t + 3, t + 8 .. t + 11, 32 bytes each) cover the
// 64 banks once.
#include "lbk_device.h"
#include "lbk_internal.h"

namespace lbk {
namespace {

constexpr int T64_TILE = 64 * 64 * 2;    // bytes of a tile, and of 64 tokens' column block

// barrier without a fence: this wave's LDS reads have returned, its loads in flight stay so
__device__ __forceinline__ void t64_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

typedef short t64_i16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) t64_i16x4 lds_t64_i16x4;
typedef __attribute__((address_space(3))) unsigned char lds_byte;

}  // namespace

template <int MODE, int MT, int ST>
__global__ __launch_bounds__(256, 2) void t64_kernel(T64Args a) {
  constexpr int NL = MODE == 1 ? 2 : 1;
  constexpr int TM = 64 * MT;
  constexpr int STEP = TM * 128 + T64_TILE;       // bytes of a step's token pieces and tile
  constexpr int NLD = 2 * MT + 2;                 // 1 KB loads of a step per wave
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = uniform(tid >> 6);
  const int i = lane & 15, g = lane >> 4;
  // workgroup -> (token block, block row): the 8 XCDs (workgroups are dealt to them round robin)
  // form tg token groups by 8 / tg row groups; an XCD takes its token blocks one after the other,
  // all of its rows for each, so that its L2 holds the block's activations while its rows' tiles
  // stream through
  const int xcd = (int)(blockIdx.x & 7), rgs = 8 / a.tg;
  const int64_t j = blockIdx.x >> 3;
  const int rl = (a.R + rgs - 1) / rgs;              // rows of a row group
  const int64_t tl = j / rl;
  const int r = (int)(j - tl * rl) * rgs + xcd / a.tg;
  const int64_t tb = tl * a.tg + xcd % a.tg;
  if (r >= a.R || tb * TM >= a.N) return;            // the whole workgroup, before any barrier
  const int64_t t0 = tb * TM;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_byte*)smem;

  // offsets of this lane's loads: token rows 16 MT w + 8 j + l / 8 (clamped to the last token),
  // chunk l % 8 of the stored order; tile rows 16 w + 8 j + l / 8
  uint32_t xoff[2 * MT], woff[2];
#pragma unroll
  for (int j = 0; j < 2 * MT; ++j) {
    const int row = 16 * MT * w + 8 * j + (lane >> 3);
    const int64_t left = a.N - 1 - t0;
    const int rc = row < left ? row : (int)left;
    xoff[j] = (uint32_t)rc * (uint32_t)(a.ldx * 2) + (uint32_t)(((lane & 7) ^ (row & 7)) << 4);
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int row = 16 * w + 8 * j + (lane >> 3);
    woff[j] = (uint32_t)(row * 128 + (((lane & 7) ^ (((row & 2)) | ((row & 8) >> 1))) << 4));
  }

  // the row's slots, 64 at a time: lane l holds the column of slot base + l, and order the lanes
  // of the live slots, gate's before up's, by ascending column: the rows that run together sweep
  // the columns together, and share the lines of a token block wider than the L2
  const int K0 = a.K0, T = MODE == 1 ? a.K0 + a.K1 : a.K0;
  int base = 0, colreg = -1, order = 0, nlive = 0, pos = 0;
  auto window = [&]() {
    const int e = base + lane;
    const int32_t* p = (MODE == 1 && e >= K0) ? a.c1 + (int64_t)r * a.K1 + (e - K0) : a.c0 + (int64_t)r * K0 + e;
    colreg = e < T ? *p : -1;
    const bool live = colreg >= 0 && colreg < a.C;
    const uint64_t lm = __ballot(live);
    const int key = (MODE == 1 && e >= K0) ? colreg | (1 << 30) : colreg;
    int rank = 0;
    for (uint64_t m = lm; m; m &= m - 1) {
      const int u = __builtin_ctzll(m);
      const int ku = __builtin_amdgcn_readlane(key, u);
      rank += (ku < key || (ku == key && u < lane)) ? 1 : 0;
    }
    nlive = __builtin_popcountll(lm);
    const int below = __builtin_amdgcn_mbcnt_hi((uint32_t)(lm >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)lm, 0));
    order = __builtin_amdgcn_ds_permute((live ? rank : nlive + lane - below) << 2, lane);
    pos = 0;
  };
  if (T > 0) window();
  const char* const xb = reinterpret_cast<const char*>(a.x + t0 * a.ldx);
  int issued = 0;
  uint32_t upmask = 0;       // bit s: ring slot s holds a step of the up weight
  // the next live slot's loads into ring slot `issued` % ST (false: no slots are left)
  auto issue = [&](int slot) {
    while (pos == nlive) {
      base += 64;
      if (base >= T) return false;
      window();
    }
    const int bit = __builtin_amdgcn_readlane(order, pos++);
    const int e = base + bit;
    const int col = __builtin_amdgcn_readlane(colreg, bit);
    const bool up = MODE == 1 && e >= K0;
    const char* wp = up ? reinterpret_cast<const char*>(a.v1) + ((int64_t)r * a.K1 + (e - K0)) * T64_TILE
                        : reinterpret_cast<const char*>(a.v0) + ((int64_t)r * K0 + e) * T64_TILE;
    const char* xp = xb + (int64_t)col * 128;
    const uint32_t l0 = lds0 + (uint32_t)(slot * STEP);
#pragma unroll
    for (int j = 0; j < 2; ++j) lds_load16(wp, woff[j], l0 + (uint32_t)(TM * 128 + (2 * w + j) * 1024));
#pragma unroll
    for (int j = 0; j < 2 * MT; ++j) lds_load16(xp, xoff[j], l0 + (uint32_t)((2 * MT * w + j) * 1024));
    if (MODE == 1) upmask = (upmask & ~(1u << slot)) | ((up ? 1u : 0u) << slot);
    ++issued;
    return true;
  };

  f32x4 acc[NL][MT][4];
#pragma unroll
  for (int l = 0; l < NL; ++l)
#pragma unroll
    for (int q = 0; q < MT; ++q)
#pragma unroll
      for (int m = 0; m < 4; ++m) acc[l][q][m] = f32x4{0.f, 0.f, 0.f, 0.f};

  // this lane's byte offsets within a step: token row 16 q + i of the wave, chunk 4 ks + g; tile
  // rows 32 ks + 8 g + i / 4 (and + 4), columns 16 m + 4 (i & 3)
  const uint32_t xl = (uint32_t)((16 * MT * w + i) * 128);
  const uint32_t xc0 = (uint32_t)((g ^ (i & 7)) << 4), xc1 = (uint32_t)(((4 + g) ^ (i & 7)) << 4);
  const uint32_t fl = (uint32_t)(((i >> 3) & 1) * 2 | (g & 1) * 4);
  const uint32_t wl = (uint32_t)(TM * 128 + (8 * g + (i >> 2)) * 128 + (i & 1) * 8 + (((i & 3) >> 1) << 4));
  auto compute = [&](uint32_t s0, f32x4 (&c)[MT][4]) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      u32x4 wf[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const uint32_t ad = s0 + wl + (uint32_t)(ks * 4096) + (((uint32_t)(2 * m) ^ fl) << 4);
        const t64_i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_t64_i16x4*)(lds_byte*)(smem + ad));
        const t64_i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_t64_i16x4*)(lds_byte*)(smem + ad + 512));
        const u32x2 p0 = __builtin_bit_cast(u32x2, lo), p1 = __builtin_bit_cast(u32x2, hi);
        wf[m] = u32x4{p0[0], p0[1], p1[0], p1[1]};
      }
#pragma unroll
      for (int q = 0; q < MT; ++q) {
        const u32x4 xf = *reinterpret_cast<const u32x4*>(smem + s0 + xl + (uint32_t)(q * 2048) + (ks ? xc1 : xc0));
#pragma unroll
        for (int m = 0; m < 4; ++m) c[q][m] = mfma_bf16(wf[m], xf, c[q][m]);
      }
    }
  };

#pragma unroll
  for (int s = 0; s < ST - 1; ++s)
    if (!issue(s)) break;
  int slot = 0, islot = ST - 1, s = 0;
  auto step = [&](f32x4 (&c)[MT][4]) {
    // this wave's loads of step s have landed once only the later steps' are in flight
    const int later = issued - s - 1;
    if (ST > 3 && later >= 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NLD) : "memory");
    else if (ST > 2 && later >= 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NLD) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    t64_barrier();           // every wave's have, and step s - 1 is read: its ring slot is free
    if (issue(islot)) islot = islot + 1 == ST ? 0 : islot + 1;
    compute((uint32_t)(slot * STEP), c);
    slot = slot + 1 == ST ? 0 : slot + 1;
    ++s;
  };
  // gate's steps, then up's (one loop each: the accumulators stay in fixed registers)
  while (s < issued && (MODE != 1 || !((upmask >> slot) & 1))) step(acc[0]);
  if (MODE == 1)
    while (s < issued) step(acc[NL - 1]);

  // lane (i, g) of acc[.][q][m]: token 16 q + i of the wave, columns 16 m + 4 g .. + 3
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const int64_t oc = (int64_t)r * 64 + 16 * m + 4 * g;
    float b0[4], b1[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      b0[v] = a.bias ? a.bias[oc + v] : 0.f;
      b1[v] = MODE == 1 && a.bias1 ? a.bias1[oc + v] : 0.f;
    }
#pragma unroll
    for (int q = 0; q < MT; ++q) {
      const int64_t t = t0 + 16 * MT * w + 16 * q + i;
      if (t >= a.N) continue;
      float o[4];
      if constexpr (MODE == 1) {
        float gv[4], uv[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          gv[v] = acc[0][q][m][v] + b0[v];
          uv[v] = acc[NL - 1][q][m][v] + b1[v];
          o[v] = silu_f(gv[v]) * uv[v];
        }
        if (a.aux0) store_bf16x<4>(a.aux0 + t * a.ldaux + oc, gv);
        if (a.aux1) store_bf16x<4>(a.aux1 + t * a.ldaux + oc, uv);
      } else {
        float rv[4] = {0.f, 0.f, 0.f, 0.f};
        if (MODE == 2 && a.resid) load_bf16x<4>(a.resid + t * a.ldr + oc, rv);
#pragma unroll
        for (int v = 0; v < 4; ++v) o[v] = acc[0][q][m][v] + b0[v] + rv[v];
        if (MODE == 0 && a.gelu) {
          if (a.aux0) store_bf16x<4>(a.aux0 + t * a.ldaux + oc, o);
#pragma unroll
          for (int v = 0; v < 4; ++v) o[v] = gelu_f(o[v]);
        }
      }
      store_bf16x<4>(a.y + t * a.ldy + oc, o);
    }
  }
}

// Token groups that the XCDs form for ntb token blocks of tm tokens: the split that moves the
// fewest bytes into one XCD's L2 -- its share of the activations, and its rows' tiles once for each
// pass over them (64 workgroups of an XCD run together: token blocks with fewer rows share a pass)
// -- among those whose last round of token blocks is at least 0.9 full.
// 4096 -> 14336 at 0.1, us a forward: 2048 tokens 114 with 8 groups, 119 / 128 / 140 with 4 / 2 / 1;
// 500 tokens 46 with 4 (down's choice), 50 with 8.
static int t64_groups(const RowblockLaunch& a, int64_t ntb) {
  const double xb = 128.0 * (double)a.N * a.C, wb = (double)T64_TILE * a.R * (a.K0 + a.K1);
  int best = 1;
  double cost = 0;
  for (int tg = 1; tg <= 8; tg *= 2) {
    const int64_t rounds = (ntb + tg - 1) / tg;
    if (tg > 1 && 10 * ntb < 9 * rounds * tg) continue;
    const int rgs = 8 / tg, rl = (a.R + rgs - 1) / rgs;
    const double passes = (double)rounds * (rl < 64 ? rl : 64) / 64;
    const double c = xb / tg + wb / rgs * (passes > 1 ? passes : 1);
    if (tg == 1 || c < cost) {
      cost = c;
      best = tg;
    }
  }
  return best;
}

template <int MODE, int MT, int ST>
static int launch_t64_t(const RowblockLaunch& a0, hipStream_t st) {
  T64Args a;
  static_cast<RowblockLaunch&>(a) = a0;
  constexpr int lds = ST * (64 * MT * 128 + T64_TILE);
  auto kern = t64_kernel<MODE, MT, ST>;
  static std::atomic<uint64_t> done{0};
  if (lds > 65536 && set_lds_limit_once(reinterpret_cast<const void*>(kern), lds, done)) return -1;
  const int64_t ntb = (a.N + 64 * MT - 1) / (64 * MT);
  a.tg = t64_groups(a, ntb);
  const int rgs = 8 / a.tg;
  const int64_t grid = 8 * ((a.R + rgs - 1) / rgs) * ((ntb + a.tg - 1) / a.tg);
  if (grid > 0x7fffffff) return -2;
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(256), lds, st, a);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_t64(int mode, const RowblockLaunch& a, hipStream_t st) {
  auto bad = [](const void* p, uintptr_t m) { return (reinterpret_cast<uintptr_t>(p) & m) != 0; };
  // 16-byte loads of activations and tiles, 8-byte stores; 32-bit offsets within a token block
  if (bad(a.x, 15) || a.ldx % 8 || bad(a.v0, 15) || (mode == 1 && bad(a.v1, 15)) || bad(a.y, 7) || a.ldy % 4 ||
      ((mode == 1 || a.gelu) && ((a.aux0 && bad(a.aux0, 7)) || (a.aux1 && bad(a.aux1, 7)) || a.ldaux % 4)) ||
      (mode == 2 && a.resid && (bad(a.resid, 7) || a.ldr % 4)) || a.ldx > (1 << 22))
    return -2;
  // one slot a row: a single step has nothing to overlap, and the row-block kernel, without the trip
  // through LDS, is faster (us here / there, products of 3000 tokens: 512 -> 2048 10.1 / 7.6, 256 -> 896 6.7 /
  // 4.8; 10000 x 2048 -> 512 9.6 / 7.1; with two slots 11.0 / 11.6, 7.7 / 7.0, 10.3 / 10.6).  Gate/up of one slot
  // each stays: within 1 us up to 700 tokens, 3 to 20 us faster from 5000.
  if (mode != 1 && !a.gelu && a.K0 <= 1 && a.R <= 65535) return -2;
  // the largest token block that leaves two workgroups per CU (2048 tokens, 2048 -> 8192 at 0.5: 159
  // us with 256 tokens two steps deep, 165 and 194 with 128 and 64; three and four steps deep, with
  // fewer workgroups resident, 175 to 236)
  auto wgs = [&](int tm) { return (int64_t)a.R * ((a.N + tm - 1) / tm); };
  const int mt = wgs(256) >= 512 ? 4 : wgs(128) >= 512 ? 2 : 1;
#define LBK_T64(MODE)                                                  \
  if (mode == MODE) {                                                  \
    if (mt == 4) return launch_t64_t<MODE, 4, 2>(a, st);               \
    if (mt == 2) return launch_t64_t<MODE, 2, 3>(a, st);               \
    return launch_t64_t<MODE, 1, 4>(a, st);                            \
  }
  LBK_T64(0) LBK_T64(1) LBK_T64(2)
#undef LBK_T64
  return -2;
}

// ---------------------------------------------------------------------------
// the transposed product: dx[:, c] = sum over the list entries of column block c of A[:, r] W[e]^T
// ---------------------------------------------------------------------------
// t64_dx_kernel<MT, ST>: the kernel above for the backward's dx at B = 64.  The steps are the entries
// of the transposed topology of an output column block, dg's and then du's, into one accumulator; the
// tile's rows are the output columns, so it is read as it lies (rows of 16-byte chunks, chunk c at
// c ^ (row & 7), as the tokens' pieces).  3000 x 1024, d_ff 4096 at 0.5: 232 us with the activations
// staged 256 columns at a time by 94 workgroups, 51 us so.
template <int MT, int ST>
__global__ __launch_bounds__(256, 2) void t64_dx_kernel(TProdArgs a, int tg) {
  constexpr int TM = 64 * MT;
  constexpr int STEP = TM * 128 + T64_TILE;
  constexpr int NLD = 2 * MT + 2;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = uniform(tid >> 6);
  const int i = lane & 15, g = lane >> 4;
  // workgroup -> (token block, output column block), as in t64_kernel
  const int xcd = (int)(blockIdx.x & 7), rgs = 8 / tg;
  const int64_t j8 = blockIdx.x >> 3;
  const int rl = (a.C + rgs - 1) / rgs;
  const int64_t tl = j8 / rl;
  const int c = (int)(j8 - tl * rl) * rgs + xcd / tg;
  const int64_t tb = tl * tg + xcd % tg;
  if (c >= a.C || tb * TM >= a.N) return;            // the whole workgroup, before any barrier
  const int64_t t0 = tb * TM;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_byte*)smem;
  const TProdSrc& S0 = a.src[0];
  const TProdSrc& S1 = a.src[a.nsrc > 1 ? 1 : 0];
  const int64_t lda = S0.lda;                        // both sources' (the launcher checks it)

  uint32_t xoff[2 * MT], woff[2];
#pragma unroll
  for (int j = 0; j < 2 * MT; ++j) {
    const int row = 16 * MT * w + 8 * j + (lane >> 3);
    const int64_t left = a.N - 1 - t0;
    const int rc = row < left ? row : (int)left;
    xoff[j] = (uint32_t)rc * (uint32_t)(lda * 2) + (uint32_t)(((lane & 7) ^ (row & 7)) << 4);
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int row = 16 * w + 8 * j + (lane >> 3);
    woff[j] = (uint32_t)(row * 128 + (((lane & 7) ^ (row & 7)) << 4));
  }

  // the list, 64 entries at a time: lane l holds entry base + l and its source block
  const int n0 = S0.cnt[c], T = n0 + (a.nsrc > 1 ? S1.cnt[c] : 0);
  int base = 0, ev = 0, rv = 0, pos = 0;
  auto window = [&]() {
    const int j = base + lane;
    const bool s1 = j >= n0;
    const int32_t* p = s1 ? S1.list + (int64_t)c * S1.cap + (j - n0) : S0.list + (int64_t)c * S0.cap + j;
    ev = j < T ? *p : 0;
    rv = ev / (s1 ? S1.K : S0.K);
    pos = 0;
  };
  if (T > 0) window();
  int issued = 0;
  auto issue = [&](int slot) {
    if (base + pos >= T) return false;
    if (pos == 64) {
      base += 64;
      window();
    }
    const int e = __builtin_amdgcn_readlane(ev, pos), r = __builtin_amdgcn_readlane(rv, pos);
    const bool s1 = base + pos >= n0;
    ++pos;
    const char* wp = reinterpret_cast<const char*>(s1 ? S1.w : S0.w) + (int64_t)e * T64_TILE;
    const char* xp = reinterpret_cast<const char*>((s1 ? S1.a : S0.a) + t0 * lda) + (int64_t)r * 128;
    const uint32_t l0 = lds0 + (uint32_t)(slot * STEP);
#pragma unroll
    for (int j = 0; j < 2; ++j) lds_load16(wp, woff[j], l0 + (uint32_t)(TM * 128 + (2 * w + j) * 1024));
#pragma unroll
    for (int j = 0; j < 2 * MT; ++j) lds_load16(xp, xoff[j], l0 + (uint32_t)((2 * MT * w + j) * 1024));
    ++issued;
    return true;
  };

  f32x4 acc[MT][4];
#pragma unroll
  for (int q = 0; q < MT; ++q)
#pragma unroll
    for (int m = 0; m < 4; ++m) acc[q][m] = f32x4{0.f, 0.f, 0.f, 0.f};
  const uint32_t xl = (uint32_t)((16 * MT * w + i) * 128), wl = (uint32_t)(TM * 128 + i * 128);
  const uint32_t ch0 = (uint32_t)((g ^ (i & 7)) << 4), ch1 = (uint32_t)(((4 + g) ^ (i & 7)) << 4);
#pragma unroll
  for (int s = 0; s < ST - 1; ++s)
    if (!issue(s)) break;
  int slot = 0, islot = ST - 1;
  for (int s = 0; s < issued; ++s) {
    // this wave's loads of step s have landed once only the later steps' are in flight
    const int later = issued - s - 1;
    if (ST > 3 && later >= 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NLD) : "memory");
    else if (ST > 2 && later >= 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NLD) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    t64_barrier();           // every wave's have, and step s - 1 is read: its ring slot is free
    if (issue(islot)) islot = islot + 1 == ST ? 0 : islot + 1;
    const uint32_t s0 = (uint32_t)(slot * STEP);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const uint32_t ch = ks ? ch1 : ch0;
      u32x4 wf[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) wf[m] = *reinterpret_cast<const u32x4*>(smem + s0 + wl + (uint32_t)(m * 2048) + ch);
#pragma unroll
      for (int q = 0; q < MT; ++q) {
        const u32x4 xf = *reinterpret_cast<const u32x4*>(smem + s0 + xl + (uint32_t)(q * 2048) + ch);
#pragma unroll
        for (int m = 0; m < 4; ++m) acc[q][m] = mfma_bf16(wf[m], xf, acc[q][m]);
      }
    }
    slot = slot + 1 == ST ? 0 : slot + 1;
  }

  // lane (i, g) of acc[q][m]: token 16 q + i of the wave, columns 16 m + 4 g .. + 3
#pragma unroll
  for (int q = 0; q < MT; ++q) {
    const int64_t t = t0 + 16 * MT * w + 16 * q + i;
    if (t >= a.N) continue;
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const int64_t off = t * a.ldo + (int64_t)c * 64 + 16 * m + 4 * g;
      float o[4], rr[4] = {0.f, 0.f, 0.f, 0.f};
      if (a.resid) load_bf16x<4>(a.resid + off, rr);
#pragma unroll
      for (int v = 0; v < 4; ++v) o[v] = acc[q][m][v] + rr[v];
      store_bf16x<4>(a.out + off, o);
    }
  }
}

template <int MT, int ST>
static int launch_t64_dx_t(const TProdArgs& a, hipStream_t st) {
  constexpr int lds = ST * (64 * MT * 128 + T64_TILE);
  auto kern = t64_dx_kernel<MT, ST>;
  static std::atomic<uint64_t> done{0};
  if (lds > 65536 && set_lds_limit_once(reinterpret_cast<const void*>(kern), lds, done)) return -1;
  const int64_t ntb = (a.N + 64 * MT - 1) / (64 * MT);
  RowblockLaunch b{};                                // the traffic that decides the token groups
  b.N = a.N;
  b.C = (int)(a.src[0].lda / 64);
  b.R = a.C;
  b.K0 = (int)(a.src[0].cap / a.C);
  b.K1 = a.nsrc > 1 ? (int)(a.src[1].cap / a.C) : 0;
  const int tg = t64_groups(b, ntb), rgs = 8 / tg;
  const int64_t grid = 8 * ((a.C + rgs - 1) / rgs) * ((ntb + tg - 1) / tg);
  if (grid > 0x7fffffff) return -2;
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(256), lds, st, a, tg);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_t64_dx(const TProdArgs& a, hipStream_t st) {
  auto bad = [](const void* p, uintptr_t m) { return (reinterpret_cast<uintptr_t>(p) & m) != 0; };
  if (a.nsrc < 1 || a.nsrc > 2 || a.C < 1 || bad(a.out, 7) || (a.resid && bad(a.resid, 7)) || a.ldo % 4) return -2;
  for (int s = 0; s < a.nsrc; ++s)
    if (bad(a.src[s].a, 15) || bad(a.src[s].w, 15) || a.src[s].lda != a.src[0].lda || a.src[s].lda % 64 ||
        a.src[s].lda > (1 << 22) || a.src[s].K < 1)
      return -2;
  auto wgs = [&](int tm) { return (int64_t)a.C * ((a.N + tm - 1) / tm); };
  if (wgs(256) >= 256) return launch_t64_dx_t<4, 2>(a, st);
  if (wgs(128) >= 256) return launch_t64_dx_t<2, 3>(a, st);
  return launch_t64_dx_t<1, 4>(a, st);
}

}  // namespace lbk
