// lbk_abi.hip — the extern "C" entry points declared in include/lbk.h.
//
// Each entry point validates its arguments on the host (pointers, tile size,
// shape consistency, alignment), chooses a kernel path and queues the kernels
// on the caller's stream.  Nothing is allocated, freed or synchronised here.
#include "lbk.h"
#include "lbk_internal.h"

#include <string.h>


using namespace lbk;

namespace {

inline bool a16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
inline bool a8(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 7u) == 0; }
inline hipStream_t S(void* s) { return reinterpret_cast<hipStream_t>(s); }
inline bool tile_ok(int B) { return B == 16 || B == 32 || B == 64; }
inline size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

int check_bell(const lbk_bell* w) {
  if (!w) return LBK_ERR_NULL;
  if (!tile_ok(w->B)) return LBK_ERR_TILE;
  if (w->R < 0 || w->K < 0) return LBK_ERR_SHAPE;
  if ((int64_t)w->R * w->K > 0 && (!w->values || !w->col_idx)) return LBK_ERR_NULL;
  if (w->values && !a8(w->values)) return LBK_ERR_ALIGN;
  return LBK_OK;
}

int check_tern(const lbk_bell_ternary* w) {
  if (!w) return LBK_ERR_NULL;
  if (!tile_ok(w->B)) return LBK_ERR_TILE;
  if (w->R < 0 || w->K < 0) return LBK_ERR_SHAPE;
  if ((int64_t)w->R * w->K > 0 && (!w->packed || !w->scales || !w->col_idx)) return LBK_ERR_NULL;
  if (w->packed && !a16(w->packed)) return LBK_ERR_ALIGN;
  return LBK_OK;
}

// Shared geometry check of a gate/up/down triple; returns status, fills d_ff.
template <typename W>
int check_ffn(const W* gate, const W* up, const W* down, int32_t d_model, int64_t* d_ff) {
  if (gate->R != up->R) return LBK_ERR_SHAPE;
  if (gate->B != up->B || gate->B != down->B) return LBK_ERR_TILE;
  const int B = gate->B;
  if (d_model <= 0 || d_model % B) return LBK_ERR_SHAPE;
  if ((int64_t)down->R * B != d_model) return LBK_ERR_SHAPE;
  *d_ff = (int64_t)gate->R * B;
  return LBK_OK;
}

// optional fp32 biases of the three projections (gate/up [d_ff], down [d_model])
struct Biases {
  const float* g;
  const float* u;
  const float* d;
};

int swiglu_general(const uint16_t* x, int64_t N, int32_t d_model, const lbk_bell* gate, const lbk_bell* up,
                   const lbk_bell* down, const uint16_t* resid, uint16_t* out, uint16_t* h,
                   uint16_t* gate_pre, uint16_t* up_out, hipStream_t st, Biases bs = {}) {
  const int B = gate->B;
  const int64_t d_ff = (int64_t)gate->R * B;
  RowblockLaunch a{};
  a.x = x; a.N = N; a.ldx = d_model; a.C = d_model / B; a.R = gate->R;
  a.v0 = gate->values; a.c0 = gate->col_idx; a.K0 = gate->K;
  a.v1 = up->values; a.c1 = up->col_idx; a.K1 = up->K;
  a.y = h; a.ldy = d_ff; a.aux0 = gate_pre; a.aux1 = up_out; a.ldaux = d_ff;
  a.bias = bs.g; a.bias1 = bs.u;
  if (launch_rowblock(B, 1, a, st) != 0) return LBK_ERR_LAUNCH;
  RowblockLaunch d{};
  d.x = h; d.N = N; d.ldx = d_ff; d.C = gate->R; d.R = down->R;
  d.v0 = down->values; d.c0 = down->col_idx; d.K0 = down->K;
  d.resid = resid; d.ldr = d_model;
  d.y = out; d.ldy = d_model; d.bias = bs.d;
  if (launch_rowblock(B, 2, d, st) != 0) return LBK_ERR_LAUNCH;
  return LBK_OK;
}

struct TernSplitLayout {
  size_t pg, pu, pd, hmax, h, total;
};

TernSplitLayout tern_split_layout(int64_t N, const lbk_bell_ternary* gate, const lbk_bell_ternary* up,
                                  const lbk_bell_ternary* down) {
  TernSplitLayout L{};
  L.pg = tprep_bytes((int64_t)gate->R * gate->K, gate->R, 0);
  L.pu = tprep_bytes((int64_t)up->R * up->K, up->R, 1);
  L.pd = tprep_bytes((int64_t)down->R * down->K, down->R, 2);
  L.hmax = align256((size_t)tgu_slices(N, gate->R) * (size_t)N * 4);
  L.h = align256((size_t)N * gate->R * gate->B * 2);
  L.total = L.pg + L.pu + L.pd + L.hmax + L.h;
  return L;
}

bool tern_split(int64_t N, int32_t d_model, const lbk_bell_ternary* gate, const lbk_bell_ternary* up,
                const lbk_bell_ternary* down) {
  return N > 0 && tsplit_supported(gate->B, d_model, gate->R, down->R, gate->K, up->K, down->K);
}

}  // namespace

extern "C" {

const char* lbk_status_string(int s) {
  switch (s) {
    case LBK_OK: return "ok";
    case LBK_ERR_NULL: return "a required pointer is NULL";
    case LBK_ERR_TILE: return "tile size B must be 16, 32 or 64 (and equal across gate/up/down)";
    case LBK_ERR_SHAPE: return "inconsistent shapes between operands";
    case LBK_ERR_ALIGN: return "pointer or row stride not suitably aligned (16 bytes for activations)";
    case LBK_ERR_WORKSPACE: return "workspace missing or too small";
    case LBK_ERR_LAUNCH: return "HIP kernel launch failed";
    case LBK_ERR_ARG: return "invalid argument";
    case LBK_ERR_COLUMN: return "column index out of range";
    case LBK_ERR_TOO_LARGE: return "geometry needs more than the no-alloc entry point's fixed scratch";
    default: return "unknown status";
  }
}

int lbk_version(void) { return LBK_VERSION; }

int lbk_check_columns(const int32_t* col_idx, int64_t count, int32_t C, int32_t* bad_count_dev, void* stream) {
  if (!bad_count_dev || (count > 0 && !col_idx)) return LBK_ERR_NULL;
  if (count < 0 || C < 0) return LBK_ERR_ARG;
  return launch_check_columns(col_idx, count, C, bad_count_dev, S(stream)) == 0 ? LBK_OK : LBK_ERR_LAUNCH;
}

int lbk_block_ell_matmul_bf16(const uint16_t* x, int64_t N, int32_t in_features, int64_t ldx, const lbk_bell* w,
                              const float* bias, uint16_t* y, int64_t ldy, void* stream) {
  int st = check_bell(w);
  if (st) return st;
  if (N < 0) return LBK_ERR_ARG;
  if (in_features <= 0 || in_features % w->B) return LBK_ERR_SHAPE;
  if (N == 0) return LBK_OK;
  if (!x || !y) return LBK_ERR_NULL;
  if (ldx < in_features || ldy < (int64_t)w->R * w->B) return LBK_ERR_SHAPE;
  if (!a16(x) || (ldx % 8) || !a16(y) || (ldy % 8)) return LBK_ERR_ALIGN;
  RowblockLaunch a{};
  a.x = x; a.N = N; a.ldx = ldx; a.C = in_features / w->B; a.R = w->R;
  a.v0 = w->values; a.c0 = w->col_idx; a.K0 = w->K;
  a.bias = bias; a.y = y; a.ldy = ldy;
  return launch_rowblock(w->B, 0, a, S(stream)) == 0 ? LBK_OK : LBK_ERR_LAUNCH;
}

// The plain product on packed tiles: the gate/up kernel's gate stream over an LDS panel of x
// (in_features <= 2048) or the down kernel (x staged 512 columns at a time); row-block kernel
// otherwise.
enum MatmulPath { MM_ROWBLOCK = 0, MM_LIN = 1, MM_STAGED = 2 };

static MatmulPath matmul_path(int32_t in_features, const lbk_bell* w) {
  if (w->B != 16 && w->B != 32) return MM_ROWBLOCK;
  if (lin_supported(w->B, in_features, w->R, w->K)) return MM_LIN;
  if (w->K >= 1 && w->K <= 128 && w->R >= 1 && in_features % 8 == 0) return MM_STAGED;
  return MM_ROWBLOCK;
}

size_t lbk_block_ell_matmul_workspace_bytes(int64_t N, int32_t in_features, const lbk_bell* w) {
  if (!w || N <= 0 || in_features <= 0 || check_bell(w) || in_features % w->B) return 0;
  if (matmul_path(in_features, w) == MM_ROWBLOCK) return 0;
  return align256(packed_bf16_bytes((int64_t)w->R * w->K, w->B));
}

// the product on tiles already packed (packed != null) or packed into the workspace
static int matmul_impl(const uint16_t* x, int64_t N, int32_t in_features, const lbk_bell* w, const void* packed,
                       size_t packed_bytes, const float* bias, uint16_t* y, void* workspace, size_t workspace_bytes,
                       hipStream_t s) {
  int st = check_bell(w);
  if (st) return st;
  if (N < 0) return LBK_ERR_ARG;
  if (in_features <= 0 || in_features % w->B) return LBK_ERR_SHAPE;
  if (N == 0) return LBK_OK;
  if (!x || !y) return LBK_ERR_NULL;
  const int64_t out_f = (int64_t)w->R * w->B;
  if (!a16(x) || (in_features % 8) || !a16(y) || (out_f % 8)) return LBK_ERR_ALIGN;
  const MatmulPath path = matmul_path(in_features, w);
  if (path == MM_ROWBLOCK)
    return lbk_block_ell_matmul_bf16(x, N, in_features, in_features, w, bias, y, out_f, s);
  const size_t need = align256(packed_bf16_bytes((int64_t)w->R * w->K, w->B));
  const void* pk = packed;
  if (pk) {
    if (packed_bytes < need) return LBK_ERR_WORKSPACE;
    if (!a16(pk)) return LBK_ERR_ALIGN;
  } else {
    if (!workspace || workspace_bytes < need) return LBK_ERR_WORKSPACE;
    if (!a16(workspace)) return LBK_ERR_ALIGN;
    const int C_in = in_features / w->B;
    PackJob job{w->values, w->col_idx, (int64_t)w->R * w->K, C_in, static_cast<uint32_t*>(workspace), 0,
                path == MM_LIN ? 1 : 0, nullptr, nullptr};
    if (launch_pack_bf16_multi(&job, 1, w->B, s) != 0) return LBK_ERR_LAUNCH;
    pk = workspace;
  }
  const int C_in = in_features / w->B;
  if (path == MM_LIN) {
    GUArgs g{};
    g.x = x; g.N = N; g.d_model = in_features;
    g.pg = pk; g.cg = w->col_idx; g.Kg = w->K;
    g.R_ff = w->R; g.h = y; g.bg = bias;
    return launch_lin(w->B, g, s) == 0 ? LBK_OK : LBK_ERR_LAUNCH;
  }
  DNArgs d{};
  d.h = x; d.N = N; d.d_ff = in_features; d.d_model = (int)out_f;
  d.pd = pk; d.cd = w->col_idx; d.Kd = w->K;
  d.R_m = w->R; d.C_d = C_in;
  d.out = y; d.bd = bias;
  return launch_dn(w->B, d, s) == 0 ? LBK_OK : LBK_ERR_LAUNCH;
}

int lbk_block_ell_matmul_ws_bf16(const uint16_t* x, int64_t N, int32_t in_features, const lbk_bell* w,
                                 const float* bias, uint16_t* y, void* workspace, size_t workspace_bytes,
                                 void* stream) {
  return matmul_impl(x, N, in_features, w, nullptr, 0, bias, y, workspace, workspace_bytes, S(stream));
}

size_t lbk_block_ell_matmul_prepacked_bytes(int32_t in_features, const lbk_bell* w) {
  return lbk_block_ell_matmul_workspace_bytes(1, in_features, w);
}

int lbk_block_ell_matmul_prepack_bf16(int32_t in_features, const lbk_bell* w, void* packed, size_t packed_bytes,
                                      void* stream) {
  int st = check_bell(w);
  if (st) return st;
  if (in_features <= 0 || in_features % w->B) return LBK_ERR_SHAPE;
  const MatmulPath path = matmul_path(in_features, w);
  if (path == MM_ROWBLOCK) return LBK_OK;        // no packed form for this geometry
  if (!packed || packed_bytes < lbk_block_ell_matmul_prepacked_bytes(in_features, w)) return LBK_ERR_WORKSPACE;
  if (!a16(packed)) return LBK_ERR_ALIGN;
  PackJob job{w->values, w->col_idx, (int64_t)w->R * w->K, in_features / w->B, static_cast<uint32_t*>(packed), 0,
              path == MM_LIN ? 1 : 0, nullptr, nullptr};
  return launch_pack_bf16_multi(&job, 1, w->B, S(stream)) == 0 ? LBK_OK : LBK_ERR_LAUNCH;
}

int lbk_block_ell_matmul_prepacked_bf16(const uint16_t* x, int64_t N, int32_t in_features, const lbk_bell* w,
                                        const void* packed, size_t packed_bytes, const float* bias, uint16_t* y,
                                        void* stream) {
  if (!w) return LBK_ERR_NULL;
  if (N > 0 && !packed && lbk_block_ell_matmul_prepacked_bytes(in_features, w) > 0) return LBK_ERR_NULL;
  return matmul_impl(x, N, in_features, w, packed, packed_bytes, bias, y, nullptr, 0, S(stream));
}

static bool use_split(const lbk_bell* gate, const lbk_bell* up, const lbk_bell* down, int32_t d_model) {
  return split_supported(gate->B, d_model, gate->R, down->R, gate->K, up->K, down->K);
}

// Packed copies of gate/up/down (fragment-major tiles) at the start of a workspace.
struct PackedFFN {
  const void* g; const void* u; const void* d;
  size_t bytes;
};

static size_t packed_ffn_bytes(const lbk_bell* gate, const lbk_bell* up, const lbk_bell* down) {
  const int B = gate->B;
  return align256(packed_bf16_bytes((int64_t)gate->R * gate->K, B)) +
         align256(packed_bf16_bytes((int64_t)up->R * up->K, B)) +
         align256(packed_bf16_bytes((int64_t)down->R * down->K, B));
}

// the three parts of a copy made by lbk_swiglu_prepack_bf16
static PackedFFN packed_ffn_at(const char* p, const lbk_bell* gate, const lbk_bell* up) {
  PackedFFN pk{};
  pk.g = p;
  p += align256(packed_bf16_bytes((int64_t)gate->R * gate->K, gate->B));
  pk.u = p;
  pk.d = p + align256(packed_bf16_bytes((int64_t)up->R * up->K, gate->B));
  return pk;
}

// fp32 master tiles of gate, up and down and the buffers of their bf16 copies
struct MasterFFN {
  const float* v[3];
  uint16_t* raw[3];
};

static int pack_ffn(const lbk_bell* gate, const lbk_bell* up, const lbk_bell* down, char* ws, PackedFFN* out,
                    hipStream_t st, const MasterFFN* master = nullptr) {
  const int B = gate->B;
  char* p = ws;
  const lbk_bell* ws3[3] = {gate, up, down};
  const void** dst[3] = {&out->g, &out->u, &out->d};
  const int cols[3] = {down->R, down->R, gate->R};   // input column blocks: d_model / B, d_model / B, d_ff / B
  PackJob jobs[3];
  for (int t = 0; t < 3; ++t) {
    const int64_t nt = (int64_t)ws3[t]->R * ws3[t]->K;
    *dst[t] = p;
    jobs[t] = PackJob{ws3[t]->values, ws3[t]->col_idx, nt, cols[t], reinterpret_cast<uint32_t*>(p), 0, t < 2,
                      master ? master->v[t] : nullptr, master ? master->raw[t] : nullptr};
    p += align256(packed_bf16_bytes(nt, B));
  }
  out->bytes = (size_t)(p - ws);
  return launch_pack_bf16_multi(jobs, 3, B, st) == 0 ? LBK_OK : LBK_ERR_LAUNCH;
}

static int swiglu_split(const uint16_t* x, const float* xf, const float* norm_scale, float eps, int64_t N,
                        int32_t d_model, const lbk_bell* gate, const lbk_bell* up, const lbk_bell* down,
                        const PackedFFN& pk, const uint16_t* resid, float* state, uint16_t* out, uint16_t* h,
                        uint16_t* gate_pre, uint16_t* up_out, hipStream_t st, Biases bs = {}) {
  GUArgs g{};
  g.x = x; g.xf = xf; g.N = N; g.d_model = d_model; g.norm_scale = norm_scale; g.eps = eps;
  g.pg = pk.g; g.cg = gate->col_idx; g.Kg = gate->K;
  g.pu = pk.u; g.cu = up->col_idx; g.Ku = up->K;
  g.R_ff = gate->R;
  g.h = h; g.gpre = gate_pre; g.uout = up_out; g.bg = bs.g; g.bu = bs.u;
  if (launch_gu(gate->B, xf != nullptr, g, st) != 0) return LBK_ERR_LAUNCH;
  DNArgs d{};
  d.h = h; d.N = N; d.d_ff = (int64_t)gate->R * gate->B; d.d_model = d_model;
  d.pd = pk.d; d.cd = down->col_idx; d.Kd = down->K;
  d.R_m = down->R; d.C_d = gate->R;
  d.resid = resid; d.state = state; d.out = out; d.bd = bs.d;
  return launch_dn(gate->B, d, st) == 0 ? LBK_OK : LBK_ERR_LAUNCH;
}

// ---- decode shape (N <= 64): gate/up and down kernels of lbk_decode.hip
static constexpr int64_t kDecodeMaxTokens = 64;

static bool use_decode(int64_t N, const lbk_bell* gate, const lbk_bell* up, const lbk_bell* down, bool inter) {
  // the decode kernels read down tiles (and the prefetch reads them) with 16-byte loads
  return !inter && N <= kDecodeMaxTokens && decode_supported(gate->K, up->K, down->K) && a16(down->values);
}

size_t lbk_swiglu_workspace_bytes(int64_t N, int32_t d_model, const lbk_bell* gate, const lbk_bell* up,
                                  const lbk_bell* down, int want_intermediates) {
  if (!gate || !up || !down || N <= 0) return 0;
  // [packed gate/up/down tiles (split path)] [h, unless it goes to the caller's h_out]
  size_t b = use_split(gate, up, down, d_model) ? packed_ffn_bytes(gate, up, down) : 0;
  if (!want_intermediates) b += align256((size_t)N * gate->R * gate->B * 2);
  // decode shapes need h only
  if (use_decode(N, gate, up, down, want_intermediates != 0)) return align256((size_t)N * gate->R * gate->B * 2);
  return b;
}

int lbk_swiglu_forward_path(int64_t N, int32_t d_model, const lbk_bell* gate, const lbk_bell* up,
                            const lbk_bell* down, int want_intermediates) {
  if (!gate || !up || !down || N <= 0) return LBK_PATH_NONE;
  if (check_bell(gate) || check_bell(up) || check_bell(down)) return LBK_PATH_NONE;
  int64_t d_ff = 0;
  if (check_ffn(gate, up, down, d_model, &d_ff)) return LBK_PATH_NONE;
  if (use_decode(N, gate, up, down, want_intermediates != 0)) return LBK_PATH_DECODE;
  return use_split(gate, up, down, d_model) ? LBK_PATH_SPLIT : LBK_PATH_ROWBLOCK;
}

int lbk_swiglu_fwd_bf16(const uint16_t* x, int64_t N, int32_t d_model, const lbk_bell* gate, const lbk_bell* up,
                        const lbk_bell* down, int add_residual, uint16_t* out, uint16_t* h_out,
                        uint16_t* gate_pre_out, uint16_t* up_out, void* workspace, size_t workspace_bytes,
                        void* stream) {
  return lbk_swiglu_fwd_bias_bf16(x, N, d_model, gate, up, down, nullptr, nullptr, nullptr, add_residual, out, h_out,
                                  gate_pre_out, up_out, workspace, workspace_bytes, stream);
}

// The forward behind lbk_swiglu_fwd_bias_bf16 and lbk_swiglu_fwd_prepacked_bf16: `prepacked`
// (may be null) holds the packed tiles of lbk_swiglu_prepack_bf16, otherwise the two-kernel
// path packs into the workspace.
static int swiglu_fwd_impl(const uint16_t* x, int64_t N, int32_t d_model, const lbk_bell* gate, const lbk_bell* up,
                           const lbk_bell* down, const char* prepacked, size_t prepacked_bytes, Biases bs,
                           int add_residual, uint16_t* out, uint16_t* h_out, uint16_t* gate_pre_out,
                           uint16_t* up_out, void* workspace, size_t workspace_bytes, hipStream_t s,
                           const MasterFFN* master = nullptr) {
  int st;
  if ((st = check_bell(gate)) || (st = check_bell(up)) || (st = check_bell(down))) return st;
  int64_t d_ff = 0;
  if ((st = check_ffn(gate, up, down, d_model, &d_ff))) return st;
  if (N < 0) return LBK_ERR_ARG;
  if (N == 0) return LBK_OK;
  if (!x || !out) return LBK_ERR_NULL;
  if (!a16(x) || !a16(out) || (d_model % 8)) return LBK_ERR_ALIGN;
  for (const void* p : {(const void*)h_out, (const void*)gate_pre_out, (const void*)up_out})
    if (p && !a16(p)) return LBK_ERR_ALIGN;
  const bool split = use_split(gate, up, down, d_model);
  const size_t pbytes = split ? packed_ffn_bytes(gate, up, down) : 0;
  // a packed copy is checked whatever path the token count selects (the decode kernels read the
  // raw tiles and do not use it)
  if (split && prepacked) {
    if (prepacked_bytes < pbytes) return LBK_ERR_WORKSPACE;
    if (!a16(prepacked)) return LBK_ERR_ALIGN;
  }
  if (use_decode(N, gate, up, down, gate_pre_out || up_out)) {
    uint16_t* hbuf = h_out;
    if (!hbuf) {
      if (!workspace || workspace_bytes < align256((size_t)N * d_ff * 2)) return LBK_ERR_WORKSPACE;
      if (!a16(workspace)) return LBK_ERR_ALIGN;
      hbuf = static_cast<uint16_t*>(workspace);
    }
    DecodeArgs a{};
    a.x = x; a.N = (int)N; a.d_model = d_model;
    a.vg = gate->values; a.cg = gate->col_idx; a.Kg = gate->K;
    a.vu = up->values; a.cu = up->col_idx; a.Ku = up->K;
    a.R_ff = gate->R;
    a.vd = down->values; a.cd = down->col_idx; a.Kd = down->K;
    a.R_m = down->R;
    a.resid = add_residual ? x : nullptr;
    a.out = out;
    a.h = hbuf;
    a.bg = bs.g; a.bu = bs.u; a.bd = bs.d;
    return launch_decode(gate->B, a, s) == 0 ? LBK_OK : LBK_ERR_LAUNCH;
  }
  const size_t own = (split && !prepacked) ? pbytes : 0;     // packed tiles built by this call
  const size_t hbytes = h_out ? 0 : align256((size_t)N * d_ff * 2);
  if (own + hbytes > 0) {
    if (!workspace || workspace_bytes < own + hbytes) return LBK_ERR_WORKSPACE;
    if (!a16(workspace)) return LBK_ERR_ALIGN;
  }
  char* ws = static_cast<char*>(workspace);
  uint16_t* h = h_out ? h_out : reinterpret_cast<uint16_t*>(ws + own);
  if (split) {
    PackedFFN pk{};
    if (prepacked) {
      pk = packed_ffn_at(prepacked, gate, up);
    } else if ((st = pack_ffn(gate, up, down, ws, &pk, s, master))) {
      return st;
    }
    return swiglu_split(x, nullptr, nullptr, 0.f, N, d_model, gate, up, down, pk, add_residual ? x : nullptr,
                        nullptr, out, h, gate_pre_out, up_out, s, bs);
  }
  return swiglu_general(x, N, d_model, gate, up, down, add_residual ? x : nullptr, out, h, gate_pre_out, up_out, s,
                        bs);
}

// a bf16 copy of fp32 tiles without a packed form (the geometries that read the raw tiles)
static int cast_ffn(const lbk_bell* gate, const lbk_bell* up, const lbk_bell* down, const MasterFFN& m,
                    hipStream_t s) {
  const lbk_bell* w3[3] = {gate, up, down};
  PackJob jobs[3];
  int n = 0;
  for (int t = 0; t < 3; ++t) {
    const int64_t nt = (int64_t)w3[t]->R * w3[t]->K;
    if (nt > 0) jobs[n++] = PackJob{nullptr, w3[t]->col_idx, nt, 0, nullptr, 0, 0, m.v[t], m.raw[t]};
  }
  return n == 0 || launch_pack_bf16_multi(jobs, n, gate->B, s) == 0 ? LBK_OK : LBK_ERR_LAUNCH;
}

int lbk_swiglu_fwd_train(const uint16_t* x, int64_t N, int32_t d_model, const lbk_bell* gate, const lbk_bell* up,
                         const lbk_bell* down, const float* v_gate, const float* v_up, const float* v_down,
                         uint16_t* vb_gate, uint16_t* vb_up, uint16_t* vb_down, const float* b_gate,
                         const float* b_up, const float* b_down, int add_residual, uint16_t* out, uint16_t* h_out,
                         uint16_t* gate_pre_out, uint16_t* up_out, void* workspace, size_t workspace_bytes,
                         void* stream) {
  if (!gate || !up || !down) return LBK_ERR_NULL;
  const MasterFFN m{{v_gate, v_up, v_down}, {vb_gate, vb_up, vb_down}};
  lbk_bell w3[3] = {*gate, *up, *down};
  int st;
  for (int t = 0; t < 3; ++t) {
    w3[t].values = m.raw[t];
    if ((st = check_bell(&w3[t]))) return st;
    if ((int64_t)w3[t].R * w3[t].K > 0) {
      if (!m.v[t]) return LBK_ERR_NULL;
      if (!a16(m.v[t]) || !a16(m.raw[t])) return LBK_ERR_ALIGN;
    }
  }
  int64_t d_ff = 0;
  if ((st = check_ffn(&w3[0], &w3[1], &w3[2], d_model, &d_ff))) return st;
  if (N < 0) return LBK_ERR_ARG;
  if (N > 0 && (!h_out || !gate_pre_out || !up_out)) return LBK_ERR_NULL;
  // without a packed form (or without tokens) only the copies are written, before the products read them
  if (N == 0 || !use_split(&w3[0], &w3[1], &w3[2], d_model)) {
    if ((st = cast_ffn(&w3[0], &w3[1], &w3[2], m, S(stream)))) return st;
  }
  return swiglu_fwd_impl(x, N, d_model, &w3[0], &w3[1], &w3[2], nullptr, 0, Biases{b_gate, b_up, b_down}, add_residual,
                         out, h_out, gate_pre_out, up_out, workspace, workspace_bytes, S(stream), &m);
}

int lbk_swiglu_fwd_bias_bf16(const uint16_t* x, int64_t N, int32_t d_model, const lbk_bell* gate,
                             const lbk_bell* up, const lbk_bell* down, const float* b_gate, const float* b_up,
                             const float* b_down, int add_residual, uint16_t* out, uint16_t* h_out,
                             uint16_t* gate_pre_out, uint16_t* up_out, void* workspace, size_t workspace_bytes,
                             void* stream) {
  return swiglu_fwd_impl(x, N, d_model, gate, up, down, nullptr, 0, Biases{b_gate, b_up, b_down}, add_residual, out,
                         h_out, gate_pre_out, up_out, workspace, workspace_bytes, S(stream));
}

size_t lbk_swiglu_prepacked_bytes(int32_t d_model, const lbk_bell* gate, const lbk_bell* up, const lbk_bell* down) {
  if (!gate || !up || !down || d_model <= 0) return 0;
  if (check_bell(gate) || check_bell(up) || check_bell(down)) return 0;
  int64_t d_ff = 0;
  if (check_ffn(gate, up, down, d_model, &d_ff)) return 0;
  return use_split(gate, up, down, d_model) ? packed_ffn_bytes(gate, up, down) : 0;
}

int lbk_swiglu_prepack_bf16(int32_t d_model, const lbk_bell* gate, const lbk_bell* up, const lbk_bell* down,
                            void* packed, size_t packed_bytes, void* stream) {
  int st;
  if ((st = check_bell(gate)) || (st = check_bell(up)) || (st = check_bell(down))) return st;
  int64_t d_ff = 0;
  if ((st = check_ffn(gate, up, down, d_model, &d_ff))) return st;
  if (!use_split(gate, up, down, d_model)) return LBK_OK;        // no packed form for this geometry
  if (!packed || packed_bytes < packed_ffn_bytes(gate, up, down)) return LBK_ERR_WORKSPACE;
  if (!a16(packed)) return LBK_ERR_ALIGN;
  PackedFFN pk{};
  return pack_ffn(gate, up, down, static_cast<char*>(packed), &pk, S(stream));
}

size_t lbk_swiglu_prepacked_workspace_bytes(int64_t N, int32_t d_model, const lbk_bell* gate, const lbk_bell* up,
                                            const lbk_bell* down, int want_intermediates) {
  if (!gate || !up || !down || N <= 0) return 0;
  if (use_decode(N, gate, up, down, want_intermediates != 0)) return align256((size_t)N * gate->R * gate->B * 2);
  if (!use_split(gate, up, down, d_model)) return lbk_swiglu_workspace_bytes(N, d_model, gate, up, down,
                                                                             want_intermediates);
  return want_intermediates ? 0 : align256((size_t)N * gate->R * gate->B * 2);
}

int lbk_swiglu_fwd_prepacked_bf16(const uint16_t* x, int64_t N, int32_t d_model, const lbk_bell* gate,
                                  const lbk_bell* up, const lbk_bell* down, const void* packed, size_t packed_bytes,
                                  const float* b_gate, const float* b_up, const float* b_down, int add_residual,
                                  uint16_t* out, uint16_t* h_out, uint16_t* gate_pre_out, uint16_t* up_out,
                                  void* workspace, size_t workspace_bytes, void* stream) {
  if (!gate || !up || !down) return LBK_ERR_NULL;
  if (use_split(gate, up, down, d_model) && !packed && N > 0) return LBK_ERR_NULL;
  return swiglu_fwd_impl(x, N, d_model, gate, up, down, static_cast<const char*>(packed), packed_bytes,
                         Biases{b_gate, b_up, b_down}, add_residual, out, h_out, gate_pre_out, up_out, workspace,
                         workspace_bytes, S(stream));
}

int lbk_rmsnorm_bf16(const uint16_t* x, int64_t N, int32_t d, const float* scale, float eps, uint16_t* out,
                     void* stream) {
  if (N < 0 || d <= 0 || !(eps >= 0.f)) return LBK_ERR_ARG;
  if (N == 0) return LBK_OK;
  if (!x || !scale || !out) return LBK_ERR_NULL;
  return launch_rmsnorm(x, N, d, scale, eps, out, S(stream)) == 0 ? LBK_OK : LBK_ERR_LAUNCH;
}

size_t lbk_rmsnorm_bwd_workspace_bytes(int64_t N, int32_t d) {
  if (N < 0 || d <= 0) return 0;
  return align256(rmsnorm_bwd_bytes(N, d));
}

int lbk_rmsnorm_bwd_bf16(const uint16_t* x, const uint16_t* dy, int64_t N, int32_t d, const float* scale, float eps,
                         uint16_t* dx, float* dscale, void* workspace, size_t workspace_bytes, void* stream) {
  if (N < 0 || d <= 0 || !(eps >= 0.f)) return LBK_ERR_ARG;
  if (!scale || !dscale) return LBK_ERR_NULL;
  if (N > 0 && (!x || !dy || !dx)) return LBK_ERR_NULL;
  const size_t need = lbk_rmsnorm_bwd_workspace_bytes(N, d);
  if (need > 0 && (!workspace || workspace_bytes < need)) return LBK_ERR_WORKSPACE;
  return launch_rmsnorm_bwd(x, dy, N, d, scale, eps, dx, dscale, static_cast<float*>(workspace), S(stream)) == 0
             ? LBK_OK
             : LBK_ERR_LAUNCH;
}

int lbk_diagonal_injection_bf16(const uint16_t* h, const uint16_t* e, const float* log_A, const float* log_dt,
                                int64_t N, int32_t d, uint16_t* h_out, void* stream) {
  if (N < 0 || d <= 0) return LBK_ERR_ARG;
  if (N == 0) return LBK_OK;
  if (!h || !e || !log_A || !log_dt || !h_out) return LBK_ERR_NULL;
  return launch_injection(h, e, log_A, log_dt, N, d, h_out, S(stream)) == 0 ? LBK_OK : LBK_ERR_LAUNCH;
}

size_t lbk_diagonal_injection_bwd_workspace_bytes(int64_t N, int32_t d) {
  if (N < 0 || d <= 0) return 0;
  return align256(injection_bwd_bytes(N, d));
}

int lbk_diagonal_injection_bwd_bf16(const uint16_t* grad_out, const uint16_t* h, const uint16_t* e,
                                    const float* log_A, const float* log_dt, int64_t N, int32_t d, uint16_t* dh,
                                    uint16_t* de, float* d_log_A, float* d_log_dt, void* workspace,
                                    size_t workspace_bytes, void* stream) {
  if (N < 0 || d <= 0) return LBK_ERR_ARG;
  if (!log_A || !log_dt) return LBK_ERR_NULL;
  if (N > 0 && (!grad_out || !h || !e)) return LBK_ERR_NULL;
  const size_t need = lbk_diagonal_injection_bwd_workspace_bytes(N, d);
  if (need > 0 && (!workspace || workspace_bytes < need)) return LBK_ERR_WORKSPACE;
  return launch_injection_bwd(grad_out, h, e, log_A, log_dt, N, d, dh, de, d_log_A, d_log_dt,
                              static_cast<float*>(workspace), S(stream)) == 0
             ? LBK_OK
             : LBK_ERR_LAUNCH;
}

size_t lbk_looped_workspace_bytes(int64_t N, int32_t d_model, const lbk_bell* gate, const lbk_bell* up,
                                  const lbk_bell* down) {
  if (!gate || !up || !down || N <= 0 || d_model <= 0) return 0;
  // [fp32 carried state (or the bf16 normed copy on the general path)] [h] [packed tiles]
  return align256((size_t)N * d_model * 4) + align256((size_t)N * gate->R * gate->B * 2) +
         (use_split(gate, up, down, d_model) ? packed_ffn_bytes(gate, up, down) : 0);
}

static int looped_persistent(const uint16_t* h_in, int64_t N, int32_t d_model, const float* norm_scale, float eps,
                             int32_t L, const lbk_bell* gate, const lbk_bell* up, const lbk_bell* down,
                             uint16_t* h_out, void* workspace, size_t workspace_bytes, void* stream, Biases bs);
static int looped_launches(const uint16_t* h_in, int64_t N, int32_t d_model, const float* norm_scale, float eps,
                           int32_t L, const lbk_bell* gate, const lbk_bell* up, const lbk_bell* down,
                           uint16_t* h_out, void* workspace, size_t workspace_bytes, void* stream, Biases bs);

int lbk_looped_swiglu_bf16(const uint16_t* h_in, int64_t N, int32_t d_model, const float* norm_scale, float eps,
                           int32_t L, const lbk_bell* gate, const lbk_bell* up, const lbk_bell* down,
                           uint16_t* h_out, void* workspace, size_t workspace_bytes, void* stream) {
  return lbk_looped_swiglu_bias_bf16(h_in, N, d_model, norm_scale, eps, L, gate, up, down, nullptr, nullptr, nullptr,
                                     h_out, workspace, workspace_bytes, stream);
}

int lbk_looped_swiglu_bias_bf16(const uint16_t* h_in, int64_t N, int32_t d_model, const float* norm_scale,
                                float eps, int32_t L, const lbk_bell* gate, const lbk_bell* up, const lbk_bell* down,
                                const float* b_gate, const float* b_up, const float* b_down, uint16_t* h_out,
                                void* workspace, size_t workspace_bytes, void* stream) {
  const Biases bs{b_gate, b_up, b_down};
  // the per-iteration launches: measured faster than the persistent launch at every token count
  // tried (d_model 1024, d_ff 4096, B = 32, L = 8: 0.21 against 1.20 ms at N = 64, 0.59 against
  // 1.21 at N = 4096, 1.29 against 1.34 at N = 16384); the persistent launch is its own entry point
  return looped_launches(h_in, N, d_model, norm_scale, eps, L, gate, up, down, h_out, workspace, workspace_bytes,
                         stream, bs);
}

int lbk_looped_swiglu_launches_bf16(const uint16_t* h_in, int64_t N, int32_t d_model, const float* norm_scale,
                                    float eps, int32_t L, const lbk_bell* gate, const lbk_bell* up,
                                    const lbk_bell* down, uint16_t* h_out, void* workspace, size_t workspace_bytes,
                                    void* stream) {
  return looped_launches(h_in, N, d_model, norm_scale, eps, L, gate, up, down, h_out, workspace, workspace_bytes,
                         stream, Biases{});
}

static int looped_launches(const uint16_t* h_in, int64_t N, int32_t d_model, const float* norm_scale, float eps,
                           int32_t L, const lbk_bell* gate, const lbk_bell* up, const lbk_bell* down,
                           uint16_t* h_out, void* workspace, size_t workspace_bytes, void* stream, Biases bs) {
  int st;
  if ((st = check_bell(gate)) || (st = check_bell(up)) || (st = check_bell(down))) return st;
  int64_t d_ff = 0;
  if ((st = check_ffn(gate, up, down, d_model, &d_ff))) return st;
  if (N < 0 || L < 0 || !(eps >= 0.f)) return LBK_ERR_ARG;
  if (N == 0) return LBK_OK;
  if (!h_in || !h_out || !norm_scale) return LBK_ERR_NULL;
  if (!a16(h_in) || !a16(h_out) || (d_model % 8)) return LBK_ERR_ALIGN;
  hipStream_t s = S(stream);
  if (L == 0) {
    if (h_out != h_in &&
        hipMemcpyAsync(h_out, h_in, (size_t)N * d_model * 2, hipMemcpyDeviceToDevice, s) != hipSuccess)
      return LBK_ERR_LAUNCH;
    return LBK_OK;
  }
  const bool split = use_split(gate, up, down, d_model) && a16(norm_scale);
  const size_t sbytes = align256((size_t)N * d_model * 4), hbytes = align256((size_t)N * d_ff * 2);
  const size_t pbytes = use_split(gate, up, down, d_model) ? packed_ffn_bytes(gate, up, down) : 0;
  if (!workspace || workspace_bytes < sbytes + hbytes + pbytes) return LBK_ERR_WORKSPACE;
  if (!a16(workspace)) return LBK_ERR_ALIGN;
  char* ws = static_cast<char*>(workspace);
  uint16_t* h = reinterpret_cast<uint16_t*>(ws + sbytes);
  if (split && N <= kDecodeMaxTokens && decode_supported(gate->K, up->K, down->K) && a16(down->values) &&
      pbytes >= align256((size_t)N * d_model * 2)) {
    // decode-sized token counts: per application the RMSNorm of the fp32 state into bf16 rows
    // (in the packed weights' part of the workspace, which this path does not use), then the
    // decode kernels, whose down kernel adds the product to the state
    float* state = reinterpret_cast<float*>(ws);
    uint16_t* xn = reinterpret_cast<uint16_t*>(ws + sbytes + hbytes);
    if (launch_bf16_to_f32(h_in, N * d_model, state, s) != 0) return LBK_ERR_LAUNCH;
    DecodeArgs a{};
    a.x = xn; a.N = (int)N; a.d_model = d_model;
    a.vg = gate->values; a.cg = gate->col_idx; a.Kg = gate->K;
    a.vu = up->values; a.cu = up->col_idx; a.Ku = up->K;
    a.R_ff = gate->R;
    a.vd = down->values; a.cd = down->col_idx; a.Kd = down->K;
    a.R_m = down->R;
    a.h = h; a.state = state;
    a.bg = bs.g; a.bu = bs.u; a.bd = bs.d;
    for (int l = 0; l < L; ++l) {
      if (launch_rmsnorm_f32(state, N, d_model, norm_scale, eps, xn, s) != 0) return LBK_ERR_LAUNCH;
      a.out = l == L - 1 ? h_out : nullptr;
      if (launch_decode(gate->B, a, s) != 0) return LBK_ERR_LAUNCH;
    }
    return LBK_OK;
  }
  if (split) {
    // fp32 state carried across the L applications; bf16 written once, after the last
    float* state = reinterpret_cast<float*>(ws);
    PackedFFN pk{};
    if ((st = pack_ffn(gate, up, down, ws + sbytes + hbytes, &pk, s))) return st;
    if (launch_bf16_to_f32(h_in, N * d_model, state, s) != 0) return LBK_ERR_LAUNCH;
    for (int l = 0; l < L; ++l)
      if ((st = swiglu_split(nullptr, state, norm_scale, eps, N, d_model, gate, up, down, pk, nullptr, state,
                             l == L - 1 ? h_out : nullptr, h, nullptr, nullptr, s, bs)))
        return st;
    return LBK_OK;
  }
  uint16_t* normed = reinterpret_cast<uint16_t*>(ws);
  const uint16_t* cur = h_in;
  for (int l = 0; l < L; ++l) {
    if (launch_rmsnorm(cur, N, d_model, norm_scale, eps, normed, s) != 0) return LBK_ERR_LAUNCH;
    if ((st = swiglu_general(normed, N, d_model, gate, up, down, cur, h_out, h, nullptr, nullptr, s, bs))) return st;
    cur = h_out;
  }
  return LBK_OK;
}

int lbk_looped_swiglu_persistent_bf16(const uint16_t* h_in, int64_t N, int32_t d_model, const float* norm_scale,
                                      float eps, int32_t L, const lbk_bell* gate, const lbk_bell* up,
                                      const lbk_bell* down, uint16_t* h_out, void* workspace,
                                      size_t workspace_bytes, void* stream) {
  return looped_persistent(h_in, N, d_model, norm_scale, eps, L, gate, up, down, h_out, workspace, workspace_bytes,
                           stream, Biases{});
}

static int looped_persistent(const uint16_t* h_in, int64_t N, int32_t d_model, const float* norm_scale, float eps,
                             int32_t L, const lbk_bell* gate, const lbk_bell* up, const lbk_bell* down,
                             uint16_t* h_out, void* workspace, size_t workspace_bytes, void* stream, Biases bs) {
  int st;
  if ((st = check_bell(gate)) || (st = check_bell(up)) || (st = check_bell(down))) return st;
  int64_t d_ff = 0;
  if ((st = check_ffn(gate, up, down, d_model, &d_ff))) return st;
  if (N < 0 || L < 0 || !(eps >= 0.f)) return LBK_ERR_ARG;
  if (!looped_persistent_supported(gate->B, d_model, gate->R, down->R, gate->K, up->K, down->K)) return LBK_ERR_SHAPE;
  if (N == 0) return LBK_OK;
  if (!h_in || !h_out || !norm_scale) return LBK_ERR_NULL;
  if (!a16(h_in) || !a16(h_out) || !a16(norm_scale)) return LBK_ERR_ALIGN;
  hipStream_t s = S(stream);
  if (L == 0) {
    if (h_out != h_in &&
        hipMemcpyAsync(h_out, h_in, (size_t)N * d_model * 2, hipMemcpyDeviceToDevice, s) != hipSuccess)
      return LBK_ERR_LAUNCH;
    return LBK_OK;
  }
  const size_t sbytes = align256((size_t)N * d_model * 4), hbytes = align256((size_t)N * d_ff * 2);
  const size_t pbytes = packed_ffn_bytes(gate, up, down);
  if (!workspace || workspace_bytes < sbytes + hbytes + pbytes) return LBK_ERR_WORKSPACE;
  if (!a16(workspace)) return LBK_ERR_ALIGN;
  char* ws = static_cast<char*>(workspace);
  float* state = reinterpret_cast<float*>(ws);
  uint16_t* h = reinterpret_cast<uint16_t*>(ws + sbytes);
  PackedFFN pk{};
  if ((st = pack_ffn(gate, up, down, ws + sbytes + hbytes, &pk, s))) return st;
  LoopArgs la{};
  la.gu.xf = state; la.gu.N = N; la.gu.d_model = d_model; la.gu.eps = eps;
  la.gu.R_ff = gate->R; la.gu.h = h;
  la.dn.h = h; la.dn.N = N; la.dn.d_ff = d_ff; la.dn.d_model = d_model;
  la.dn.R_m = down->R; la.dn.C_d = gate->R; la.dn.state = state; la.dn.out = h_out;
  la.h_in = h_in; la.L = L;
  la.n_core = 1;
  la.core[0] = CoreW{pk.g, pk.u, pk.d, gate->col_idx, up->col_idx, down->col_idx, gate->K, down->K, norm_scale,
                     bs.g, bs.u, bs.d};
  // h_out may alias h_in: the kernel reads a token block's h_in rows before any write to them
  return launch_looped(gate->B, la, s) == 0 ? LBK_OK : LBK_ERR_LAUNCH;
}

// ---- looped core: injection -> n_core blocks -> depth freeze, L iterations
enum { CORE_DECODE = 1, CORE_SPLIT = 2, CORE_GENERAL = 3 };
struct CorePlan {
  int path;
  int64_t d_ff;                 // widest d_ff of the blocks
  size_t state, h, tdep, coef, xn, y, packed[LBK_MAX_CORE_BLOCKS], total;
};

// validates the blocks and lays out the workspace:
// [fp32 state][h][per-token depths][injection coefficients][xn, y (decode / row-block paths) or
// the packed tiles of every block (two-kernel path)]
static int core_plan(int64_t N, int32_t d_model, int32_t n_core, const lbk_core_block* blocks, CorePlan* p) {
  if (!blocks) return LBK_ERR_NULL;
  if (n_core < 1 || n_core > LBK_MAX_CORE_BLOCKS || N < 0 || d_model <= 0) return LBK_ERR_ARG;
  *p = CorePlan{};
  bool dec = N <= kDecodeMaxTokens, split = true;
  for (int c = 0; c < n_core; ++c) {
    const lbk_core_block& b = blocks[c];
    int st;
    if ((st = check_bell(&b.gate)) || (st = check_bell(&b.up)) || (st = check_bell(&b.down))) return st;
    int64_t d_ff = 0;
    if ((st = check_ffn(&b.gate, &b.up, &b.down, d_model, &d_ff))) return st;
    if (!b.norm_scale) return LBK_ERR_NULL;
    p->d_ff = d_ff > p->d_ff ? d_ff : p->d_ff;
    dec = dec && use_decode(N, &b.gate, &b.up, &b.down, false);
    split = split && use_split(&b.gate, &b.up, &b.down, d_model) && a16(b.norm_scale);
  }
  p->path = dec ? CORE_DECODE : (split ? CORE_SPLIT : CORE_GENERAL);
  p->state = align256((size_t)N * d_model * 4);
  p->h = align256((size_t)N * p->d_ff * 2);
  p->tdep = align256((size_t)N * 4);
  p->coef = align256((size_t)d_model * 8);
  // after the fixed part: the packed tiles (two-kernel path, and the persistent form of any
  // two-kernel geometry) or xn and y (decode and row-block paths), whichever is larger
  size_t packed = 0, rows = 0;
  if (split) {
    for (int c = 0; c < n_core; ++c) {
      p->packed[c] = packed_ffn_bytes(&blocks[c].gate, &blocks[c].up, &blocks[c].down);
      packed += p->packed[c];
    }
  }
  if (p->path != CORE_SPLIT) {
    p->xn = p->y = align256((size_t)N * d_model * 2);
    rows = p->xn + p->y;
  }
  p->total = p->state + p->h + p->tdep + p->coef + (packed > rows ? packed : rows);
  return LBK_OK;
}

size_t lbk_looped_core_workspace_bytes(int64_t N, int32_t d_model, int32_t n_core, const lbk_core_block* blocks) {
  CorePlan p{};
  if (N <= 0 || core_plan(N, d_model, n_core, blocks, &p)) return 0;
  return p.total;
}

static int looped_core_impl(const uint16_t* h_in, const uint16_t* e, const float* log_A, const float* log_dt,
                            int64_t N, int32_t d_model, int32_t n_core, const lbk_core_block* blocks, float eps,
                            int32_t L, const int32_t* depths, int64_t seq_len, uint16_t* h_out, void* workspace,
                            size_t workspace_bytes, hipStream_t s, bool persistent) {
  CorePlan p{};
  int st;
  if ((st = core_plan(N, d_model, n_core, blocks, &p))) return st;
  if (L < 0 || !(eps >= 0.f) || (depths && seq_len < 1)) return LBK_ERR_ARG;
  if (e && (!log_A || !log_dt)) return LBK_ERR_NULL;
  if (persistent) {
    // one kernel for every block: the same tile size, the persistent launch's shapes
    const int B = blocks[0].gate.B;
    int kmax = 0;
    for (int c = 0; c < n_core; ++c) {
      const lbk_core_block& b = blocks[c];
      if (b.gate.B != B || b.gate.R != blocks[0].gate.R || !a16(b.norm_scale)) return LBK_ERR_SHAPE;
      if (!looped_persistent_supported(B, d_model, b.gate.R, b.down.R, b.gate.K, b.up.K, b.down.K))
        return LBK_ERR_SHAPE;
      kmax = b.gate.K > kmax ? b.gate.K : kmax;
      // one kernel for every block: all or none share their gate/up column buffer
      if ((b.gate.col_idx == b.up.col_idx) != (blocks[0].gate.col_idx == blocks[0].up.col_idx)) return LBK_ERR_SHAPE;
    }
    if (!looped_persistent_supported(B, d_model, blocks[0].gate.R, blocks[0].down.R, kmax, kmax, 1))
      return LBK_ERR_SHAPE;
    p.path = CORE_SPLIT;
  }
  if (N == 0) return LBK_OK;
  if (!h_in || !h_out) return LBK_ERR_NULL;
  if (!a16(h_in) || !a16(h_out) || (e && !a16(e)) || (d_model % 8)) return LBK_ERR_ALIGN;
  if (L == 0) {
    if (h_out != h_in &&
        hipMemcpyAsync(h_out, h_in, (size_t)N * d_model * 2, hipMemcpyDeviceToDevice, s) != hipSuccess)
      return LBK_ERR_LAUNCH;
    return LBK_OK;
  }
  if (!workspace || workspace_bytes < p.total) return LBK_ERR_WORKSPACE;
  if (!a16(workspace)) return LBK_ERR_ALIGN;
  char* ws = static_cast<char*>(workspace);
  float* state = reinterpret_cast<float*>(ws);
  uint16_t* h = reinterpret_cast<uint16_t*>(ws + p.state);
  int32_t* tdepth = depths ? reinterpret_cast<int32_t*>(ws + p.state + p.h) : nullptr;
  float* coef = e ? reinterpret_cast<float*>(ws + p.state + p.h + p.tdep) : nullptr;
  char* rest = ws + p.state + p.h + p.tdep + p.coef;
  if (launch_core_prep(log_A, log_dt, d_model, coef, depths, seq_len, N, tdepth, s) != 0) return LBK_ERR_LAUNCH;

  if (p.path == CORE_SPLIT) {
    PackedFFN pk[LBK_MAX_CORE_BLOCKS];
    for (int c = 0; c < n_core; ++c) {
      if ((st = pack_ffn(&blocks[c].gate, &blocks[c].up, &blocks[c].down, rest, &pk[c], s))) return st;
      rest += p.packed[c];
    }
    if (persistent) {
      LoopArgs la{};
      la.gu.xf = state; la.gu.N = N; la.gu.d_model = d_model; la.gu.eps = eps;
      la.gu.R_ff = blocks[0].gate.R; la.gu.h = h;
      la.dn.h = h; la.dn.N = N; la.dn.d_ff = p.d_ff; la.dn.d_model = d_model;
      la.dn.R_m = blocks[0].down.R; la.dn.C_d = blocks[0].gate.R; la.dn.state = state; la.dn.out = h_out;
      la.h_in = h_in; la.L = L; la.n_core = n_core;
      for (int c = 0; c < n_core; ++c) {
        const lbk_core_block& b = blocks[c];
        la.core[c] = CoreW{pk[c].g, pk[c].u, pk[c].d, b.gate.col_idx, b.up.col_idx, b.down.col_idx, b.gate.K, b.down.K,
                           b.norm_scale, b.b_gate, b.b_up, b.b_down};
      }
      la.tdepth = tdepth; la.e = e; la.inj_coef = coef;
      // h_out may alias h_in: the kernel reads a token block's h_in rows before any write to them
      return launch_looped(blocks[0].gate.B, la, s) == 0 ? LBK_OK : LBK_ERR_LAUNCH;
    }
    if (launch_core_init(h_in, e, coef, tdepth, L, N, d_model, state, s) != 0) return LBK_ERR_LAUNCH;
    for (int l = 0; l < L; ++l)
      for (int c = 0; c < n_core; ++c) {
        const lbk_core_block& b = blocks[c];
        GUArgs g{};
        g.xf = state; g.N = N; g.d_model = d_model; g.norm_scale = b.norm_scale; g.eps = eps;
        g.pg = pk[c].g; g.cg = b.gate.col_idx; g.Kg = b.gate.K;
        g.pu = pk[c].u; g.cu = b.up.col_idx; g.Ku = b.up.K;
        g.R_ff = b.gate.R; g.h = h; g.bg = b.b_gate; g.bu = b.b_up;
        g.tdepth = tdepth; g.it = l;
        if (launch_gu(b.gate.B, true, g, s) != 0) return LBK_ERR_LAUNCH;
        DNArgs d{};
        d.h = h; d.N = N; d.d_ff = (int64_t)b.gate.R * b.gate.B; d.d_model = d_model;
        d.pd = pk[c].d; d.cd = b.down.col_idx; d.Kd = b.down.K;
        d.R_m = b.down.R; d.C_d = b.gate.R;
        d.state = state; d.out = (l == L - 1 && c == n_core - 1) ? h_out : nullptr; d.bd = b.b_down;
        d.tdepth = tdepth; d.it = l;
        d.inj_e = (c == n_core - 1 && l + 1 < L) ? e : nullptr; d.inj_coef = coef;
        if (launch_dn(b.gate.B, d, s) != 0) return LBK_ERR_LAUNCH;
      }
    return LBK_OK;
  }

  // decode / row-block kernels: RMSNorm of the state into xn, the block's FFN into y, then the
  // elementwise state update (depth mask, next injection, output after the last block)
  uint16_t* xn = reinterpret_cast<uint16_t*>(rest);
  uint16_t* y = reinterpret_cast<uint16_t*>(rest + p.xn);
  if (launch_core_init(h_in, e, coef, tdepth, L, N, d_model, state, s) != 0) return LBK_ERR_LAUNCH;
  for (int l = 0; l < L; ++l)
    for (int c = 0; c < n_core; ++c) {
      const lbk_core_block& b = blocks[c];
      if (launch_rmsnorm_f32(state, N, d_model, b.norm_scale, eps, xn, s) != 0) return LBK_ERR_LAUNCH;
      if (p.path == CORE_DECODE) {
        DecodeArgs a{};
        a.x = xn; a.N = (int)N; a.d_model = d_model;
        a.vg = b.gate.values; a.cg = b.gate.col_idx; a.Kg = b.gate.K;
        a.vu = b.up.values; a.cu = b.up.col_idx; a.Ku = b.up.K;
        a.R_ff = b.gate.R;
        a.vd = b.down.values; a.cd = b.down.col_idx; a.Kd = b.down.K;
        a.R_m = b.down.R;
        a.out = y; a.h = h;
        a.bg = b.b_gate; a.bu = b.b_up; a.bd = b.b_down;
        if (launch_decode(b.gate.B, a, s) != 0) return LBK_ERR_LAUNCH;
      } else if ((st = swiglu_general(xn, N, d_model, &b.gate, &b.up, &b.down, nullptr, y, h, nullptr, nullptr, s,
                                      Biases{b.b_gate, b.b_up, b.b_down}))) {
        return st;
      }
      if (launch_core_update(state, y, tdepth, l, (c == n_core - 1 && l + 1 < L) ? e : nullptr, coef, N, d_model,
                             (l == L - 1 && c == n_core - 1) ? h_out : nullptr, s) != 0)
        return LBK_ERR_LAUNCH;
    }
  return LBK_OK;
}

int lbk_looped_core_bf16(const uint16_t* h_in, const uint16_t* e, const float* log_A, const float* log_dt,
                         int64_t N, int32_t d_model, int32_t n_core, const lbk_core_block* blocks, float eps,
                         int32_t L, const int32_t* depths, int64_t seq_len, uint16_t* h_out, void* workspace,
                         size_t workspace_bytes, void* stream) {
  return looped_core_impl(h_in, e, log_A, log_dt, N, d_model, n_core, blocks, eps, L, depths, seq_len, h_out,
                          workspace, workspace_bytes, S(stream), false);
}

int lbk_looped_core_persistent_bf16(const uint16_t* h_in, const uint16_t* e, const float* log_A,
                                    const float* log_dt, int64_t N, int32_t d_model, int32_t n_core,
                                    const lbk_core_block* blocks, float eps, int32_t L, const int32_t* depths,
                                    int64_t seq_len, uint16_t* h_out, void* workspace, size_t workspace_bytes,
                                    void* stream) {
  return looped_core_impl(h_in, e, log_A, log_dt, N, d_model, n_core, blocks, eps, L, depths, seq_len, h_out,
                          workspace, workspace_bytes, S(stream), true);
}

int lbk_quantize_act_int8(const uint16_t* x, int64_t N, int32_t F, int64_t ldx, int8_t* xq, float* sx,
                          void* stream) {
  if (N < 0 || F <= 0 || ldx < F) return LBK_ERR_ARG;
  if (N == 0) return LBK_OK;
  if (!x || !xq || !sx) return LBK_ERR_NULL;
  if ((F % 8) || (ldx % 8) || !a16(x) || !a8(xq)) return LBK_ERR_ALIGN;
  return launch_quantize_act(x, N, F, ldx, xq, sx, S(stream)) == 0 ? LBK_OK : LBK_ERR_LAUNCH;
}

int lbk_pack_ternary(const int8_t* t, int32_t R, int32_t K, int32_t B, uint32_t* packed, void* stream) {
  if (!tile_ok(B)) return LBK_ERR_TILE;
  if (R < 0 || K < 0) return LBK_ERR_SHAPE;
  if ((int64_t)R * K == 0) return LBK_OK;
  if (!t || !packed) return LBK_ERR_NULL;
  return launch_pack_ternary(t, R, K, B, packed, S(stream)) == 0 ? LBK_OK : LBK_ERR_LAUNCH;
}

int lbk_ternary_quantize_weights_bf16(const uint16_t* values, int32_t R, int32_t K, int32_t B, uint32_t* packed,
                                      float* scales, void* stream) {
  if (!tile_ok(B)) return LBK_ERR_TILE;
  if (R < 0 || K < 0) return LBK_ERR_SHAPE;
  if ((int64_t)R * K == 0) return LBK_OK;
  if (!values || !packed || !scales) return LBK_ERR_NULL;
  return launch_ternary_quantize_weights(values, R, K, B, packed, scales, S(stream)) == 0 ? LBK_OK
                                                                                           : LBK_ERR_LAUNCH;
}

int lbk_ternary_matmul(const int8_t* xq, const float* sx, int64_t N, int32_t in_features,
                       const lbk_bell_ternary* w, uint16_t* y, int32_t* partials, void* stream) {
  int st = check_tern(w);
  if (st) return st;
  if (N < 0) return LBK_ERR_ARG;
  if (in_features <= 0 || in_features % w->B) return LBK_ERR_SHAPE;
  if (N == 0) return LBK_OK;
  if (!xq || !sx || !y) return LBK_ERR_NULL;
  if (!a16(xq) || !a8(y)) return LBK_ERR_ALIGN;
  TernaryLaunch a{};
  a.xq = xq; a.sx = sx; a.N = N; a.C = in_features / w->B;
  a.p0 = w->packed; a.s0 = w->scales; a.c0 = w->col_idx; a.K0 = w->K;
  a.R = w->R; a.y = y; a.partials = partials;
  return launch_ternary(w->B, 0, a, S(stream)) == 0 ? LBK_OK : LBK_ERR_LAUNCH;
}

size_t lbk_ternary_swiglu_workspace_bytes(int64_t N, int32_t d_model, const lbk_bell_ternary* gate,
                                          const lbk_bell_ternary* up, const lbk_bell_ternary* down) {
  if (!gate || !up || !down || N <= 0) return 0;
  if (check_tern(gate) || check_tern(up) || check_tern(down)) return 0;
  int64_t d_ff = 0;
  if (check_ffn(gate, up, down, d_model, &d_ff)) return 0;
  if (tern_split(N, d_model, gate, up, down)) return tern_split_layout(N, gate, up, down).total;
  return align256((size_t)N * d_ff * 2) + align256((size_t)N * d_ff) + align256((size_t)N * 4);
}

int lbk_swiglu_fwd_ternary(const int8_t* xq, const float* sx, int64_t N, int32_t d_model,
                           const lbk_bell_ternary* gate, const lbk_bell_ternary* up, const lbk_bell_ternary* down,
                           const uint16_t* x_resid, uint16_t* out, uint16_t* h_out, int8_t* hq_out,
                           float* sh_out, void* workspace, size_t workspace_bytes, void* stream) {
  return lbk_swiglu_fwd_ternary_acc(xq, sx, N, d_model, gate, up, down, x_resid, out, h_out, hq_out, sh_out, nullptr,
                                    workspace, workspace_bytes, stream);
}

// prepared weights of the B = 64 two-kernel path: gate | up | down regions of tprep_bytes each
static size_t tern_prepared_bytes(const lbk_bell_ternary* gate, const lbk_bell_ternary* up,
                                  const lbk_bell_ternary* down) {
  const TernSplitLayout L = tern_split_layout(1, gate, up, down);
  return L.pg + L.pu + L.pd;
}

// The ternary forward behind lbk_swiglu_fwd_ternary_acc and lbk_swiglu_fwd_ternary_prepared:
// `prepared` (may be null) holds the weights of lbk_ternary_prepare, otherwise the two-kernel
// path prepares them into the workspace.
static int tern_fwd_impl(const int8_t* xq, const float* sx, int64_t N, int32_t d_model, const lbk_bell_ternary* gate,
                         const lbk_bell_ternary* up, const lbk_bell_ternary* down, const char* prepared,
                         size_t prepared_bytes, const uint16_t* x_resid, uint16_t* out, uint16_t* h_out,
                         int8_t* hq_out, float* sh_out, const lbk_ternary_acc* acc, void* workspace,
                         size_t workspace_bytes, hipStream_t s) {
  int st;
  if ((st = check_tern(gate)) || (st = check_tern(up)) || (st = check_tern(down))) return st;
  int64_t d_ff = 0;
  if ((st = check_ffn(gate, up, down, d_model, &d_ff))) return st;
  if (N < 0) return LBK_ERR_ARG;
  if (N == 0) return LBK_OK;
  if (!xq || !sx || !out) return LBK_ERR_NULL;
  if (!a16(xq) || !a16(out)) return LBK_ERR_ALIGN;
  // the down kernels read the residual with vector loads
  if (x_resid && !a16(x_resid)) return LBK_ERR_ALIGN;
  lbk_ternary_acc ax{};
  if (acc) {
    ax = *acc;
    // gate and up accumulators (and pre-activations) come as pairs
    if (!ax.acc_gate != !ax.acc_up || !ax.gate_pre != !ax.up_pre) return LBK_ERR_NULL;
    for (const void* p : {(const void*)ax.acc_gate, (const void*)ax.acc_up, (const void*)ax.acc_down,
                          (const void*)ax.gate_pre, (const void*)ax.up_pre})
      if (p && !a16(p)) return LBK_ERR_ALIGN;
  }
  char* ws = static_cast<char*>(workspace);

  if (tern_split(N, d_model, gate, up, down)) {
    const TernSplitLayout L = tern_split_layout(N, gate, up, down);
    // [prepared gate | up | down (unless given)] [per-slice maxima of h] [h]
    const size_t pbytes = L.pg + L.pu + L.pd;
    if (prepared) {
      if (prepared_bytes < pbytes) return LBK_ERR_WORKSPACE;
      if (!a16(prepared)) return LBK_ERR_ALIGN;
    }
    const size_t own = prepared ? 0 : pbytes;
    if (!ws || workspace_bytes < L.total - pbytes + own) return LBK_ERR_WORKSPACE;
    if (!a16(ws)) return LBK_ERR_ALIGN;
    char* pb = prepared ? const_cast<char*>(prepared) : ws;
    uint16_t* h = h_out ? h_out : reinterpret_cast<uint16_t*>(ws + own + L.hmax);
    if (!a16(h) || (hq_out && !a16(hq_out))) return LBK_ERR_ALIGN;
    const int C_in = d_model / gate->B;
    TGUArgs g{};
    TDNArgs d{};
    const TPrepWeight pw[3] = {{gate->packed, gate->scales, gate->col_idx, gate->R, gate->K, C_in},
                               {up->packed, up->scales, up->col_idx, up->R, up->K, C_in},
                               {down->packed, down->scales, down->col_idx, down->R, down->K, gate->R}};
    void* const po[3] = {pb, pb + L.pg, pb + L.pg + L.pu};
    const tu32x4* ptw[3];
    const int32_t* pm[3];
    const float* pr[3];
    if (launch_tprep(pw, po, ptw, pm, pr, s, prepared == nullptr) != 0) return LBK_ERR_LAUNCH;
    g.twg = ptw[0]; g.mg = pm[0]; g.rmg = pr[0];
    g.twu = ptw[1]; g.mu = pm[1]; g.rmu = pr[1];
    d.twd = ptw[2]; d.md = pm[2]; d.rmd = pr[2];
    float* hmax = reinterpret_cast<float*>(ws + own);
    g.xq = xq; g.sx = sx; g.N = N; g.d_model = d_model;
    g.cg = gate->col_idx; g.cu = up->col_idx; g.K = gate->K;
    g.R_ff = gate->R; g.H = tgu_slices(N, gate->R); g.h = h; g.hmax = hmax;
    g.acc_g = ax.acc_gate; g.acc_u = ax.acc_up; g.g_pre = ax.gate_pre; g.u_pre = ax.up_pre;
    if (launch_tgu(g, s) != 0) return LBK_ERR_LAUNCH;
    d.h = h; d.hmax = hmax; d.H = g.H; d.N = N; d.d_ff = (int)d_ff; d.d_model = d_model;
    d.cd = down->col_idx; d.Kd = down->K; d.R_m = down->R; d.C_d = gate->R;
    d.resid = x_resid; d.out = out; d.hq_out = hq_out; d.sh_out = sh_out; d.acc_d = ax.acc_down;
    if (launch_tdn(d, s) != 0) return LBK_ERR_LAUNCH;
    return LBK_OK;
  }

  const size_t hb = align256((size_t)N * d_ff * 2), qb = align256((size_t)N * d_ff);
  const bool need_ws = !h_out || !hq_out || !sh_out;
  if (need_ws) {
    if (!ws || workspace_bytes < lbk_ternary_swiglu_workspace_bytes(N, d_model, gate, up, down))
      return LBK_ERR_WORKSPACE;
    if (!a16(ws)) return LBK_ERR_ALIGN;
  }
  uint16_t* h = h_out ? h_out : reinterpret_cast<uint16_t*>(ws);
  int8_t* hq = hq_out ? hq_out : reinterpret_cast<int8_t*>(ws + hb);
  float* sh = sh_out ? sh_out : reinterpret_cast<float*>(ws + hb + qb);
  if (!a16(h) || !a16(hq)) return LBK_ERR_ALIGN;
  TernaryLaunch a{};
  a.xq = xq; a.sx = sx; a.N = N; a.C = d_model / gate->B;
  a.p0 = gate->packed; a.s0 = gate->scales; a.c0 = gate->col_idx; a.K0 = gate->K;
  a.p1 = up->packed; a.s1 = up->scales; a.c1 = up->col_idx; a.K1 = up->K;
  a.R = gate->R; a.y = h;
  a.acc0 = ax.acc_gate; a.acc1 = ax.acc_up; a.pre0 = ax.gate_pre; a.pre1 = ax.up_pre;
  if (launch_ternary(gate->B, 1, a, s) != 0) return LBK_ERR_LAUNCH;
  if (launch_quantize_act(h, N, (int)d_ff, d_ff, hq, sh, s) != 0) return LBK_ERR_LAUNCH;
  TernaryLaunch d{};
  d.xq = hq; d.sx = sh; d.N = N; d.C = gate->R;
  d.p0 = down->packed; d.s0 = down->scales; d.c0 = down->col_idx; d.K0 = down->K;
  d.R = down->R; d.resid = x_resid; d.y = out; d.acc0 = ax.acc_down;
  if (launch_ternary(gate->B, 0, d, s) != 0) return LBK_ERR_LAUNCH;
  return LBK_OK;
}

int lbk_swiglu_fwd_ternary_acc(const int8_t* xq, const float* sx, int64_t N, int32_t d_model,
                               const lbk_bell_ternary* gate, const lbk_bell_ternary* up,
                               const lbk_bell_ternary* down, const uint16_t* x_resid, uint16_t* out,
                               uint16_t* h_out, int8_t* hq_out, float* sh_out, const lbk_ternary_acc* acc,
                               void* workspace, size_t workspace_bytes, void* stream) {
  return tern_fwd_impl(xq, sx, N, d_model, gate, up, down, nullptr, 0, x_resid, out, h_out, hq_out, sh_out, acc,
                       workspace, workspace_bytes, S(stream));
}

size_t lbk_ternary_prepared_bytes(int32_t d_model, const lbk_bell_ternary* gate, const lbk_bell_ternary* up,
                                  const lbk_bell_ternary* down) {
  if (!gate || !up || !down) return 0;
  if (check_tern(gate) || check_tern(up) || check_tern(down)) return 0;
  int64_t d_ff = 0;
  if (check_ffn(gate, up, down, d_model, &d_ff)) return 0;
  return tern_split(1, d_model, gate, up, down) ? tern_prepared_bytes(gate, up, down) : 0;
}

int lbk_ternary_prepare(int32_t d_model, const lbk_bell_ternary* gate, const lbk_bell_ternary* up,
                        const lbk_bell_ternary* down, void* prepared, size_t prepared_bytes, void* stream) {
  int st;
  if ((st = check_tern(gate)) || (st = check_tern(up)) || (st = check_tern(down))) return st;
  int64_t d_ff = 0;
  if ((st = check_ffn(gate, up, down, d_model, &d_ff))) return st;
  if (!tern_split(1, d_model, gate, up, down)) return LBK_OK;        // no prepared form for this geometry
  const TernSplitLayout L = tern_split_layout(1, gate, up, down);
  if (!prepared || prepared_bytes < L.pg + L.pu + L.pd) return LBK_ERR_WORKSPACE;
  if (!a16(prepared)) return LBK_ERR_ALIGN;
  char* pb = static_cast<char*>(prepared);
  const int C_in = d_model / gate->B;
  const TPrepWeight pw[3] = {{gate->packed, gate->scales, gate->col_idx, gate->R, gate->K, C_in},
                             {up->packed, up->scales, up->col_idx, up->R, up->K, C_in},
                             {down->packed, down->scales, down->col_idx, down->R, down->K, gate->R}};
  void* const po[3] = {pb, pb + L.pg, pb + L.pg + L.pu};
  const tu32x4* ptw[3];
  const int32_t* pm[3];
  const float* pr[3];
  return launch_tprep(pw, po, ptw, pm, pr, S(stream)) == 0 ? LBK_OK : LBK_ERR_LAUNCH;
}

size_t lbk_ternary_prepared_workspace_bytes(int64_t N, int32_t d_model, const lbk_bell_ternary* gate,
                                            const lbk_bell_ternary* up, const lbk_bell_ternary* down) {
  const size_t all = lbk_ternary_swiglu_workspace_bytes(N, d_model, gate, up, down);
  if (all == 0 || !tern_split(N, d_model, gate, up, down)) return all;
  return all - tern_prepared_bytes(gate, up, down);
}

int lbk_swiglu_fwd_ternary_prepared(const int8_t* xq, const float* sx, int64_t N, int32_t d_model,
                                    const lbk_bell_ternary* gate, const lbk_bell_ternary* up,
                                    const lbk_bell_ternary* down, const void* prepared, size_t prepared_bytes,
                                    const uint16_t* x_resid, uint16_t* out, uint16_t* h_out, int8_t* hq_out,
                                    float* sh_out, const lbk_ternary_acc* acc, void* workspace,
                                    size_t workspace_bytes, void* stream) {
  if (!gate || !up || !down) return LBK_ERR_NULL;
  if (N > 0 && !prepared && tern_split(N, d_model, gate, up, down)) return LBK_ERR_NULL;
  return tern_fwd_impl(xq, sx, N, d_model, gate, up, down, static_cast<const char*>(prepared), prepared_bytes,
                       x_resid, out, h_out, hq_out, sh_out, acc, workspace, workspace_bytes, S(stream));
}

// ---- backward of the SwiGLU FFN
// workspace: [transposed lists of down, gate, up] [dg] [du] [fp32 partial tiles]
static size_t tlist_bytes(const lbk_bell* w, int C) {
  return align256((size_t)C * 4) + align256((size_t)C * w->R * w->K * 4);
}
// floats of the column sums that dh's kernel forms per token block (blocks of 32 tokens at most 2 N / 64 + 1)
static size_t dh_sum_floats(int64_t N, int64_t d_ff) { return (size_t)((N + 31) / 32) * (size_t)d_ff; }
// fp32 partial tiles of one weight's tile gradients (the token chunking of launch_dw)
static size_t dw_part_floats(int64_t N, const lbk_bell* w, int C, int64_t ldg) {
  const int64_t ch = dw_job_chunk(w->B, w->R, w->K, C, ldg, N);
  return (size_t)((N + ch - 1) / ch) * w->R * w->K * w->B * w->B;
}

size_t lbk_swiglu_bwd_workspace_bytes(int64_t N, int32_t d_model, const lbk_bell* gate, const lbk_bell* up,
                                      const lbk_bell* down) {
  if (!gate || !up || !down || N < 0 || d_model <= 0 || !tile_ok(gate->B)) return 0;
  const int B = gate->B;
  const int C_in = d_model / B, C_d = gate->R;
  const size_t d_ff = (size_t)gate->R * B;
  const size_t parts = dw_part_floats(N, gate, C_in, (int64_t)d_ff) + dw_part_floats(N, up, C_in, (int64_t)d_ff) +
                       dw_part_floats(N, down, C_d, d_model);
  return tlist_bytes(down, C_d) + tlist_bytes(gate, C_in) + tlist_bytes(up, C_in) +
         2 * align256((size_t)N * d_ff * 2) + align256(parts * 4);
}

size_t lbk_swiglu_bwd_bias_workspace_bytes(int64_t N, int32_t d_model, const lbk_bell* gate, const lbk_bell* up,
                                           const lbk_bell* down) {
  const size_t base = lbk_swiglu_bwd_workspace_bytes(N, d_model, gate, up, down);
  if (!base) return 0;
  const int64_t d_ff = (int64_t)gate->R * gate->B;
  return base + align256(colsum_bytes(N, 2 * d_ff + d_model)) + 2 * align256(dh_sum_floats(N, d_ff) * 4);
}

int lbk_swiglu_bwd_bf16(const uint16_t* grad_out, const uint16_t* x, const uint16_t* gate_pre_act,
                        const uint16_t* up_output, const uint16_t* h, int64_t N, int32_t d_model,
                        const lbk_bell* gate, const lbk_bell* up, const lbk_bell* down, int add_residual,
                        uint16_t* dx, uint16_t* d_gate_values, uint16_t* d_up_values, uint16_t* d_down_values,
                        void* workspace, size_t workspace_bytes, void* stream) {
  return lbk_swiglu_bwd_bias_bf16(grad_out, x, gate_pre_act, up_output, h, N, d_model, gate, up, down, add_residual,
                                  dx, d_gate_values, d_up_values, d_down_values, nullptr, nullptr, nullptr,
                                  workspace, workspace_bytes, stream);
}

// outputs of the backward: tile gradients in bf16 (dv) or fp32 (dv32), for gate, up and down
struct BwdGrads {
  uint16_t* dv[3];
  float* dv32[3];
  const void* any(int t) const { return dv32[t] ? static_cast<const void*>(dv32[t]) : dv[t]; }
};

static int swiglu_bwd_impl(const uint16_t* grad_out, const uint16_t* x, const uint16_t* gate_pre_act,
                           const uint16_t* up_output, const uint16_t* h, int64_t N, int32_t d_model,
                           const lbk_bell* gate, const lbk_bell* up, const lbk_bell* down, int add_residual,
                           uint16_t* dx, const BwdGrads& dw, float* d_b_gate, float* d_b_up, float* d_b_down,
                           void* workspace, size_t workspace_bytes, void* stream) {
  const bool want_db = d_b_gate || d_b_up || d_b_down;
  int st;
  if ((st = check_bell(gate)) || (st = check_bell(up)) || (st = check_bell(down))) return st;
  int64_t d_ff = 0;
  if ((st = check_ffn(gate, up, down, d_model, &d_ff))) return st;
  if (N < 0) return LBK_ERR_ARG;
  const int B = gate->B;
  const int64_t tg = (int64_t)gate->R * gate->K, tu = (int64_t)up->R * up->K, td = (int64_t)down->R * down->K;
  if ((tg && !dw.any(0)) || (tu && !dw.any(1)) || (td && !dw.any(2))) return LBK_ERR_NULL;
  for (int t = 0; t < 3; ++t)
    if (dw.any(t) && !a16(dw.any(t))) return LBK_ERR_ALIGN;
  if (N > 0) {
    if (!grad_out || !x || !gate_pre_act || !up_output || !h || !dx) return LBK_ERR_NULL;
    for (const void* p : {(const void*)grad_out, (const void*)x, (const void*)gate_pre_act, (const void*)up_output,
                          (const void*)h, (const void*)dx})
      if (!a16(p)) return LBK_ERR_ALIGN;
    if (d_model % 8) return LBK_ERR_ALIGN;
  }
  for (const lbk_bell* w : {gate, up, down})
    if ((int64_t)w->R * w->K > 0 && !a16(w->values)) return LBK_ERR_ALIGN;
  const size_t need = want_db ? lbk_swiglu_bwd_bias_workspace_bytes(N, d_model, gate, up, down)
                              : lbk_swiglu_bwd_workspace_bytes(N, d_model, gate, up, down);
  if (!workspace || workspace_bytes < need) return LBK_ERR_WORKSPACE;
  if (!a16(workspace)) return LBK_ERR_ALIGN;
  hipStream_t s = S(stream);
  const int C_in = d_model / B, C_d = gate->R;
  char* p = static_cast<char*>(workspace);
  auto take = [&](size_t bytes) {
    char* q = p;
    p += align256(bytes);
    return q;
  };
  const lbk_bell* w3[3] = {down, gate, up};
  const int c3[3] = {C_d, C_in, C_in};
  TListJob lj[3];
  for (int t = 0; t < 3; ++t) {
    lj[t].col = w3[t]->col_idx; lj[t].R = w3[t]->R; lj[t].K = w3[t]->K; lj[t].C = c3[t];
    lj[t].cnt = reinterpret_cast<int32_t*>(take((size_t)c3[t] * 4));
    lj[t].list = reinterpret_cast<int32_t*>(take((size_t)c3[t] * w3[t]->R * w3[t]->K * 4));
  }
  uint16_t* dg = reinterpret_cast<uint16_t*>(take((size_t)N * d_ff * 2));
  uint16_t* du = reinterpret_cast<uint16_t*>(take((size_t)N * d_ff * 2));
  float* part = reinterpret_cast<float*>(p);
  // after the tile partials: the column sums of dg and du that dh's kernel forms, and the partials of
  // those (and of grad_out) read as matrices
  const size_t parts = dw_part_floats(N, gate, C_in, d_ff) + dw_part_floats(N, up, C_in, d_ff) +
                       dw_part_floats(N, down, C_d, d_model);
  char* tail = reinterpret_cast<char*>(part) + align256(parts * 4);
  float* gsum = reinterpret_cast<float*>(tail);
  float* usum = reinterpret_cast<float*>(tail + align256(dh_sum_floats(N, d_ff) * 4));
  float* cpart = reinterpret_cast<float*>(tail + 2 * align256(dh_sum_floats(N, d_ff) * 4));
  int64_t sum_rows = 0;
  // slots of a weight with no tiles (R * K == 0) take no part in the lists
  int nl = 0;
  TListJob ljn[3];
  for (int t = 0; t < 3; ++t)
    if ((int64_t)lj[t].R * lj[t].K > 0) ljn[nl++] = lj[t];
  if (N > 0) {
    if (nl && launch_tlist(ljn, nl, s)) return LBK_ERR_LAUNCH;
    // dh = dy W_down -> dg, du
    TProdArgs a{};
    a.nsrc = 0;
    if (td > 0) a.src[a.nsrc++] = TProdSrc{grad_out, d_model, down->values, down->K, lj[0].cnt, lj[0].list, td};
    a.N = N; a.C = C_d; a.ldo = d_ff;
    a.g = gate_pre_act; a.u = up_output; a.dg = dg; a.du = du;
    if (d_b_gate || d_b_up) sum_rows = dh_sum_blocks(B, a);
    if (sum_rows) { a.dgsum = gsum; a.dusum = usum; }
    if (launch_tprod(B, 0, a, s)) return LBK_ERR_LAUNCH;
    // dx = dg W_gate + du W_up (+ dy)
    TProdArgs b{};
    b.nsrc = 0;
    if (tg > 0) b.src[b.nsrc++] = TProdSrc{dg, d_ff, gate->values, gate->K, lj[1].cnt, lj[1].list, tg};
    if (tu > 0) b.src[b.nsrc++] = TProdSrc{du, d_ff, up->values, up->K, lj[2].cnt, lj[2].list, tu};
    b.N = N; b.C = C_in; b.ldo = d_model;
    b.resid = add_residual ? grad_out : nullptr; b.out = dx;
    if (launch_tprod(B, 1, b, s)) return LBK_ERR_LAUNCH;
  }
  // tile gradients: gate (x, dg), up (x, du), down (h, dy)
  DWJob dj[3];
  int nj = 0;
  size_t poff = 0;
  auto add = [&](const uint16_t* xx, int64_t ldx, const uint16_t* gy, int64_t ldg, const lbk_bell* w, int C,
                 int t, const TListJob* tl) {
    const int64_t nt = (int64_t)w->R * w->K;
    if (nt == 0) return;
    dj[nj++] = DWJob{xx, ldx, gy, ldg, w->col_idx, w->R, w->K, C, part + poff, dw.dv[t], dw.dv32[t], 0,
                     tl ? tl->cnt : nullptr, tl ? tl->list : nullptr, 0, 0};
    poff += dw_part_floats(N, w, C, ldg);
  };
  add(x, d_model, dg, d_ff, gate, C_in, 0, nullptr);
  add(x, d_model, du, d_ff, up, C_in, 1, nullptr);
  // the down weight's transposed lists (built above when N > 0) serve its tile gradients too
  add(h, d_ff, grad_out, d_model, down, C_d, 2, N > 0 ? &lj[0] : nullptr);
  if (nj && launch_dw(B, dj, nj, N, s)) return LBK_ERR_LAUNCH;
  // bias gradients: column sums of dg, du and grad_out (the partials after the tile partials)
  if (want_db) {
    ColsumJob cj[3];
    int nc = 0;
    const bool have = sum_rows > 0;
    if (d_b_gate) cj[nc++] = ColsumJob{have ? nullptr : dg, d_ff, (int)d_ff, d_b_gate, gsum, (int)sum_rows, 0};
    if (d_b_up) cj[nc++] = ColsumJob{have ? nullptr : du, d_ff, (int)d_ff, d_b_up, usum, (int)sum_rows, 0};
    if (d_b_down) cj[nc++] = ColsumJob{grad_out, d_model, d_model, d_b_down, nullptr, 0, 0};
    if (launch_colsum(cj, nc, N, cpart, s)) return LBK_ERR_LAUNCH;
  }
  return LBK_OK;
}

int lbk_swiglu_bwd_bias_bf16(const uint16_t* grad_out, const uint16_t* x, const uint16_t* gate_pre_act,
                             const uint16_t* up_output, const uint16_t* h, int64_t N, int32_t d_model,
                             const lbk_bell* gate, const lbk_bell* up, const lbk_bell* down, int add_residual,
                             uint16_t* dx, uint16_t* d_gate_values, uint16_t* d_up_values,
                             uint16_t* d_down_values, float* d_b_gate, float* d_b_up, float* d_b_down,
                             void* workspace, size_t workspace_bytes, void* stream) {
  return swiglu_bwd_impl(grad_out, x, gate_pre_act, up_output, h, N, d_model, gate, up, down, add_residual, dx,
                         BwdGrads{{d_gate_values, d_up_values, d_down_values}, {}}, d_b_gate, d_b_up, d_b_down,
                         workspace, workspace_bytes, stream);
}

int lbk_swiglu_bwd_train(const uint16_t* grad_out, const uint16_t* x, const uint16_t* gate_pre_act,
                         const uint16_t* up_output, const uint16_t* h, int64_t N, int32_t d_model,
                         const lbk_bell* gate, const lbk_bell* up, const lbk_bell* down, int add_residual,
                         uint16_t* dx, float* d_gate_values, float* d_up_values, float* d_down_values,
                         float* d_b_gate, float* d_b_up, float* d_b_down, void* workspace, size_t workspace_bytes,
                         void* stream) {
  return swiglu_bwd_impl(grad_out, x, gate_pre_act, up_output, h, N, d_model, gate, up, down, add_residual, dx,
                         BwdGrads{{}, {d_gate_values, d_up_values, d_down_values}}, d_b_gate, d_b_up, d_b_down,
                         workspace, workspace_bytes, stream);
}

// ---- training of the looped block h <- h + SwiGLU(RMSNorm(h)), L times with shared weights
size_t lbk_looped_fwd_train_workspace_bytes(int64_t N, int32_t d_model, const lbk_bell* gate, const lbk_bell* up,
                                            const lbk_bell* down) {
  if (!gate || !up || !down || N <= 0 || d_model <= 0) return 0;
  // [fp32 state] [y, the products' result where the down kernel does not add to the state] [packed tiles]
  return align256((size_t)N * d_model * 4) + align256((size_t)N * d_model * 2) +
         (use_split(gate, up, down, d_model) ? packed_ffn_bytes(gate, up, down) : 0);
}

int lbk_looped_fwd_train(const uint16_t* h_in, int64_t N, int32_t d_model, const float* norm_scale, float eps,
                         int32_t L, const lbk_bell* gate, const lbk_bell* up, const lbk_bell* down,
                         const float* v_gate, const float* v_up, const float* v_down, uint16_t* vb_gate,
                         uint16_t* vb_up, uint16_t* vb_down, const float* b_gate, const float* b_up,
                         const float* b_down, uint16_t* out, uint16_t* states, uint16_t* normed, uint16_t* h,
                         uint16_t* gate_pre, uint16_t* up_out, void* workspace, size_t workspace_bytes,
                         void* stream) {
  if (!gate || !up || !down) return LBK_ERR_NULL;
  const MasterFFN m{{v_gate, v_up, v_down}, {vb_gate, vb_up, vb_down}};
  lbk_bell w3[3] = {*gate, *up, *down};
  int st;
  for (int t = 0; t < 3; ++t) {
    w3[t].values = m.raw[t];
    if ((st = check_bell(&w3[t]))) return st;
    if ((int64_t)w3[t].R * w3[t].K > 0) {
      if (!m.v[t]) return LBK_ERR_NULL;
      if (!a16(m.v[t]) || !a16(m.raw[t])) return LBK_ERR_ALIGN;
    }
  }
  int64_t d_ff = 0;
  if ((st = check_ffn(&w3[0], &w3[1], &w3[2], d_model, &d_ff))) return st;
  if (N <= 0 || L < 1 || !(eps >= 0.f)) return LBK_ERR_ARG;
  for (const void* q : {(const void*)h_in, (const void*)out, (const void*)states, (const void*)normed, (const void*)h,
                        (const void*)gate_pre, (const void*)up_out}) {
    if (!q) return LBK_ERR_NULL;
    if (!a16(q)) return LBK_ERR_ALIGN;
  }
  if (!norm_scale) return LBK_ERR_NULL;
  if (d_model % 8) return LBK_ERR_ALIGN;
  if (!workspace || workspace_bytes < lbk_looped_fwd_train_workspace_bytes(N, d_model, gate, up, down))
    return LBK_ERR_WORKSPACE;
  if (!a16(workspace)) return LBK_ERR_ALIGN;
  hipStream_t s = S(stream);
  char* p = static_cast<char*>(workspace);
  float* state = reinterpret_cast<float*>(p);
  p += align256((size_t)N * d_model * 4);
  uint16_t* y = reinterpret_cast<uint16_t*>(p);
  p += align256((size_t)N * d_model * 2);
  const bool split = use_split(&w3[0], &w3[1], &w3[2], d_model);
  PackedFFN pk{};
  if ((st = split ? pack_ffn(&w3[0], &w3[1], &w3[2], p, &pk, s, &m) : cast_ffn(&w3[0], &w3[1], &w3[2], m, s)))
    return st;
  const Biases bs{b_gate, b_up, b_down};
  const int64_t nd = N * d_model, nf = N * d_ff;
  if (launch_state_init(h_in, nd, state, states, s)) return LBK_ERR_LAUNCH;
  for (int l = 0; l < L; ++l) {
    const uint16_t* xn = normed + l * nd;
    uint16_t* next = l + 1 < L ? states + (l + 1) * nd : out;     // bf16 of the state after this application
    if (launch_rmsnorm(states + l * nd, N, d_model, norm_scale, eps, normed + l * nd, s)) return LBK_ERR_LAUNCH;
    if (split) {
      if ((st = swiglu_split(xn, nullptr, nullptr, 0.f, N, d_model, &w3[0], &w3[1], &w3[2], pk, nullptr, state, next,
                             h + l * nf, gate_pre + l * nf, up_out + l * nf, s, bs)))
        return st;
    } else {
      if ((st = swiglu_general(xn, N, d_model, &w3[0], &w3[1], &w3[2], nullptr, y, h + l * nf, gate_pre + l * nf,
                               up_out + l * nf, s, bs)))
        return st;
      if (launch_core_update(state, y, nullptr, 0, nullptr, nullptr, N, d_model, next, s)) return LBK_ERR_LAUNCH;
    }
  }
  return LBK_OK;
}

// Applications whose dg, du and dy the backward keeps before one pass over all of their tokens sums
// the weight gradients: as many as fit 2 GiB of dg and du
static int64_t loop_group(int64_t N, int64_t d_ff, int32_t L) {
  const int64_t g = ((int64_t)1 << 31) / (N * d_ff * 4 > 0 ? N * d_ff * 4 : 1);
  return g < 1 ? 1 : g < L ? g : L;
}

struct LoopBwdLayout {
  size_t lists, dg, dy, dy_next, dxn, tmp, g, dw, cs, sums, rms, total;
};
static LoopBwdLayout loop_bwd_layout(int64_t N, int32_t d_model, int32_t L, const lbk_bell* gate, const lbk_bell* up,
                                     const lbk_bell* down) {
  const int C_in = d_model / gate->B, C_d = gate->R;
  const int64_t d_ff = (int64_t)gate->R * gate->B, G = loop_group(N, d_ff, L);
  LoopBwdLayout l{};
  l.lists = tlist_bytes(down, C_d) + tlist_bytes(gate, C_in) + tlist_bytes(up, C_in);
  l.dg = align256((size_t)G * N * d_ff * 2);
  l.dy = align256((size_t)G * N * d_model * 2);
  l.dy_next = l.dxn = l.tmp = align256((size_t)N * d_model * 2);
  l.g = align256((size_t)N * d_model * 4);
  // token counts of the passes: whole groups, and the last one
  for (const int64_t n : {G * N, (L % G) * N}) {
    if (n == 0) continue;
    const size_t dw = align256((dw_part_floats(n, gate, C_in, d_ff) + dw_part_floats(n, up, C_in, d_ff) +
                                dw_part_floats(n, down, C_d, d_model)) * 4);
    const size_t cs = align256(colsum_bytes(n, 2 * d_ff + d_model));
    l.dw = dw > l.dw ? dw : l.dw;
    l.cs = cs > l.cs ? cs : l.cs;
  }
  l.rms = align256((size_t)G * rmsnorm_bwd_bytes(N, d_model));
  l.sums = align256((size_t)G * dh_sum_floats(N, d_ff) * 4);
  l.total = l.lists + 2 * l.dg + l.dy + l.dy_next + l.dxn + l.tmp + l.g + l.dw + l.cs + 2 * l.sums + l.rms;
  return l;
}

size_t lbk_looped_bwd_train_workspace_bytes(int64_t N, int32_t d_model, int32_t L, const lbk_bell* gate,
                                            const lbk_bell* up, const lbk_bell* down) {
  int64_t d_ff = 0;
  if (check_bell(gate) || check_bell(up) || check_bell(down) || check_ffn(gate, up, down, d_model, &d_ff)) return 0;
  if (N <= 0 || L < 1) return 0;
  return loop_bwd_layout(N, d_model, L, gate, up, down).total;
}

int lbk_looped_bwd_train(const uint16_t* grad_out, const uint16_t* states, const uint16_t* normed, const uint16_t* h,
                         const uint16_t* gate_pre, const uint16_t* up_out, int64_t N, int32_t d_model,
                         const float* norm_scale, float eps, int32_t L, const lbk_bell* gate, const lbk_bell* up,
                         const lbk_bell* down, uint16_t* dh, float* d_scale, float* d_gate_values, float* d_up_values,
                         float* d_down_values, float* d_b_gate, float* d_b_up, float* d_b_down, void* workspace,
                         size_t workspace_bytes, void* stream) {
  int st;
  if ((st = check_bell(gate)) || (st = check_bell(up)) || (st = check_bell(down))) return st;
  int64_t d_ff = 0;
  if ((st = check_ffn(gate, up, down, d_model, &d_ff))) return st;
  if (N <= 0 || L < 1 || !(eps >= 0.f)) return LBK_ERR_ARG;
  const int B = gate->B;
  const int64_t tg = (int64_t)gate->R * gate->K, tu = (int64_t)up->R * up->K, td = (int64_t)down->R * down->K;
  if (!norm_scale || !d_scale || (tg && !d_gate_values) || (tu && !d_up_values) || (td && !d_down_values))
    return LBK_ERR_NULL;
  for (const void* q : {(const void*)grad_out, (const void*)states, (const void*)normed, (const void*)h,
                        (const void*)gate_pre, (const void*)up_out, (const void*)dh}) {
    if (!q) return LBK_ERR_NULL;
    if (!a16(q)) return LBK_ERR_ALIGN;
  }
  for (const void* q : {(const void*)d_gate_values, (const void*)d_up_values, (const void*)d_down_values,
                        (const void*)gate->values, (const void*)up->values, (const void*)down->values})
    if (q && !a16(q)) return LBK_ERR_ALIGN;
  if (d_model % 8) return LBK_ERR_ALIGN;
  const LoopBwdLayout lay = loop_bwd_layout(N, d_model, L, gate, up, down);
  if (!workspace || workspace_bytes < lay.total) return LBK_ERR_WORKSPACE;
  if (!a16(workspace)) return LBK_ERR_ALIGN;
  hipStream_t s = S(stream);
  const int C_in = d_model / B, C_d = gate->R;
  char* p = static_cast<char*>(workspace);
  auto take = [&](size_t bytes) {
    char* q = p;
    p += align256(bytes);
    return q;
  };
  const lbk_bell* w3[3] = {down, gate, up};
  const int c3[3] = {C_d, C_in, C_in};
  TListJob lj[3], ljn[3];
  int nl = 0;
  for (int t = 0; t < 3; ++t) {
    lj[t] = TListJob{w3[t]->col_idx, w3[t]->R, w3[t]->K, c3[t], nullptr, nullptr};
    lj[t].cnt = reinterpret_cast<int32_t*>(take((size_t)c3[t] * 4));
    lj[t].list = reinterpret_cast<int32_t*>(take((size_t)c3[t] * w3[t]->R * w3[t]->K * 4));
    if ((int64_t)w3[t]->R * w3[t]->K > 0) ljn[nl++] = lj[t];
  }
  uint16_t* dg = reinterpret_cast<uint16_t*>(take(lay.dg));
  uint16_t* du = reinterpret_cast<uint16_t*>(take(lay.dg));
  uint16_t* dy = reinterpret_cast<uint16_t*>(take(lay.dy));
  uint16_t* dy_next = reinterpret_cast<uint16_t*>(take(lay.dy_next));
  uint16_t* dxn = reinterpret_cast<uint16_t*>(take(lay.dxn));
  uint16_t* tmp = reinterpret_cast<uint16_t*>(take(lay.tmp));
  float* g = reinterpret_cast<float*>(take(lay.g));
  float* part = reinterpret_cast<float*>(take(lay.dw));
  float* cpart = reinterpret_cast<float*>(take(lay.cs));
  float* gsum = reinterpret_cast<float*>(take(lay.sums));
  float* usum = reinterpret_cast<float*>(take(lay.sums));
  float* rpart = reinterpret_cast<float*>(p);
  if (nl && launch_tlist(ljn, nl, s)) return LBK_ERR_LAUNCH;
  const int64_t nd = N * d_model, nf = N * d_ff, G = loop_group(N, d_ff, L);
  for (int64_t hi = L; hi > 0;) {
    const int64_t lo = hi > G ? hi - G : 0, n = hi - lo;
    const int acc = hi < L;
    // the gradient of the state after application hi - 1, into its slot (and, at the end of the
    // block, into the fp32 state gradient)
    if (launch_state_init(acc ? dy_next : grad_out, nd, acc ? nullptr : g, dy + (n - 1) * nd, s)) return LBK_ERR_LAUNCH;
    int64_t nblk = 0, sum_rows = 0;
    for (int64_t t = hi - 1; t >= lo; --t) {
      const int64_t q = t - lo;
      TProdArgs a{};
      if (td > 0) a.src[a.nsrc++] = TProdSrc{dy + q * nd, d_model, down->values, down->K, lj[0].cnt, lj[0].list, td};
      a.N = N; a.C = C_d; a.ldo = d_ff;
      a.g = gate_pre + t * nf; a.u = up_out + t * nf; a.dg = dg + q * nf; a.du = du + q * nf;
      if (d_b_gate || d_b_up) sum_rows = dh_sum_blocks(B, a);
      if (sum_rows) {
        a.dgsum = gsum + q * sum_rows * d_ff;
        a.dusum = usum + q * sum_rows * d_ff;
      }
      if (launch_tprod(B, 0, a, s)) return LBK_ERR_LAUNCH;
      TProdArgs b{};
      if (tg > 0) b.src[b.nsrc++] = TProdSrc{dg + q * nf, d_ff, gate->values, gate->K, lj[1].cnt, lj[1].list, tg};
      if (tu > 0) b.src[b.nsrc++] = TProdSrc{du + q * nf, d_ff, up->values, up->K, lj[2].cnt, lj[2].list, tu};
      b.N = N; b.C = C_in; b.ldo = d_model;
      b.out = dxn;
      if (launch_tprod(B, 1, b, s)) return LBK_ERR_LAUNCH;
      uint16_t* prev = t == 0 ? dh : q > 0 ? dy + (q - 1) * nd : dy_next;
      nblk = rmsnorm_bwd_blocks(states + t * nd, dxn, N, d_model, norm_scale, prev);
      if (launch_rmsnorm_bwd_part(states + t * nd, dxn, N, d_model, norm_scale, eps, g, prev, tmp,
                                  rpart + q * nblk * d_model, s))
        return LBK_ERR_LAUNCH;
    }
    // the group's weight, bias and scale gradients over its n N tokens
    DWJob dj[3];
    int nj = 0;
    size_t poff = 0;
    auto add = [&](const uint16_t* xx, int64_t ldx, const uint16_t* gy, int64_t ldg, const lbk_bell* w, int C,
                   float* dst, const TListJob* tl) {
      if ((int64_t)w->R * w->K == 0) return;
      dj[nj++] = DWJob{xx, ldx, gy, ldg, w->col_idx, w->R, w->K, C, part + poff, nullptr, dst, acc,
                       tl ? tl->cnt : nullptr, tl ? tl->list : nullptr, 0, 0};
      poff += dw_part_floats(n * N, w, C, ldg);
    };
    add(normed + lo * nd, d_model, dg, d_ff, gate, C_in, d_gate_values, nullptr);
    add(normed + lo * nd, d_model, du, d_ff, up, C_in, d_up_values, nullptr);
    add(h + lo * nf, d_ff, dy, d_model, down, C_d, d_down_values, &lj[0]);
    if (nj && launch_dw(B, dj, nj, n * N, s)) return LBK_ERR_LAUNCH;
    ColsumJob cj[3];
    int nc = 0;
    const bool have = sum_rows > 0;
    const int rows = (int)(n * sum_rows);
    if (d_b_gate) cj[nc++] = ColsumJob{have ? nullptr : dg, d_ff, (int)d_ff, d_b_gate, gsum, rows, acc};
    if (d_b_up) cj[nc++] = ColsumJob{have ? nullptr : du, d_ff, (int)d_ff, d_b_up, usum, rows, acc};
    if (d_b_down) cj[nc++] = ColsumJob{dy, d_model, d_model, d_b_down, nullptr, 0, acc};
    if (nc && launch_colsum(cj, nc, n * N, cpart, s)) return LBK_ERR_LAUNCH;
    if (launch_rmsnorm_dscale(rpart, n * nblk, d_model, d_scale, acc, s)) return LBK_ERR_LAUNCH;
    hi = lo;
  }
  return LBK_OK;
}

// ---- the GELU FFN out = W2 gelu(W1 x + b1) + b2
static int check_gelu(int64_t N, int32_t d_model, const lbk_bell* w1, const lbk_bell* w2) {
  int st;
  if ((st = check_bell(w1)) || (st = check_bell(w2))) return st;
  if (w1->B != w2->B) return LBK_ERR_TILE;
  if (N < 0) return LBK_ERR_ARG;
  if (d_model <= 0 || d_model % w1->B || (int64_t)w2->R * w2->B != d_model) return LBK_ERR_SHAPE;
  return LBK_OK;
}

static size_t gelu_packed_bytes(int32_t in_features, const lbk_bell* w) {
  return lbk_block_ell_matmul_workspace_bytes(1, in_features, w);
}

size_t lbk_gelu_workspace_bytes(int64_t N, int32_t d_model, const lbk_bell* w1, const lbk_bell* w2, int prepacked,
                                int want_h) {
  if (!w1 || !w2 || check_gelu(N, d_model, w1, w2)) return 0;
  const size_t h = want_h ? 0 : align256((size_t)N * w1->R * w1->B * 2);
  return h + (prepacked ? 0 : gelu_packed_bytes(d_model, w1) + gelu_packed_bytes(w1->R * w1->B, w2));
}

// h = gelu(x W1 + b1), the pre-activation to `pre` (optional): in the epilogue where the product's
// kernel has one, else a pass over it
static int gelu_product(const uint16_t* x, int64_t N, int32_t d_model, const lbk_bell* w, const void* pk,
                        const float* bias, uint16_t* h, uint16_t* pre, hipStream_t s) {
  const int64_t out_f = (int64_t)w->R * w->B;
  if (matmul_path(d_model, w) == MM_LIN) {
    GUArgs g{};
    g.x = x; g.N = N; g.d_model = d_model;
    g.pg = pk; g.cg = w->col_idx; g.Kg = w->K;
    g.R_ff = w->R; g.h = h; g.gpre = pre; g.bg = bias;
    return launch_lin_gelu(w->B, g, s) == 0 ? LBK_OK : LBK_ERR_LAUNCH;
  }
  if (w->B == 64 && w->R > 0) {
    RowblockLaunch a{};
    a.x = x; a.N = N; a.ldx = d_model; a.C = d_model / w->B; a.R = w->R;
    a.v0 = w->values; a.c0 = w->col_idx; a.K0 = w->K;
    a.bias = bias; a.y = h; a.ldy = out_f;
    a.gelu = 1; a.aux0 = pre; a.ldaux = out_f;
    const int rc = launch_t64(0, a, s);
    if (rc != -2) return rc == 0 ? LBK_OK : LBK_ERR_LAUNCH;
  }
  uint16_t* y = pre ? pre : h;
  const int st = matmul_impl(x, N, d_model, w, pk, pk ? gelu_packed_bytes(d_model, w) : 0, bias, y, nullptr, 0, s);
  if (st) return st;
  return launch_gelu(y, N * out_f, h, s) == 0 ? LBK_OK : LBK_ERR_LAUNCH;
}

static int gelu_fwd_impl(const uint16_t* x, int64_t N, int32_t d_model, const lbk_bell* w1, const lbk_bell* w2,
                         const void* packed1, size_t packed1_bytes, const void* packed2, size_t packed2_bytes,
                         const float* const master[2], uint16_t* const raw[2], const float* b1, const float* b2,
                         uint16_t* out, uint16_t* h_out, uint16_t* pre_out, void* workspace, size_t workspace_bytes,
                         hipStream_t s) {
  int st = check_gelu(N, d_model, w1, w2);
  if (st) return st;
  const int32_t d_ff = w1->R * w1->B;
  const lbk_bell* w[2] = {w1, w2};
  const int32_t in[2] = {d_model, d_ff};
  const size_t pb[2] = {gelu_packed_bytes(d_model, w1), gelu_packed_bytes(d_ff, w2)};
  if (N > 0) {
    if (!x || !out) return LBK_ERR_NULL;
    for (const void* p : {(const void*)x, (const void*)out, (const void*)h_out, (const void*)pre_out})
      if (p && !a16(p)) return LBK_ERR_ALIGN;
    if (d_model % 8) return LBK_ERR_ALIGN;
  }
  const size_t need = lbk_gelu_workspace_bytes(N, d_model, w1, w2, master ? 0 : 1, h_out != nullptr);
  if (need > 0 && (!workspace || workspace_bytes < need)) return LBK_ERR_WORKSPACE;
  if (need > 0 && !a16(workspace)) return LBK_ERR_ALIGN;
  char* p = static_cast<char*>(workspace);
  const void* pk[2] = {packed1, packed2};
  if (master) {
    PackJob jobs[2];
    int nj = 0;
    for (int t = 0; t < 2; ++t) {
      const int64_t nt = (int64_t)w[t]->R * w[t]->K;
      pk[t] = pb[t] ? p : nullptr;
      if (nt > 0 || pb[t])
        jobs[nj++] = PackJob{w[t]->values, w[t]->col_idx, nt, in[t] / w[t]->B, reinterpret_cast<uint32_t*>(pb[t] ? p : nullptr),
                             0, matmul_path(in[t], w[t]) == MM_LIN, master[t], raw[t]};
      p += pb[t];
    }
    if (nj && launch_pack_bf16_multi(jobs, nj, w1->B, s)) return LBK_ERR_LAUNCH;
  } else if (N > 0) {
    const size_t got[2] = {packed1_bytes, packed2_bytes};
    for (int t = 0; t < 2; ++t) {
      if (pb[t] == 0) continue;
      if (!pk[t]) return LBK_ERR_NULL;
      if (got[t] < pb[t]) return LBK_ERR_WORKSPACE;
      if (!a16(pk[t])) return LBK_ERR_ALIGN;
    }
  }
  if (N == 0) return LBK_OK;
  uint16_t* h = h_out ? h_out : reinterpret_cast<uint16_t*>(p);
  if ((st = gelu_product(x, N, d_model, w1, pb[0] ? pk[0] : nullptr, b1, h, pre_out, s))) return st;
  return matmul_impl(h, N, d_ff, w2, pb[1] ? pk[1] : nullptr, pb[1], b2, out, nullptr, 0, s);
}

int lbk_gelu_fwd_prepacked_bf16(const uint16_t* x, int64_t N, int32_t d_model, const lbk_bell* w1,
                                const lbk_bell* w2, const void* packed1, size_t packed1_bytes, const void* packed2,
                                size_t packed2_bytes, const float* b1, const float* b2, uint16_t* out,
                                void* workspace, size_t workspace_bytes, void* stream) {
  return gelu_fwd_impl(x, N, d_model, w1, w2, packed1, packed1_bytes, packed2, packed2_bytes, nullptr, nullptr, b1, b2,
                       out, nullptr, nullptr, workspace, workspace_bytes, S(stream));
}

int lbk_gelu_fwd_train(const uint16_t* x, int64_t N, int32_t d_model, const lbk_bell* w1, const lbk_bell* w2,
                       const float* v1, const float* v2, uint16_t* vb1, uint16_t* vb2, const float* b1,
                       const float* b2, uint16_t* out, uint16_t* h_out, uint16_t* pre_out, void* workspace,
                       size_t workspace_bytes, void* stream) {
  if (!w1 || !w2) return LBK_ERR_NULL;
  lbk_bell w[2] = {*w1, *w2};
  const float* m[2] = {v1, v2};
  uint16_t* raw[2] = {vb1, vb2};
  for (int t = 0; t < 2; ++t) {
    w[t].values = raw[t];
    const int st = check_bell(&w[t]);
    if (st) return st;
    if ((int64_t)w[t].R * w[t].K > 0) {
      if (!m[t]) return LBK_ERR_NULL;
      if (!a16(m[t]) || !a16(raw[t])) return LBK_ERR_ALIGN;
    }
  }
  if (N > 0 && (!h_out || !pre_out)) return LBK_ERR_NULL;
  return gelu_fwd_impl(x, N, d_model, &w[0], &w[1], nullptr, 0, nullptr, 0, m, raw, b1, b2, out, h_out, pre_out,
                       workspace, workspace_bytes, S(stream));
}

size_t lbk_gelu_bwd_workspace_bytes(int64_t N, int32_t d_model, const lbk_bell* w1, const lbk_bell* w2) {
  if (!w1 || !w2 || check_gelu(N, d_model, w1, w2)) return 0;
  const int64_t d_ff = (int64_t)w1->R * w1->B;
  const int C_in = d_model / w1->B, C_d = w1->R;
  return tlist_bytes(w2, C_d) + tlist_bytes(w1, C_in) + align256((size_t)N * d_ff * 2) +
         align256((dw_part_floats(N, w1, C_in, d_ff) + dw_part_floats(N, w2, C_d, d_model)) * 4) +
         align256(dh_sum_floats(N, d_ff) * 4) + align256(colsum_bytes(N, d_ff + d_model));
}

int lbk_gelu_bwd_train(const uint16_t* grad_out, const uint16_t* x, const uint16_t* pre, const uint16_t* h,
                       int64_t N, int32_t d_model, const lbk_bell* w1, const lbk_bell* w2, uint16_t* dx,
                       float* d_v1, float* d_v2, float* d_b1, float* d_b2, void* workspace, size_t workspace_bytes,
                       void* stream) {
  int st = check_gelu(N, d_model, w1, w2);
  if (st) return st;
  const int B = w1->B;
  const int64_t d_ff = (int64_t)w1->R * B, t1 = (int64_t)w1->R * w1->K, t2 = (int64_t)w2->R * w2->K;
  const int C_in = d_model / B, C_d = w1->R;
  if ((t1 && !d_v1) || (t2 && !d_v2)) return LBK_ERR_NULL;
  for (const void* q : {(const void*)d_v1, (const void*)d_v2, (const void*)w1->values, (const void*)w2->values})
    if (q && !a16(q)) return LBK_ERR_ALIGN;
  if (N > 0) {
    if (!grad_out || !x || !pre || !h || !dx) return LBK_ERR_NULL;
    for (const void* q : {(const void*)grad_out, (const void*)x, (const void*)pre, (const void*)h, (const void*)dx})
      if (!a16(q)) return LBK_ERR_ALIGN;
    if (d_model % 8) return LBK_ERR_ALIGN;
  }
  const size_t need = lbk_gelu_bwd_workspace_bytes(N, d_model, w1, w2);
  if (!workspace || workspace_bytes < need) return LBK_ERR_WORKSPACE;
  if (!a16(workspace)) return LBK_ERR_ALIGN;
  hipStream_t s = S(stream);
  char* p = static_cast<char*>(workspace);
  auto take = [&](size_t bytes) {
    char* q = p;
    p += align256(bytes);
    return q;
  };
  const lbk_bell* w[2] = {w2, w1};
  const int c[2] = {C_d, C_in};
  TListJob lj[2], ljn[2];
  int nl = 0;
  for (int t = 0; t < 2; ++t) {
    lj[t] = TListJob{w[t]->col_idx, w[t]->R, w[t]->K, c[t], nullptr, nullptr};
    lj[t].cnt = reinterpret_cast<int32_t*>(take((size_t)c[t] * 4));
    lj[t].list = reinterpret_cast<int32_t*>(take((size_t)c[t] * w[t]->R * w[t]->K * 4));
    if ((int64_t)w[t]->R * w[t]->K > 0) ljn[nl++] = lj[t];
  }
  uint16_t* da = reinterpret_cast<uint16_t*>(take((size_t)N * d_ff * 2));
  const size_t f1 = dw_part_floats(N, w1, C_in, d_ff), f2 = dw_part_floats(N, w2, C_d, d_model);
  float* part = reinterpret_cast<float*>(take((f1 + f2) * 4));
  float* asum = reinterpret_cast<float*>(take(dh_sum_floats(N, d_ff) * 4));
  float* cpart = reinterpret_cast<float*>(p);
  int64_t sum_rows = 0;
  if (N > 0) {
    if (nl && launch_tlist(ljn, nl, s)) return LBK_ERR_LAUNCH;
    // da = (dy W2) gelu'(pre)
    TProdArgs a{};
    if (t2 > 0) a.src[a.nsrc++] = TProdSrc{grad_out, d_model, w2->values, w2->K, lj[0].cnt, lj[0].list, t2};
    a.N = N; a.C = C_d; a.ldo = d_ff;
    a.g = pre; a.dg = da;
    if (d_b1) sum_rows = dh_sum_blocks(B, a);
    if (sum_rows) a.dgsum = asum;
    if (launch_tprod(B, 2, a, s)) return LBK_ERR_LAUNCH;
    // dx = da W1
    TProdArgs b{};
    if (t1 > 0) b.src[b.nsrc++] = TProdSrc{da, d_ff, w1->values, w1->K, lj[1].cnt, lj[1].list, t1};
    b.N = N; b.C = C_in; b.ldo = d_model;
    b.out = dx;
    if (launch_tprod(B, 1, b, s)) return LBK_ERR_LAUNCH;
  }
  DWJob dj[2];
  int nj = 0;
  if (t1 > 0)
    dj[nj++] = DWJob{x, d_model, da, d_ff, w1->col_idx, w1->R, w1->K, C_in, part, nullptr, d_v1, 0, nullptr, nullptr, 0, 0};
  if (t2 > 0)
    dj[nj++] = DWJob{h, d_ff, grad_out, d_model, w2->col_idx, w2->R, w2->K, C_d, part + f1, nullptr, d_v2, 0,
                     N > 0 ? lj[0].cnt : nullptr, N > 0 ? lj[0].list : nullptr, 0, 0};
  if (nj && launch_dw(B, dj, nj, N, s)) return LBK_ERR_LAUNCH;
  ColsumJob cj[2];
  int nc = 0;
  if (d_b1 && d_ff > 0)
    cj[nc++] = ColsumJob{sum_rows ? nullptr : da, d_ff, (int)d_ff, d_b1, asum, (int)sum_rows, 0};
  if (d_b2) cj[nc++] = ColsumJob{grad_out, d_model, d_model, d_b2, nullptr, 0, 0};
  if (nc && launch_colsum(cj, nc, N, cpart, s)) return LBK_ERR_LAUNCH;
  return LBK_OK;
}

size_t lbk_block_ell_matmul_bwd_workspace_bytes(int64_t N, int32_t in_features, const lbk_bell* w) {
  if (!w || N < 0 || in_features <= 0 || !tile_ok(w->B) || in_features % w->B) return 0;
  const int C = in_features / w->B;
  return tlist_bytes(w, C) + align256(dw_part_floats(N, w, C, (int64_t)w->R * w->B) * 4);
}

size_t lbk_block_ell_matmul_bwd_bias_workspace_bytes(int64_t N, int32_t in_features, const lbk_bell* w) {
  const size_t base = lbk_block_ell_matmul_bwd_workspace_bytes(N, in_features, w);
  return base ? base + align256(colsum_bytes(N, (int64_t)w->R * w->B)) : 0;
}

int lbk_block_ell_matmul_bwd_bf16(const uint16_t* grad_out, const uint16_t* x, int64_t N, int32_t in_features,
                                  const lbk_bell* w, uint16_t* dx, uint16_t* d_values, void* workspace,
                                  size_t workspace_bytes, void* stream) {
  return lbk_block_ell_matmul_bwd_bias_bf16(grad_out, x, N, in_features, w, dx, d_values, nullptr, workspace,
                                            workspace_bytes, stream);
}

int lbk_block_ell_matmul_bwd_bias_bf16(const uint16_t* grad_out, const uint16_t* x, int64_t N, int32_t in_features,
                                       const lbk_bell* w, uint16_t* dx, uint16_t* d_values, float* d_bias,
                                       void* workspace, size_t workspace_bytes, void* stream) {
  int st;
  if ((st = check_bell(w))) return st;
  if (N < 0 || in_features <= 0) return LBK_ERR_ARG;
  const int B = w->B;
  if (in_features % B) return LBK_ERR_SHAPE;
  const int C = in_features / B;
  const int64_t nt = (int64_t)w->R * w->K, out_f = (int64_t)w->R * B;
  if (d_values && !a16(d_values)) return LBK_ERR_ALIGN;
  if (nt > 0 && !a16(w->values)) return LBK_ERR_ALIGN;
  if (N > 0 && (dx || d_values || d_bias)) {
    if (!grad_out || (d_values && !x)) return LBK_ERR_NULL;
    if (!a16(grad_out) || (x && !a16(x)) || (dx && !a16(dx)) || in_features % 8) return LBK_ERR_ALIGN;
  }
  const size_t need = d_bias ? lbk_block_ell_matmul_bwd_bias_workspace_bytes(N, in_features, w)
                             : lbk_block_ell_matmul_bwd_workspace_bytes(N, in_features, w);
  if (!workspace || workspace_bytes < need) return LBK_ERR_WORKSPACE;
  if (!a16(workspace)) return LBK_ERR_ALIGN;
  hipStream_t s = S(stream);
  char* p = static_cast<char*>(workspace);
  auto take = [&](size_t bytes) {
    char* q = p;
    p += align256(bytes);
    return q;
  };
  TListJob lj{};
  lj.col = w->col_idx; lj.R = w->R; lj.K = w->K; lj.C = C;
  lj.cnt = reinterpret_cast<int32_t*>(take((size_t)C * 4));
  lj.list = reinterpret_cast<int32_t*>(take((size_t)C * w->R * w->K * 4));
  float* part = reinterpret_cast<float*>(p);
  if (dx && N > 0) {
    // dx = dy W: out[:, c] = sum over the slots of column block c of dy[:, r] W[r,k]^T (with no
    // tiles at all the product kernel writes zeros)
    if (nt > 0 && launch_tlist(&lj, 1, s)) return LBK_ERR_LAUNCH;
    TProdArgs a{};
    a.nsrc = 0;
    if (nt > 0) a.src[a.nsrc++] = TProdSrc{grad_out, out_f, w->values, w->K, lj.cnt, lj.list, nt};
    a.N = N; a.C = C; a.ldo = in_features;
    a.out = dx;
    if (launch_tprod(B, 1, a, s)) return LBK_ERR_LAUNCH;
  }
  if (d_values && nt > 0) {
    // the transposed lists exist when dx was computed above
    const bool lists = dx && N > 0;
    DWJob dj{x, in_features, grad_out, out_f, w->col_idx, w->R, w->K, C, part, d_values, nullptr, 0,
             lists ? lj.cnt : nullptr, lists ? lj.list : nullptr, 0, 0};
    if (launch_dw(B, &dj, 1, N, s)) return LBK_ERR_LAUNCH;
  }
  if (d_bias && out_f > 0) {
    // the column-sum partials follow the tile partials
    float* cpart = reinterpret_cast<float*>(reinterpret_cast<char*>(part) +
                                            align256(dw_part_floats(N, w, C, out_f) * 4));
    const ColsumJob cj{grad_out, out_f, (int)out_f, d_bias, nullptr, 0};
    if (launch_colsum(&cj, 1, N, cpart, s)) return LBK_ERR_LAUNCH;
  }
  return LBK_OK;
}

// ---- topology transforms
int lbk_topology_alive_counts(const uint8_t* alive, int32_t R, int32_t K, int32_t* counts, int32_t* max_count,
                              void* stream) {
  if (R < 0 || K < 0) return LBK_ERR_ARG;
  if (!max_count || (R > 0 && (!counts || (K > 0 && !alive)))) return LBK_ERR_NULL;
  return launch_topo_count(alive, R, K, counts, max_count, S(stream)) == 0 ? LBK_OK : LBK_ERR_LAUNCH;
}

int lbk_topology_compact_bf16(const uint16_t* values, const int32_t* col_idx, const uint8_t* alive, int32_t R,
                              int32_t K, int32_t B, int32_t K_new, uint16_t* out_values, int32_t* out_col_idx,
                              uint8_t* out_alive, void* stream) {
  if (!tile_ok(B)) return LBK_ERR_TILE;
  if (R < 0 || K < 1 || K_new < 1 || K_new > K) return LBK_ERR_ARG;
  if (R == 0) return LBK_OK;
  if (!values || !col_idx || !alive || !out_values || !out_col_idx || !out_alive) return LBK_ERR_NULL;
  if (!a16(values) || !a16(out_values)) return LBK_ERR_ALIGN;
  return launch_topo_compact(values, col_idx, alive, R, K, B, K_new, out_values, out_col_idx, out_alive,
                             S(stream)) == 0 ? LBK_OK : LBK_ERR_LAUNCH;
}

int lbk_column_importance(const int32_t* fc1_col_idx, const uint8_t* fc1_alive, int32_t R1, int32_t K1,
                          const uint8_t* fc2_alive, int32_t R2, int32_t K2, int32_t C_ff, float* importance,
                          void* stream) {
  if (R1 < 0 || K1 < 0 || R2 < 0 || K2 < 0 || C_ff < 1 || C_ff > 16384) return LBK_ERR_ARG;
  if (!importance || ((int64_t)R1 * K1 > 0 && (!fc1_col_idx || !fc1_alive)) || ((int64_t)R2 * K2 > 0 && !fc2_alive))
    return LBK_ERR_NULL;
  return launch_topo_importance(fc1_col_idx, fc1_alive, (int64_t)R1 * K1, fc2_alive, R2, K2, C_ff, importance,
                                S(stream)) == 0 ? LBK_OK : LBK_ERR_LAUNCH;
}

int lbk_column_permutation(const float* importance, int32_t C_ff, int32_t* perm, void* stream) {
  if (C_ff < 1 || C_ff > 16384) return LBK_ERR_ARG;
  if (!importance || !perm) return LBK_ERR_NULL;
  return launch_topo_perm(importance, C_ff, perm, S(stream)) == 0 ? LBK_OK : LBK_ERR_LAUNCH;
}

int lbk_apply_permutation_bf16(const uint16_t* values, const int32_t* col_idx, const uint8_t* alive, int32_t R,
                               int32_t K, int32_t B, const int32_t* perm, int32_t C_ff, int32_t is_column_dim,
                               uint16_t* out_values, int32_t* out_col_idx, uint8_t* out_alive, void* stream) {
  if (!tile_ok(B)) return LBK_ERR_TILE;
  if (R < 0 || K < 0 || C_ff < 1 || C_ff > 16384) return LBK_ERR_ARG;
  if (!is_column_dim && R != C_ff) return LBK_ERR_SHAPE;
  if ((int64_t)R * K == 0) return LBK_OK;
  if (!col_idx || !perm || !out_col_idx) return LBK_ERR_NULL;
  // column mode leaves tiles and flags in place when out_values / out_alive are null
  if (!is_column_dim && (!out_values || !out_alive)) return LBK_ERR_NULL;
  if ((out_values && !values) || (out_alive && !alive)) return LBK_ERR_NULL;
  if (out_values && (!a16(values) || !a16(out_values))) return LBK_ERR_ALIGN;
  return launch_topo_apply(values, col_idx, alive, R, K, B, perm, C_ff, is_column_dim ? 1 : 0, out_values,
                           out_col_idx, out_alive, S(stream)) == 0 ? LBK_OK : LBK_ERR_LAUNCH;
}

int lbk_k_active_macros(const int32_t* col_idx, const uint8_t* alive, int32_t R, int32_t K, int32_t tiles_per_macro,
                        int32_t* k_active, void* stream) {
  if (R < 0 || K < 0 || tiles_per_macro < 1) return LBK_ERR_ARG;
  if (!k_active || ((int64_t)R * K > 0 && (!col_idx || !alive))) return LBK_ERR_NULL;
  return launch_topo_kactive(col_idx, alive, (int64_t)R * K, tiles_per_macro, k_active, S(stream)) == 0
             ? LBK_OK
             : LBK_ERR_LAUNCH;
}

int lbk_gather_rows(const void* src, int64_t n_src, int64_t row_bytes, const int32_t* perm, int64_t n_dst,
                    void* dst, void* stream) {
  if (n_src < 0 || n_dst < 0 || row_bytes < 0 || n_src > INT32_MAX || n_dst > INT32_MAX) return LBK_ERR_ARG;
  if (n_dst == 0 || row_bytes == 0) return LBK_OK;
  if (n_src == 0) return LBK_ERR_SHAPE;
  if (!src || !perm || !dst) return LBK_ERR_NULL;
  return launch_topo_gather(src, row_bytes, perm, (int)n_src, (int)n_dst, dst, S(stream)) == 0 ? LBK_OK
                                                                                                : LBK_ERR_LAUNCH;
}

int lbk_transposed_index(const int32_t* col_idx, int32_t R, int32_t K, int32_t C, int32_t* col_ptr,
                         int32_t* entries, void* stream) {
  if (R < 0 || K < 0 || C < 1 || C > 16384 || (int64_t)R * K > INT32_MAX) return LBK_ERR_ARG;
  if (!col_ptr || ((int64_t)R * K > 0 && (!col_idx || !entries))) return LBK_ERR_NULL;
  return launch_topo_csc(col_idx, R, K, C, col_ptr, entries, S(stream)) == 0 ? LBK_OK : LBK_ERR_LAUNCH;
}

static bool elem_ok(int e, const void* p) {
  return (e == 2 || e == 4) && (reinterpret_cast<uintptr_t>(p) % (uintptr_t)e) == 0;
}

int lbk_dense_to_block_ell(const void* dense, int64_t ld, int32_t elem_bytes, int32_t R, int32_t C, int32_t B,
                           const int32_t* col_idx, int32_t K, void* values, void* stream) {
  if (!tile_ok(B)) return LBK_ERR_TILE;
  if (R < 0 || C < 1 || K < 0 || R > 65535 || ld < (int64_t)C * B) return LBK_ERR_ARG;
  if ((int64_t)R * K == 0) return LBK_OK;
  if (!dense || !col_idx || !values) return LBK_ERR_NULL;
  if (!elem_ok(elem_bytes, dense) || !elem_ok(elem_bytes, values)) return LBK_ERR_ALIGN;
  return launch_fmt_from_dense(dense, ld, elem_bytes, R, C, B, col_idx, K, values, S(stream)) == 0
             ? LBK_OK
             : LBK_ERR_LAUNCH;
}

int lbk_block_ell_to_dense(const void* values, const int32_t* col_idx, int32_t R, int32_t K, int32_t B, int32_t C,
                           int32_t elem_bytes, void* dense, int64_t ld, void* stream) {
  if (!tile_ok(B)) return LBK_ERR_TILE;
  if (R < 0 || C < 0 || K < 0 || R > 65535 || ld < (int64_t)C * B) return LBK_ERR_ARG;
  if ((int64_t)R * C == 0) return LBK_OK;
  if (!dense || (K > 0 && (!values || !col_idx))) return LBK_ERR_NULL;
  if (!elem_ok(elem_bytes, dense) || (K > 0 && !elem_ok(elem_bytes, values))) return LBK_ERR_ALIGN;
  return launch_fmt_to_dense(values, col_idx, R, K, B, C, elem_bytes, dense, ld, S(stream)) == 0 ? LBK_OK
                                                                                                : LBK_ERR_LAUNCH;
}

int lbk_block_ell_topk_columns(const void* dense, int64_t ld, int32_t elem_bytes, int32_t R, int32_t C, int32_t B,
                               int32_t K, int32_t* col_idx_out, void* stream) {
  if (!tile_ok(B)) return LBK_ERR_TILE;
  if (R < 0 || C < 1 || C > 16384 || K < 1 || K > C || ld < (int64_t)C * B) return LBK_ERR_ARG;
  if (R == 0) return LBK_OK;
  if (!dense || !col_idx_out) return LBK_ERR_NULL;
  // the norms read 16-byte chunks: rows and the base must be 16-byte aligned
  if (!elem_ok(elem_bytes, dense) || !a16(dense) || (ld * elem_bytes) % 16) return LBK_ERR_ALIGN;
  return launch_fmt_topk(dense, ld, elem_bytes, R, C, B, K, col_idx_out, S(stream)) == 0 ? LBK_OK : LBK_ERR_LAUNCH;
}

int lbk_ternary_check_codes(const uint32_t* words, int64_t n_words, int32_t* bad_count, void* stream) {
  if (n_words < 0) return LBK_ERR_ARG;
  if (!bad_count || (n_words > 0 && !words)) return LBK_ERR_NULL;
  return launch_fmt_ternary_check(words, n_words, bad_count, S(stream)) == 0 ? LBK_OK : LBK_ERR_LAUNCH;
}

}  // extern "C"
