// Factored (Adafactor row/column) optimizer step for MI355X (gfx950).
//
// One group step is a few launches over every tensor of the group:
//   k_fstats   2-D tiles of up to kTRS rows x 1024 columns: row sums and column
//              sums of g^2 (and sum p^2 for the relative step size), written as
//              per-tile partials -- no atomics, so the result is deterministic;
//   k_fcolsum  (tensors of more than 1024 rows) the column partials summed over
//              groups of strips, in parallel;
//   k_fblock   one workgroup per AL block of each row/column vector: reduce the
//              partials in a fixed order, EMA the second moment, refit and
//              re-encode the block (columns: inv_col in place);
//   k_frows    one workgroup per tensor: the row mean, inv_row, the step size
//              and the weight-decay factor;
//   k_fupdt    on tiles of 32 rows x 1024 columns (k_fupdate, flat 2048-element units, for
//              the few tensors whose column count rules tiles out): the update
//              u = (x * inv_row) * inv_col with x = g or the momentum EMA, the
//              parameter write and the momentum re-encode.  With RMS clipping
//              or Fira it runs twice: first for sum(u^2) per tile, then (after
//              k_fnorm) to apply;
//   k_fnorm    one workgroup per tensor: ||u||, the Fira limiter and the step.
// CAME (beta3) adds, between k_frows and the update:
//   k_fclip    the RMS clip factor of U = (g * inv_row) * inv_col (after a
//              norm pass over U, only when d > 0);
//   k_came1    the same 2-D tiles as k_fstats: U / clip, the momentum EMA M',
//              and row/column sums of the residual (U - M')^2 + eps_came;
//   k_fcolsum, k_fblock, k_frows again, on the residual sums: the confidence
//              EMA, its AL re-encode and inv_conf_row / inv_conf_col;
// and the update becomes (M' * inv_conf_row) * inv_conf_col (optimizer.py:929-956).
// Numbers follow the reference's PyTorch path (optimizer.py:2198-2252 and
// _fallback_2d_update 920-970): means are sum/count of the fp32 squares,
// inv_row = 1/sqrt(row/r) and inv_col = 1/sqrt(col) with IEEE division and
// square root, and u is formed as (x * inv_row) * inv_col.
#include "a8_common.cuh"
#include "a8_mcodec.cuh"
#include "a8_abi_impl.h"

namespace a8 {

constexpr int kTR = 32;      // minimum rows per statistics tile
constexpr int kTC = 1024;    // columns per statistics tile (256 lanes x 4)
constexpr int kUnit = 2048;  // elements per update workgroup
constexpr int kScal = 8;     // per-tensor scalars in the workspace
constexpr int kMkFp32 = 5;   // HyperF::mk of fp32 momentum (codecs are 1-4)

// Per-tensor workspace layout (offsets in floats).  The partial sums are doubles:
// every statistic (row / column means, sum p^2, ||u||^2) is accumulated in double
// from its first term and rounded to float once, so it is the correctly rounded
// sum in all but vanishingly rare cases, whatever the tiling.  The double regions
// come first and have even sizes, so each starts 8-byte aligned (the workspace
// itself is 256-byte aligned).
struct FWs {
  int64_t rowpart;   // double [nchunk][B*R]       row partial sums
  int64_t colpart;   // double [B][nstrip][C]      column partial sums
  int64_t colsum;    // double [B][nsplit][C]      column sums over groups of gss strips of kTRS rows
  int64_t p2;        // double [ntile]             partial sum p^2
  int64_t npart;     // double [max(nunit, nutile)] partial sums u^2 (per unit or per update tile)
  int64_t invr;      // [B*R]              new row V, then inv_row
  int64_t invc;      // [B*C]              new column V, then inv_col
  int64_t icr;       // [B*R]              CAME: new row confidence, then its inverse root
  int64_t icc;       // [B*C]              CAME: new column confidence, then its inverse root
  int64_t scal;      // [8]: alpha, step, fira scale, decay, CAME clip factor
  int64_t total;
  int64_t nchunk, nstrip, ntile, nunit;
  int64_t nsplit;    // strip groups of the column reduction (1: k_fblock reads colpart)
  int64_t tr;        // rows per statistics tile
  int64_t fold;      // strips per kTRS rows
  int64_t nss, gss;  // strips of kTRS rows, and how many of them a k_fcolsum workgroup sums
  int64_t nustrip, nutile;   // update tiles: kTR rows x 1024 columns
};

// Tile geometry.  The update passes (k_fupdt) run on tiles of kTR = 32 rows x
// 1024 columns, which stream best for them.  The statistics passes (k_fstats,
// k_came1) take kTRS rows per tile in large groups: each tile ends with a write of its row
// and column partials, and such writes spread through the read stream cost far
// more bandwidth than their bytes, so fewer, taller tiles write less often.  The
// column partials of tall matrices are reduced in parallel by k_fcolsum before k_fblock.
//
// The order of every sum over rows (the columns' and sum p^2) is a function of the tensor
// alone: rows in kTR at a time, those partials in turn over kTRS rows, and these over groups
// of gss.  A tall tile adds its kTR-row partials itself; short tiles leave them to the
// reductions.  So a matrix steps to the same bits alone and in any group.
#ifndef A8_TRS
#define A8_TRS 256
#endif
constexpr int kTRS = A8_TRS;
static_assert(kTRS % kTR == 0, "a tall tile holds whole short ones");

// Rows of the statistics tiles of a group of `total` elements.  Tall tiles need about 900 of
// them, three and a half workgroups for each of the 256 CUs: a 44 M-parameter layer had 176
// tiles of 256 rows, less than one workgroup per CU (k_fstats 64 -> 24 us in tiles of 32
// rows, k_came1 144 -> 52).  Steps, tiles of 32 / 256 rows: 141 M bf16 elements CAME 605 /
// 663 us; 201 M Adafactor bf16 508 / 520, fp32 943 / 941, CAME bf16 821 / 850; 262 M
// Adafactor bf16 674 / 636, fp32 1222 / 1127, CAME bf16 1013 / 977.
static int64_t fws_tile_rows(int64_t R, int64_t total) {
  const int64_t rows = total > (int64_t)kTRS * kTC * 896 ? kTRS : kTR;
  const int64_t r = (R + kTR - 1) / kTR * kTR;
  return r < rows ? r : rows;
}

__host__ __device__ inline FWs fws_layout(int64_t B, int64_t R, int64_t C, int64_t tr) {
  FWs w;
  w.nchunk = (C + kTC - 1) / kTC;
  w.tr = tr;
  w.nstrip = (R + w.tr - 1) / w.tr;
  w.ntile = B * w.nstrip * w.nchunk;
  w.nustrip = (R + kTR - 1) / kTR;
  w.nutile = B * w.nustrip * w.nchunk;
  w.nunit = (B * R * C + kUnit - 1) / kUnit;
  w.fold = tr == kTR ? kTRS / kTR : 1;   // (fewer than kTRS rows make one tile, or are folded)
  w.nss = (R + kTRS - 1) / kTRS;
  int lg = 2;
  while (w.nss > (int64_t)64 << lg) ++lg;
  w.gss = (int64_t)1 << lg;
  w.nsplit = (w.nss + w.gss - 1) >> lg;
  w.rowpart = 0;
  w.colpart = w.rowpart + 2 * w.nchunk * B * R;
  w.colsum = w.colpart + 2 * B * w.nstrip * C;
  w.p2 = w.colsum + (w.nsplit > 1 ? 2 * B * w.nsplit * C : 0);
  w.npart = w.p2 + 2 * w.ntile;
  w.invr = (w.npart + 2 * (w.nunit > w.nutile ? w.nunit : w.nutile) + 31) / 32 * 32;   // whole lines
  w.invc = w.invr + B * R;
  w.icr = w.invc + B * C;
  w.icc = w.icr + B * R;
  w.scal = w.icc + B * C;
  w.total = w.scal + kScal;
  return w;
}

__device__ __forceinline__ double* ws_dp(float* ws, int64_t off) { return reinterpret_cast<double*>(ws + off); }
__device__ __forceinline__ const double* ws_dp(const float* ws, int64_t off) {
  return reinterpret_cast<const double*>(ws + off);
}

struct DescF {
  void* param;
  const void* grad;
  uint8_t* m_q;
  float* m_scale;
  void* row_q;
  float* row_scale;
  float* row_min_log;
  float* row_var;
  void* col_q;
  float* col_scale;
  float* col_min_log;
  float* col_var;
  void* crow_q;        // CAME confidence state (codes or fp32), as row/col V
  float* crow_scale;
  float* crow_min_log;
  float* crow_var;
  void* ccol_q;
  float* ccol_scale;
  float* ccol_min_log;
  float* ccol_var;
  float* ws;
  const float* lr;
  float* fira_prev;
  float* m;            // fp32 momentum (MK 3), or null
  int64_t B, R, C, numel;
  int64_t tile_begin;  // first statistics tile of this tensor
  int64_t utile_begin; // first update tile
  int64_t unit_begin;
  int64_t fblk_begin;  // first k_fblock workgroup of this tensor
  int64_t cs_begin;    // first k_fcolsum workgroup of this tensor
  int64_t nbr;         // AL blocks of the row vector (the column vector follows)
  uint64_t sr_seed;
  int has_fira_prev;
  int tiled;           // update runs on tiles (k_fupdt; 2: C % 4 != 0), 0: flat units
  int tr;              // rows per statistics tile
  int elem;            // statistics load element by element (fewer than 4 columns, rows of 4 GB and more)
};

struct HyperF {
  float bv;            // V lerp weight
  float eps1;
  float eps2;
  float lr_val;
  float bias_factor;
  float wd;
  float d;
  float margin;        // 1 + fira_margin
  float floor_;
  float w_m;           // momentum lerp weight (1 - beta1)
  float w_c;           // CAME confidence lerp weight (1 - beta3)
  float eps_came;
  int came;
  int bias_mode;
  int scale_param;
  int wd_mode;
  int fira;
  int block_size;      // V block size
  int mk;              // momentum codec (0 none, 1 UF8, 2 UF4, 3 D8, 4 D4)
  int lbm;             // log2(m_block_size); -1: B_M not a power of two in [32, 2048]
  int bm;              // B_M when lbm < 0 (k_fupdate_gen), else 0
  int unit;            // elements per k_fupdate_gen workgroup (a whole number of M blocks)
  uint64_t sr_step;
  const a8_step_scalars* dsc;   // if set: this step's V lerp weight, lr, bias factor and SR step
};

// The per-step fields from the device block of a8_step_advance, when given.
__device__ __forceinline__ void hf_step(HyperF& h) {
  if (!h.dsc) return;
  const a8_step_scalars sc = load_step_scalars(h.dsc);
  h.bv = (float)sc.beta_val;
  h.lr_val = sc.rho;
  h.bias_factor = sc.bias_factor;
  h.sr_step = sc.step;
}

__device__ __forceinline__ const DescF* find_tile(const DescF* tab, int n, int64_t wg) {
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (tab[mid].tile_begin <= wg) lo = mid; else hi = mid - 1;
  }
  return tab + lo;
}

__device__ __forceinline__ const DescF* find_utile(const DescF* tab, int n, int64_t wg) {
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (tab[mid].utile_begin <= wg) lo = mid; else hi = mid - 1;
  }
  return tab + lo;
}

__device__ __forceinline__ const DescF* find_unit(const DescF* tab, int n, int64_t wg) {
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (tab[mid].unit_begin <= wg) lo = mid; else hi = mid - 1;
  }
  return tab + lo;
}

// Workgroup-wide reductions (256 lanes, 4 waves) through 4 LDS slots; every
// lane gets the result.  The cross-wave order is fixed.
__device__ __forceinline__ double wg_sum_d(double x, double* s4) {
  x = grp_sum_d(x, 64);
  const int lane = threadIdx.x;
  __syncthreads();
  if ((lane & 63) == 0) s4[lane >> 6] = x;
  __syncthreads();
  return ((s4[0] + s4[1]) + s4[2]) + s4[3];
}

__device__ __forceinline__ uint32_t nz_key_f(float v) { return __float_as_uint(v) - 1u; }

// Maximum and minimum key over a workgroup of up to 16 waves; s32: 32 floats of LDS.
__device__ __forceinline__ void wg_maxkey(float& mx, uint32_t& key, float* s32) {
  mx = grp_max(mx, 64);
  key = grp_umin(key, 64);
  const int lane = threadIdx.x, nw = (int)blockDim.x >> 6;
  __syncthreads();
  if ((lane & 63) == 0) {
    s32[lane >> 6] = mx;
    s32[16 + (lane >> 6)] = __uint_as_float(key);
  }
  __syncthreads();
  for (int w = 0; w < nw; ++w) {
    mx = fmaxf(mx, s32[w]);
    key = min(key, __float_as_uint(s32[16 + w]));
  }
}

// ------------------------------------------------------------ statistics
// Tile layout of the two statistics kernels (k_fstats, k_came1): wave w of the
// workgroup owns columns c_base + 256 w .. + 255 of every row of the tile, a lane
// one 4-column window.  A lane's column sums therefore cover the whole tile in
// four registers (double), written straight to the column partials; the row sums
// are kept per lane for kRB rows at a time and then reduce-scattered across the
// wave (one 6-step butterfly for all kRB rows), the four waves' row partials
// meeting in LDS at the end of the tile.  Every load of a batch of rows is issued
// before its arithmetic: rows beyond the tile and windows beyond C read a valid
// address (the tile's first row, column 0) and count zero.
constexpr int kRB = 4;   // rows per row-sum batch

// Sum of v[0..3] over the 64 lanes of the wave for each k, scattered: on return
// every lane holds the total of v[k] for k = row_of_lane(lane).
__device__ __forceinline__ double reduce_scatter4(const double* v, int wl) {
  const bool b5 = (wl & 32) != 0, b4 = (wl & 16) != 0;
  double a[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const double mine = b5 ? v[k + 2] : v[k];
    const double other = b5 ? v[k] : v[k + 2];
    a[k] = mine + __shfl_xor(other, 32, 64);
  }
  double x = (b4 ? a[1] : a[0]) + __shfl_xor(b4 ? a[0] : a[1], 16, 64);
  x += __shfl_xor(x, 8, 64);
  x += __shfl_xor(x, 4, 64);
  x += __shfl_xor(x, 2, 64);
  x += __shfl_xor(x, 1, 64);
  return x;
}

__device__ __forceinline__ int row_of_lane(int wl) { return ((wl >> 5) & 1) * 2 + ((wl >> 4) & 1); }

// Four consecutive elements at a per-lane 32-bit element offset from a
// workgroup-uniform row pointer.  The offset is scaled to bytes in 32 bits (rows
// of a tensor are far below 4 GiB apart... the offset is below C * sizeof(T)), so
// the address is a scalar base plus a zero-extended vector offset: the saddr form
// of the global load, with no 64-bit address per lane.
// (The row pointer passes through readfirstlane: it is uniform anyway, and the
// opaque step keeps loop strength reduction from turning base + offset back into
// one 64-bit induction pointer per load.)
template <typename T>
__device__ __forceinline__ const char* at_off(const T* row, uint32_t off) {
  const uint64_t v = reinterpret_cast<uint64_t>(row);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return reinterpret_cast<const char*>(((uint64_t)hi << 32) | lo) + (off * (uint32_t)sizeof(T));
}

// The types say what alignment the address has: a row of a tensor whose column count is
// no multiple of the vector starts on any element, and global loads need no more (one
// instruction all the same; a lane that straddles a cache line costs a second request).
typedef f32x4 f32x4_e __attribute__((aligned(4)));
typedef u32x2 u32x2_e __attribute__((aligned(2)));
typedef uint32_t u32_e __attribute__((aligned(1)));
typedef f64x2 f64x2_e __attribute__((aligned(8)));

template <typename T, typename V>
__device__ __forceinline__ void load4o(const T* row, uint32_t off, V* out) {
  if constexpr (sizeof(T) == 8) {
    const A8_G f64x2_e* p = ((const A8_G f64x2_e*)(at_off(row, off)));
    const f64x2 a = __builtin_nontemporal_load(p), b = __builtin_nontemporal_load(p + 1);
    out[0] = (V)a.x; out[1] = (V)a.y; out[2] = (V)b.x; out[3] = (V)b.y;
  } else if constexpr (sizeof(T) == 4) {
    const f32x4 a = __builtin_nontemporal_load(((const A8_G f32x4_e*)(at_off(row, off))));
    out[0] = a.x; out[1] = a.y; out[2] = a.z; out[3] = a.w;
  } else {
    const u32x2 a = __builtin_nontemporal_load(((const A8_G u32x2_e*)(at_off(row, off))));
    const T* h = reinterpret_cast<const T*>(&a);
#pragma unroll
    for (int k = 0; k < 4; ++k) out[k] = to_f<T>(h[k]);
  }
}

// A lane's window of four columns in a row of C (a multiple of 4 or not, C >= 4).  The
// window that C cuts loads the row's last four elements instead and moves its own to the
// front (win_fix), zeros behind them, so every load is a full one inside the row.
struct Win {
  uint32_t cl;   // column the load starts at
  int n;         // columns of the window inside C (0: none, the load reads the base column)
};
__device__ __forceinline__ Win win_at(int64_t c0, int64_t C, int64_t base) {
  Win w;
  w.n = c0 >= C ? 0 : (C - c0 >= 4 ? 4 : (int)(C - c0));
  // an empty window reads the base column's window, itself moved left when C cuts it
  const int64_t c = w.n > 0 ? c0 : base;
  w.cl = (uint32_t)(c + 4 <= C ? c : C - 4);
  return w;
}
// cut: the columns a cut window keeps, C % 4 (uniform)
template <typename V>
__device__ __forceinline__ void win_fix(const Win& w, int cut, V* v) {
  V t[4] = {v[3], (V)0, (V)0, (V)0};
  if (cut == 2) { t[0] = v[2]; t[1] = v[3]; }
  if (cut == 3) { t[0] = v[1]; t[1] = v[2]; t[2] = v[3]; }
#pragma unroll
  for (int k = 0; k < 4; ++k) v[k] = (w.n & 3) ? t[k] : v[k];
}

// A window element by element (DescF::elem); every load is issued, inside the row.
template <typename T, typename V>
__device__ __forceinline__ void load_tiny(const T* row, int64_t c0, int64_t C, V* out) {
#pragma unroll
  for (int k = 0; k < 4; ++k) out[k] = ld1<T, V>(row, c0 + k < C ? c0 + k : C - 1);
#pragma unroll
  for (int k = 0; k < 4; ++k) out[k] = c0 + k < C ? out[k] : (V)0;
}

// Where a statistics workgroup sits: tensor-local tile t, chunk, strip, batch.
struct TilePos {
  int64_t t, ch, s, b, r_lo, r_hi, c_base;
};

// (UPD: an update tile of kTR rows, else a statistics tile of W.tr rows.)
template <bool UPD>
__device__ __forceinline__ TilePos tile_pos(const DescF& D, const FWs& W) {
  TilePos q;
  q.t = (int64_t)blockIdx.x - (UPD ? D.utile_begin : D.tile_begin);
  const int64_t tr = UPD ? kTR : W.tr;
  const uint32_t t32 = (uint32_t)q.t, nch = (uint32_t)W.nchunk, nst = (uint32_t)(UPD ? W.nustrip : W.nstrip);
  const uint32_t bs = t32 / nch;
  q.ch = (int64_t)(t32 - bs * nch);
  q.b = (int64_t)(bs / nst);
  q.s = (int64_t)(bs - (uint32_t)q.b * nst);
  q.r_lo = q.s * tr;
  q.r_hi = (q.r_lo + tr < D.R) ? q.r_lo + tr : D.R;
  q.c_base = q.ch * kTC;
  return q;
}

// The four waves' row partials of the tile (LDS, [4][kTRS]) summed in a fixed
// order into the chunk's row partials.
__device__ __forceinline__ void tile_rows_out(const double* s_row, double* rowpart, int64_t r_lo, int64_t r_hi) {
  __syncthreads();
  for (int i = threadIdx.x; i < r_hi - r_lo; i += 256) {
    const double v = ((s_row[i] + s_row[kTRS + i]) + s_row[2 * kTRS + i]) + s_row[3 * kTRS + i];
    gp(rowpart)[r_lo + i] = v;
  }
}

// A lane's column sums of kTR rows (acc) to its sums of the tile so far in LDS (tot; in
// registers they cost a wave per SIMD).  The tile's last kTR rows stay in acc.
__device__ __forceinline__ void col_fold(double* acc, double* tot) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    tot[256 * e] += acc[e];
    acc[e] = 0.0;
  }
}
__device__ __forceinline__ double col_sum(const double* acc, const double* tot, int e, const TilePos& q) {
  return q.r_hi - q.r_lo > kTR ? tot[256 * e] + acc[e] : acc[e];
}

// CUT: C cuts one of the wave's windows (C % 4 columns remain of it).  TINY: DescF::elem.
template <typename T, bool PSQ, bool CUT, bool TINY>
__device__ __forceinline__ void fstats_tile(const DescF& D, const TilePos& q, int64_t c0, double* acc, double* tot,
                                            double* s_psq, double* s_row) {
  const T* G = reinterpret_cast<const T*>(D.grad);
  const T* P = reinterpret_cast<const T*>(D.param);
  const int64_t R = D.R, C = D.C;
  const int wl = threadIdx.x & 63;
  const Win w = win_at(c0, C, 0);
  const bool act = w.n > 0;
  const int cut = (int)(C & 3);
  float g[kRB][4], pv[kRB][PSQ ? 4 : 1];
  bool rv[kRB];
  auto issue = [&](int64_t r0) {
#pragma unroll
    for (int k = 0; k < kRB; ++k) {
      const int64_t r = r0 + k;
      rv[k] = r < q.r_hi;
      const int64_t rowbase = (q.b * R + (rv[k] ? r : q.r_lo)) * C;
      if constexpr (TINY) {
        load_tiny<T>(G + rowbase, c0, C, g[k]);
        if constexpr (PSQ) load_tiny<T>(P + rowbase, c0, C, pv[k]);
      } else {
        load4o<T>(G + rowbase, w.cl, g[k]);
        if constexpr (PSQ) load4o<T>(P + rowbase, w.cl, pv[k]);
      }
    }
  };
  double rp[kRB], psq = 0.0;
  auto fold_psq = [&](int64_t r0) {   // of the kTR rows before r0
    if constexpr (PSQ) {
      psq = grp_sum_d(psq, 64);
      if (wl == 0) s_psq[4 * ((r0 - q.r_lo - 1) / kTR)] = psq;
      psq = 0.0;
    }
  };
  auto consume = [&]() {
#pragma unroll
    for (int k = 0; k < kRB; ++k) {
      if constexpr (CUT) {
        win_fix(w, cut, g[k]);
        if constexpr (PSQ) win_fix(w, cut, pv[k]);
      }
      const bool ok = rv[k] && act;
      double rk = 0.0;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        // the float square g*g is the reference's term (g32.square(), optimizer.py:2213)
        const float gg = ok ? scrub(g[k][e]) : 0.0f;
        const double sq = (double)(gg * gg);
        acc[e] += sq;
        rk += sq;
        if constexpr (PSQ) {
          const double pd = ok ? (double)pv[k][e] : 0.0;
          psq = __builtin_fma(pd, pd, psq);
        }
      }
      rp[k] = rk;
    }
  };
  auto reduce = [&](int64_t r0) {
    const double tot = reduce_scatter4(rp, wl);
    if ((wl & 15) == 0) s_row[(r0 - q.r_lo) + row_of_lane(wl)] = tot;
  };
  // Each batch's row-sum reduction runs while the next batch's loads are in
  // flight (issued just before it).
  issue(q.r_lo);
  __builtin_amdgcn_sched_barrier(0);
  consume();
  int64_t r0 = q.r_lo + kRB;
  for (; r0 < q.r_hi; r0 += kRB) {
    __builtin_amdgcn_sched_barrier(0);
    issue(r0);
    __builtin_amdgcn_sched_barrier(0);
    reduce(r0 - kRB);
    if ((r0 - q.r_lo) % kTR == 0) {
      col_fold(acc, tot);
      fold_psq(r0);
    }
    __builtin_amdgcn_sched_barrier(0);
    consume();
  }
  reduce(r0 - kRB);
  fold_psq(r0);
}

// Row sums and column sums of g^2 (and sum p^2) as per-tile partials, accumulated
// in double (optimizer.py:2211-2219).
template <typename T, bool PSQ>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 8 ? (PSQ ? 4 : 6) : (PSQ ? 5 : 7))))
void k_fstats(const DescF* __restrict__ table, int ntab) {
  __shared__ double s_row[4 * kTRS];
  __shared__ double s_psq[4 * (kTRS / kTR)];   // [kTR rows][wave]
  const DescF D = *find_tile(table, ntab, (int64_t)blockIdx.x);
  const FWs W = fws_layout(D.B, D.R, D.C, D.tr);
  const TilePos q = tile_pos<false>(D, W);
  const int lane = threadIdx.x, wl = lane & 63;
  const int wave = __builtin_amdgcn_readfirstlane(lane >> 6);
  const int64_t C = D.C;
  const int64_t cw = q.c_base + 256 * wave, c0 = cw + 4 * wl;   // the wave's first column, the lane's
  __shared__ double s_tot[4 * 256];
  double* tot = s_tot + lane;
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  if (q.r_hi - q.r_lo > kTR) {
#pragma unroll
    for (int e = 0; e < 4; ++e) tot[256 * e] = 0.0;
  }
  double* srow = s_row + kTRS * wave;
  if (cw >= C) {   // the wave's columns lie beyond C
    for (int i = wl; i < kTRS; i += 64) srow[i] = 0.0;
    if (PSQ && wl < kTRS / kTR) s_psq[4 * wl + wave] = 0.0;
  }
  else if (D.elem) fstats_tile<T, PSQ, false, true>(D, q, c0, acc, tot, s_psq + wave, srow);
  else if ((C & 3) == 0 || cw + 256 <= C) fstats_tile<T, PSQ, false, false>(D, q, c0, acc, tot, s_psq + wave, srow);
  else fstats_tile<T, PSQ, true, false>(D, q, c0, acc, tot, s_psq + wave, srow);
  float* ws = D.ws;
  double* colp = ws_dp(ws, W.colpart) + (q.b * W.nstrip + q.s) * C;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (c0 + e < C) gp(colp)[c0 + e] = col_sum(acc, tot, e, q);
  tile_rows_out(s_row, ws_dp(ws, W.rowpart) + q.ch * (D.B * D.R) + q.b * D.R, q.r_lo, q.r_hi);   // (a barrier first)
  if (PSQ && lane == 0) {
    double p = 0.0;
    for (int k = 0; k < (q.r_hi - q.r_lo + kTR - 1) / kTR; ++k)
      p += ((s_psq[4 * k] + s_psq[4 * k + 1]) + s_psq[4 * k + 2]) + s_psq[4 * k + 3];
    gp(ws_dp(ws, W.p2))[q.t] = p;
  }
}

// ------------------------------------------------------------ CAME residual statistics
// Old momentum of the element at flat index e (codec mk: 1 UF8, 2 UF4, 3 D8,
// 4 D4; UF4/D4 keep the even element in the high nibble).
// M block of flat index e: a shift for the power-of-two sizes (lbm >= 0), else a
// division by B_M.
__device__ __forceinline__ int64_t m_blk(int64_t e, int lbm, int bm) { return lbm >= 0 ? e >> lbm : e / bm; }

__device__ __forceinline__ float m_old_at(int mk, const uint8_t* mq, const float* msc, int64_t e, int lbm, int bm) {
  const float ms = gp(msc)[m_blk(e, lbm, bm)];
  uint32_t q;
  if (mk == 2 || mk == 4) {
    const uint32_t byte = gp(mq)[e >> 1];
    q = (e & 1) ? (byte & 0x0Fu) : (byte >> 4);
  } else {
    q = gp(mq)[e];
  }
  return m_decode(mk, q, ms);
}

// Old momentum of four consecutive elements e .. e+3 of one row (zero beyond `avail`).
template <int MK>
__device__ __forceinline__ void m_old4(int mkr, const uint8_t* mq, const float* msc, int64_t e, int64_t avail,
                                       int lbm, int bm, float* out) {
  const int mk = MK == 1 ? 1 : mkr;
#pragma unroll
  for (int k = 0; k < 4; ++k) out[k] = (k < avail) ? m_old_at(mk, mq, msc, e + k, lbm, bm) : 0.0f;
}

// CAME pass 1 over the statistics tiles of one workgroup (layout of fstats_tile):
// U = ((g * inv_row) * inv_col) / clip, M' = lerp(M, U, 1 - beta1),
// res = (U - M')^2 + eps_came, row and column sums of res (optimizer.py:929-937).
// RAGGED: C is no multiple of 4, so rows start anywhere and a window's codes may straddle
// two M blocks.  TINY: DescF::elem.
template <typename T, int MK, bool RAGGED, bool TINY>
__device__ __forceinline__ void came1_tile(const DescF& D, const FWs& W, const TilePos& q, const HyperF& h,
                                           int64_t c0, const float* icol, float clip, double* acc, double* tot,
                                           double* s_row) {
  const T* G = reinterpret_cast<const T*>(D.grad);
  const int64_t R = D.R, C = D.C;
  const int wl = threadIdx.x & 63;
  const Win w = win_at(c0, C, 0);
  const uint32_t cl = w.cl;
  const bool act = w.n > 0;
  const int cut = (int)(C & 3);
  const float* ws = D.ws;
  const int mk = MK == 1 ? 1 : h.mk;
  const bool nib = (mk == 2 || mk == 4);
  const LerpW lw = lerp_weight(h.w_m);
  const float rclip = 1.0f / clip;
  float g[kRB][4], mo[kRB][4], ir[kRB];
  uint32_t qv[kRB];
  float ms[kRB], ms3[RAGGED ? kRB : 1];
  int nf[RAGGED ? kRB : 1];   // elements of the window in its first M block
  bool rv[kRB];
  auto issue = [&](int64_t r0) {
#pragma unroll
    for (int k = 0; k < kRB; ++k) {
      const int64_t r = r0 + k;
      rv[k] = r < q.r_hi;
      const int64_t rr = rv[k] ? r : q.r_lo;
      const int64_t rowbase = (q.b * R + rr) * C;
      ir[k] = cp(ws)[W.invr + q.b * R + rr];
      if constexpr (TINY) {
        load_tiny<T>(G + rowbase, c0, C, g[k]);
        if constexpr (MK == 3) load_tiny<float>(D.m + rowbase, c0, C, mo[k]);
        else m_old4<MK>(h.mk, D.m_q, D.m_scale, rowbase + c0, C - c0, h.lbm, h.bm, mo[k]);
      } else {
        load4o<T>(G + rowbase, cl, g[k]);
        if constexpr (MK == 3) {
          load4o<float>(D.m + rowbase, cl, mo[k]);
        } else if constexpr (RAGGED) {
          // codes of elements e .. e + 3 from any e, and the scales of the first's and
          // the last's M block
          const int64_t e = rowbase + cl;
          const int64_t b0 = m_blk(e, h.lbm, h.bm), b3 = m_blk(e + 3, h.lbm, h.bm);
          ms[k] = gp(D.m_scale)[b0];
          ms3[k] = gp(D.m_scale)[b3];
          nf[k] = b3 == b0 ? 4 : (int)(b3 * (h.lbm >= 0 ? (int64_t)1 << h.lbm : (int64_t)h.bm) - e);
          if (MK == 1 || !nib) {
            qv[k] = *((const A8_G u32_e*)(D.m_q + e));
          } else {   // five nibbles from byte e / 2 on, read inside the codes
            const uint32_t lo16 = gp(D.m_q)[e >> 1] | ((uint32_t)gp(D.m_q)[(e >> 1) + 1] << 8);
            const uint32_t w24 = lo16 | ((uint32_t)gp(D.m_q)[(e + 3) >> 1] << 16);
            // nibbles in element order (the even element of a byte is its high nibble)
            const uint32_t sw = ((w24 & 0x0F0F0Fu) << 4) | ((w24 >> 4) & 0x0F0F0Fu);
            qv[k] = (e & 1) ? sw >> 4 : sw;
          }
        } else {
          const int64_t e = rowbase + cl;
          ms[k] = gp(D.m_scale)[m_blk(e, h.lbm, h.bm)];
          if (MK == 1 || !nib) qv[k] = __builtin_nontemporal_load(gp(reinterpret_cast<const uint32_t*>(D.m_q + e)));
          else qv[k] = __builtin_nontemporal_load(gp(reinterpret_cast<const uint16_t*>(D.m_q + (e >> 1))));
        }
      }
    }
  };
  double rp[kRB];
  auto consume = [&]() {
    float mk4[kRB][4];
#pragma unroll
    for (int k = 0; k < kRB; ++k) {
      if constexpr (RAGGED && !TINY && MK != 3) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          mk4[k][e] = m_decode(mk, nib ? (qv[k] >> (4 * e)) & 0xFu : (qv[k] >> (8 * e)) & 0xFFu, e < nf[k] ? ms[k] : ms3[k]);
      } else if constexpr (!TINY && MK != 3) {
        if (MK == 1 || !nib) {
#pragma unroll
          for (int e = 0; e < 4; ++e) mk4[k][e] = m_decode(mk, (qv[k] >> (8 * e)) & 0xFFu, ms[k]);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const uint32_t byte = (qv[k] >> (8 * (e >> 1))) & 0xFFu;
            mk4[k][e] = m_decode(mk, (e & 1) ? (byte & 0x0Fu) : (byte >> 4), ms[k]);
          }
        }
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) mk4[k][e] = mo[k][e];
      }
    }
#pragma unroll
    for (int k = 0; k < kRB; ++k) {
      if constexpr (RAGGED && !TINY) {
        win_fix(w, cut, g[k]);
        win_fix(w, cut, mk4[k]);
      }
      float xs[4], ug[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) xs[e] = (scrub(g[k][e]) * ir[k]) * icol[e];
      div_by<4>(ug, xs, clip, rclip);
      double rk = 0.0;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const bool ok = rv[k] && (RAGGED ? e < w.n : act);
        const float mn = lerp_u(mk4[k][e], ug[e], lw);
        const float dd = ug[e] - mn;
        const double res = ok ? (double)(dd * dd + h.eps_came) : 0.0;
        acc[e] += res;
        rk += res;
      }
      rp[k] = rk;
    }
  };
  auto reduce = [&](int64_t r0) {
    const double tot = reduce_scatter4(rp, wl);
    if ((wl & 15) == 0) s_row[(r0 - q.r_lo) + row_of_lane(wl)] = tot;
  };
  // next batch's loads in flight during the row-sum reduction, as in fstats_tile
  issue(q.r_lo);
  __builtin_amdgcn_sched_barrier(0);
  consume();
  int64_t r0 = q.r_lo + kRB;
  for (; r0 < q.r_hi; r0 += kRB) {
    __builtin_amdgcn_sched_barrier(0);
    issue(r0);
    __builtin_amdgcn_sched_barrier(0);
    reduce(r0 - kRB);
    if ((r0 - q.r_lo) % kTR == 0) col_fold(acc, tot);
    __builtin_amdgcn_sched_barrier(0);
    consume();
  }
  reduce(r0 - kRB);
}

// CAME pass 1: the residual's row and column sums as per-tile partials in the
// g^2 partial arrays (consumed by then).
template <typename T, int MK>
__global__ __launch_bounds__(256) void k_came1(const DescF* __restrict__ table, int ntab, HyperF h) {
  __shared__ double s_row[4 * kTRS];
  const DescF D = *find_tile(table, ntab, (int64_t)blockIdx.x);
  const FWs W = fws_layout(D.B, D.R, D.C, D.tr);
  const TilePos q = tile_pos<false>(D, W);
  const int lane = threadIdx.x, wl = lane & 63;
  const int wave = __builtin_amdgcn_readfirstlane(lane >> 6);
  const int64_t C = D.C;
  const int64_t c0 = q.c_base + 256 * wave + 4 * wl;
  float* ws = D.ws;
  const float clip = cp(ws)[W.scal + 4];
  float icol[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) icol[e] = (c0 + e < C) ? gp(ws)[W.invc + q.b * C + c0 + e] : 0.0f;
  __shared__ double s_tot[4 * 256];
  double* tot = s_tot + lane;
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  if (q.r_hi - q.r_lo > kTR) {
#pragma unroll
    for (int e = 0; e < 4; ++e) tot[256 * e] = 0.0;
  }
  double* srow = s_row + kTRS * wave;
  if (q.c_base + 256 * wave >= C) {   // the wave's columns lie beyond C
    for (int i = wl; i < kTRS; i += 64) srow[i] = 0.0;
  }
  else if (D.elem) came1_tile<T, MK, true, true>(D, W, q, h, c0, icol, clip, acc, tot, srow);
  else if ((C & 3) == 0) came1_tile<T, MK, false, false>(D, W, q, h, c0, icol, clip, acc, tot, srow);
  else came1_tile<T, MK, true, false>(D, W, q, h, c0, icol, clip, acc, tot, srow);
  double* colp = ws_dp(ws, W.colpart) + (q.b * W.nstrip + q.s) * C;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (c0 + e < C) gp(colp)[c0 + e] = col_sum(acc, tot, e, q);
  tile_rows_out(s_row, ws_dp(ws, W.rowpart) + q.ch * (D.B * D.R) + q.b * D.R, q.r_lo, q.r_hi);
}

// ------------------------------------------------------------ row/column V EMA
template <int VB>
__device__ __forceinline__ float fv_decode(const void* q, const float* sc, const float* ml, int64_t i,
                                           int64_t bsz) {
  if constexpr (VB == 8) {
    const uint32_t c = gp(reinterpret_cast<const uint8_t*>(q))[i];
    const int64_t bi = i / bsz;
    return al_decode<254>(c, gp(sc)[bi], gp(ml)[bi], false);
  } else {
    const uint32_t c = gp(reinterpret_cast<const uint16_t*>(q))[i];
    const int64_t bi = i / bsz;
    return al_decode<65534>(c, gp(sc)[bi], gp(ml)[bi], false);
  }
}

__device__ __forceinline__ const DescF* find_cs(const DescF* tab, int n, int64_t wg) {
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (tab[mid].cs_begin <= wg) lo = mid; else hi = mid - 1;
  }
  return tab + lo;
}

// Strip partials src[k C], k0 <= k < k1, in order, those of `fold` strips (8 or 1) first added
// by themselves; eight loads in flight.
__device__ __forceinline__ double strip_sum(const double* src, int64_t C, int64_t k0, int64_t k1, int64_t fold) {
  double sum = 0.0;
  int64_t k = k0;
  for (; k + 8 <= k1; k += 8) {
    double t[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) t[u] = gp(src)[(k + u) * C];
    double s = fold == 1 ? sum : 0.0;
#pragma unroll
    for (int u = 0; u < 8; ++u) s += t[u];
    sum = fold == 1 ? s : sum + s;
  }
  double s = fold == 1 ? sum : 0.0;
  for (; k < k1; ++k) s += gp(src)[k * C];
  return fold == 1 ? s : sum + s;
}
static_assert(kTRS / kTR == 8, "strip_sum");

// First level of the column reduction for tensors of more than gss strips of kTRS rows: one
// workgroup per (batch, 256 columns, group of gss) sums its strips' partials (double) into
// colsum.  k_fblock then adds the nsplit group sums in order.
__global__ __launch_bounds__(256) void k_fcolsum(const DescF* __restrict__ table, int ntab) {
  const DescF D = *find_cs(table, ntab, (int64_t)blockIdx.x);
  const FWs W = fws_layout(D.B, D.R, D.C, D.tr);
  if (W.nsplit <= 1) return;
  const int64_t C = D.C;
  const int64_t ncg = (C + 255) / 256;
  const int64_t w = (int64_t)blockIdx.x - D.cs_begin;
  const int64_t sg = w % W.nsplit;
  const int64_t cg = (w / W.nsplit) % ncg;
  const int64_t b = w / (W.nsplit * ncg);
  const int64_t c = cg * 256 + threadIdx.x;
  if (c >= C) return;
  const int64_t ks = W.gss * W.fold, k0 = sg * ks;
  const int64_t k1 = (k0 + ks < W.nstrip) ? k0 + ks : W.nstrip;
  gp(ws_dp(D.ws, W.colsum))[(b * W.nsplit + sg) * C + c] =
      strip_sum(ws_dp(D.ws, W.colpart) + b * W.nstrip * C + c, C, k0, k1, W.fold);
}

__device__ __forceinline__ const DescF* find_fblk(const DescF* tab, int n, int64_t wg) {
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (tab[mid].fblk_begin <= wg) lo = mid; else hi = mid - 1;
  }
  return tab + lo;
}

// Row/column second moment (CONF = false) or CAME confidence (CONF = true), one
// workgroup per AL block of the flattened row or column vector of a tensor:
// reduce the statistics tiles' partials in a fixed order (double), mean (g^2:
// sum/count + eps1; residual: sum/count), EMA with the decoded state (lerp
// weight 1 - beta2 / step^decay, or 1 - beta3), refit and re-encode the block
// (optimizer.py:2204-2238, 941-948).  The new values go to the workspace vector;
// on the column side they are replaced by inv_col = 1/sqrt(v) (optimizer.py:818-821,
// 951-953).  VB is the state's codec (8 / 16 bits, 0 = fp32 state, blocks of the
// same size only partition the work).
template <int VB, bool CONF>
__global__ __launch_bounds__(1024) void k_fblock(const DescF* __restrict__ table, int ntab, HyperF h) {
  hf_step(h);
  __shared__ float sf[32];
  const int nl = (int)blockDim.x;
  const DescF D = *find_fblk(table, ntab, (int64_t)blockIdx.x);
  const FWs W = fws_layout(D.B, D.R, D.C, D.tr);
  const int64_t lb = (int64_t)blockIdx.x - D.fblk_begin;
  const bool is_row = lb < D.nbr;
  const int64_t bi = is_row ? lb : lb - D.nbr;
  const int lane = threadIdx.x;
  const int64_t B = D.B, R = D.R, C = D.C;
  const int64_t n = is_row ? B * R : B * C;
  float* ws = D.ws;
  float* vec;
  void* q;
  float *sc, *ml, *fst;
  if constexpr (CONF) {
    vec = ws + (is_row ? W.icr : W.icc);
    q = is_row ? D.crow_q : D.ccol_q;
    sc = is_row ? D.crow_scale : D.ccol_scale;
    ml = is_row ? D.crow_min_log : D.ccol_min_log;
    fst = is_row ? D.crow_var : D.ccol_var;
  } else {
    vec = ws + (is_row ? W.invr : W.invc);
    q = is_row ? D.row_q : D.col_q;
    sc = is_row ? D.row_scale : D.col_scale;
    ml = is_row ? D.row_min_log : D.col_min_log;
    fst = is_row ? D.row_var : D.col_var;
  }
  const float cnt = is_row ? (float)C : (float)R;
  const int64_t bsz = h.block_size;
  const float w = CONF ? h.w_c : h.bv;
  const int64_t i0 = bi * bsz;
  const int64_t i1 = (i0 + bsz < n) ? i0 + bsz : n;

  // 1. means and EMA (each lane keeps its own entries for step 2)
  float mx = 0.0f;
  uint32_t key = 0xFFFFFFFFu;
  for (int64_t i = i0 + lane; i < i1; i += nl) {
    double sum = 0.0;
    if (is_row) {
      const double* rp = ws_dp(ws, W.rowpart) + i;
      int64_t k = 0;
      for (; k + 4 <= W.nchunk; k += 4) {   // loads in flight, summed in order
        double t[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) t[u] = gp(rp)[(k + u) * n];
#pragma unroll
        for (int u = 0; u < 4; ++u) sum += t[u];
      }
      for (; k < W.nchunk; ++k) sum += gp(rp)[k * n];
    } else {
      // the column's strip partials, or k_fcolsum's sums
      const int64_t b = i / C, c = i - b * C;
      const bool cs = W.nsplit > 1;
      const int64_t np = cs ? W.nsplit : W.nstrip;
      sum = strip_sum(ws_dp(ws, cs ? W.colsum : W.colpart) + b * np * C + c, C, 0, np, cs ? 1 : W.fold);
    }
    float mean = (float)sum / cnt;
    if constexpr (!CONF) mean = mean + h.eps1;
    float old;
    if constexpr (VB == 0) old = gp(fst)[i];
    else old = fv_decode<VB>(q, sc, ml, i, bsz);
    const float nv = lerp_ref(old, mean, w);
    gp(vec)[i] = nv;
    if constexpr (VB == 0) {
      gp(fst)[i] = nv;
      if (!is_row) gp(vec)[i] = 1.0f / sqrtf(nv);
    }
    mx = fmaxf(mx, nv);
    key = min(key, nz_key_f(nv));
  }

  // 2. refit and re-encode the block (zero padding beyond n -> code 0)
  if constexpr (VB != 0) {
    constexpr int LM2 = VB == 8 ? 254 : 65534;
    wg_maxkey(mx, key, sf);
    const float mnz = (key == 0xFFFFFFFFu) ? __builtin_inff() : __uint_as_float(key + 1u);
    const ALFit f = al_refit(mx, mnz, h.floor_, (float)LM2);
    for (int64_t k = lane; k < bsz; k += nl) {
      const int64_t i = i0 + k;
      const float v = i < n ? gp(vec)[i] : 0.0f;
      uint32_t code;
      al_codes<LM2, 1>(&v, f, &code);
      if constexpr (VB == 8) gp(reinterpret_cast<uint8_t*>(q))[i] = (uint8_t)code;
      else gp(reinterpret_cast<uint16_t*>(q))[i] = (uint16_t)code;
      if (!is_row && i < n) gp(vec)[i] = 1.0f / sqrtf(v);
    }
    if (lane == 0) { gp(sc)[bi] = f.s; gp(ml)[bi] = f.lmin; }
  }
}

// One workgroup per tensor: r = max(mean_r(row), eps1) per batch and
// inv_row = 1/sqrt(row / r) (optimizer.py:2221, 818-821; the confidence's r_c,
// 951-952), then (CONF = false) the step size and weight-decay factor
// (optimizer.py:832-856, 2020-2039).
template <bool CONF>
__global__ __launch_bounds__(256) void k_frows(const DescF* __restrict__ table, HyperF h) {
  hf_step(h);
  __shared__ double sd[4];
  const DescF D = table[blockIdx.x];
  const FWs W = fws_layout(D.B, D.R, D.C, D.tr);
  const int lane = threadIdx.x;
  const int64_t B = D.B, R = D.R;
  float* ws = D.ws;
  float* vec = ws + (CONF ? W.icr : W.invr);
  for (int64_t b = 0; b < B; ++b) {
    float* v = vec + b * R;
    double s = 0.0;
    int64_t r = lane;
    for (; r + 7 * 256 < R; r += 8 * 256) {   // eight loads in flight, summed in order
      float t[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) t[u] = gp(v)[r + 256 * u];
#pragma unroll
      for (int u = 0; u < 8; ++u) s += (double)t[u];
    }
    for (; r < R; r += 256) s += (double)gp(v)[r];
    s = wg_sum_d(s, sd);
    const float rmv = fmaxf((float)s / (float)R, h.eps1);
    r = lane;
    for (; r + 3 * 256 < R; r += 4 * 256) {
      float t[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) t[u] = gp(v)[r + 256 * u];
#pragma unroll
      for (int u = 0; u < 4; ++u) gp(v)[r + 256 * u] = 1.0f / sqrtf(t[u] / rmv);
    }
    for (; r < R; r += 256) gp(v)[r] = 1.0f / sqrtf(gp(v)[r] / rmv);
  }
  if constexpr (!CONF) {
    const float rho = D.lr ? *gp(D.lr) : h.lr_val;
    float alpha = rho;
    if (h.scale_param) {
      double s = 0.0;
      // tiles of kTRS rows, or the short ones of the same rows first (index (b, strip, chunk)),
      // their loads in flight
      const double* p2 = ws_dp(ws, W.p2);
      const uint32_t nch = (uint32_t)W.nchunk, nss = (uint32_t)W.nss, fold = (uint32_t)W.fold;
      for (uint32_t k = lane; fold == 1 && k < (uint32_t)B * nss * nch; k += 256) s += gp(p2)[k];
      for (uint32_t k = lane; fold != 1 && k < (uint32_t)B * nss * nch; k += 256) {
        const uint32_t bs = k / nch, ch = k - bs * nch, b = bs / nss, s0 = (bs - b * nss) * fold;
        const int64_t left = W.nstrip - s0, at = (b * W.nstrip + s0) * W.nchunk + ch;
        double t[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) t[j] = j < left ? gp(p2)[at + j * W.nchunk] : 0.0;
        double f = 0.0;
#pragma unroll
        for (int j = 0; j < 8; ++j) f += t[j];
        s += f;
      }
      s = wg_sum_d(s, sd);
      const float nrm = sqrtf((float)s);
      const float rms = nrm / (float)sqrt((double)D.numel);
      alpha = fmaxf(rms, h.eps2) * rho;
    }
    if (h.bias_mode == 1) alpha = alpha * h.bias_factor;
    else if (h.bias_mode == 2) alpha = alpha / h.bias_factor;
    if (lane == 0) {
      float* sl = ws + W.scal;
      gp(sl)[0] = alpha;
      gp(sl)[1] = alpha;
      gp(sl)[2] = 1.0f;
      float dec = 1.0f;
      if (h.wd_mode == 1) dec = 1.0f - alpha * h.wd;
      else if (h.wd_mode == 2) dec = 1.0f - rho * h.wd;
      gp(sl)[3] = dec;
      gp(sl)[4] = 1.0f;   // CAME clip factor unless k_fclip sets it
    }
  }
}

// ------------------------------------------------------------ update
// MODE 0: write with step = alpha; 1: sum(u^2) per unit; 2: write with the
// step and Fira scale of k_fnorm.  MK: 0 no momentum, 1 UF8, 2 other codecs, 3 fp32 momentum.
// CM (CAME): the momentum EMA runs on U = ((g * inv_row) * inv_col) / clip and
// the update is (M' * inv_conf_row) * inv_conf_col (optimizer.py:929-956).
template <typename T, int MODE, bool SR, int MK, bool CM>
__global__ __launch_bounds__(256) void k_fupdate(const DescF* __restrict__ table, int ntab, HyperF h) {
  if constexpr (SR) hf_step(h);
  static_assert(!CM || MK != 0, "CAME needs momentum");
  __shared__ float s4[8];
  __shared__ double s4d[4];
  constexpr bool kHasM = MK != 0;
  const DescF D = *find_unit(table, ntab, (int64_t)blockIdx.x);
  if (D.tiled) return;   // updated by k_fupdt
  const FWs W = fws_layout(D.B, D.R, D.C, D.tr);
  const int64_t wl = (int64_t)blockIdx.x - D.unit_begin;
  const int lane = threadIdx.x;
  const int64_t n = D.numel;
  const int64_t e0 = wl * kUnit + (int64_t)lane * 8;
  const int64_t rem = n - e0;
  const int cnt = rem <= 0 ? 0 : (rem >= 8 ? 8 : (int)rem);
  const int64_t R = D.R, C = D.C;
  const float* ws = D.ws;
  const float* invr = ws + W.invr;
  const float* invc = ws + W.invc;
  const float* icr = ws + W.icr;
  const float* icc = ws + W.icc;
  const float* sl = ws + W.scal;
  const int lbm = h.lbm;
  const int BM = 1 << lbm;
  const int ML = BM >> 3;
  const int64_t mb = e0 >> lbm;
  const int mk = (MK == 1) ? 1 : h.mk;

  float g[8], mn[8], u[8], mo[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) { g[k] = 0.0f; mn[k] = 0.0f; u[k] = 0.0f; mo[k] = 0.0f; }
  double sq = 0.0;   // sum u^2 (MODE 1), accumulated in double
  uint32_t amaxb = 0u;
  if (cnt > 0) {
    load8<T>(reinterpret_cast<const T*>(D.grad), e0, n, g);
#pragma unroll
    for (int k = 0; k < 8; ++k) g[k] = scrub(g[k]);
    if constexpr (MK == 3) {
      load8<float>(D.m, e0, n, mo);
    } else if constexpr (kHasM) {
      const float ms = gp(D.m_scale)[mb];
      if (MK == 1) {
        const u32x2 qv = *gp(reinterpret_cast<const u32x2*>(D.m_q + e0));
        const float s128 = ms / 128.0f, b128 = -128.0f * s128;
#pragma unroll
        for (int k = 0; k < 8; ++k)
          mo[k] = __builtin_fmaf((float)(((k < 4 ? qv.x : qv.y) >> (8 * (k & 3))) & 0xFFu), s128, b128);
      } else if (mk == 2 || mk == 4) {
        const uint32_t qw = *gp(reinterpret_cast<const uint32_t*>(D.m_q + (e0 >> 1)));
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const uint32_t byte = (qw >> (8 * (k >> 1))) & 0xFFu;
          mo[k] = m_decode(mk, (k & 1) ? (byte & 0x0Fu) : (byte >> 4), ms);
        }
      } else {
        const u32x2 qv = *gp(reinterpret_cast<const u32x2*>(D.m_q + e0));
#pragma unroll
        for (int k = 0; k < 8; ++k) mo[k] = m_decode(mk, ((k < 4 ? qv.x : qv.y) >> (8 * (k & 3))) & 0xFFu, ms);
      }
    }
    if constexpr (kHasM && !CM) {
#pragma unroll
      for (int k = 0; k < 8; ++k) mn[k] = (k < cnt) ? lerp_ref(mo[k], g[k], h.w_m) : 0.0f;
    }
    const float clip = CM ? gp(sl)[4] : 1.0f;
    // element (row, column): row = e / C, column index b*C + c with b = row / R
    int64_t row = e0 / C;
    int64_t c = e0 - row * C;
    int64_t b = row / R;
    int64_t rr = row - b * R;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      if (k < cnt) {
        if constexpr (CM) {
          const float ug = ((g[k] * gp(invr)[row]) * gp(invc)[b * C + c]) / clip;
          mn[k] = lerp_ref(mo[k], ug, h.w_m);
          u[k] = (mn[k] * gp(icr)[row]) * gp(icc)[b * C + c];
        } else {
          const float x = kHasM ? mn[k] : g[k];
          u[k] = (x * gp(invr)[row]) * gp(invc)[b * C + c];
        }
        if (MODE == 1) sq = __builtin_fma((double)u[k], (double)u[k], sq);
      }
      if (++c == C) {
        c = 0;
        ++row;
        if (++rr == R) { rr = 0; ++b; }
      }
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) amaxb = max(amaxb, __float_as_uint(mn[k]) & 0x7FFFFFFFu);

    if constexpr (MODE != 1) {
      const float step = (MODE == 0) ? gp(sl)[0] : gp(sl)[1];
      const float fs = (MODE == 2) ? gp(sl)[2] : 1.0f;
      const float dec = gp(sl)[3];
      const bool has_dec = h.wd_mode != 0;
      if (MODE == 2) {
#pragma unroll
        for (int k = 0; k < 8; ++k) u[k] = u[k] * fs;
      }
      T* P = reinterpret_cast<T*>(D.param);
      if constexpr (SR) {
        float p[8];
        load8<T>(P, e0, n, p);
#pragma unroll
        for (int k = 0; k < 8; ++k) p[k] = (has_dec ? p[k] * dec : p[k]) - step * u[k];
        const uint64_t z = sr_base(D.sr_seed, h.sr_step) + 0x9E3779B97F4A7C15ULL + (uint64_t)(wl * kUnit);
        const SrUnit srs = sr_unit<kUnit>(z);
        T* Pu = P + wl * kUnit;
        const uint32_t i0 = (uint32_t)lane * 8u, in = (uint32_t)(n - wl * kUnit < kUnit ? n - wl * kUnit : kUnit);
        sr_store4<T>(Pu, i0, in, p, z + i0, srs);
        if (i0 + 4 < in) sr_store4<T>(Pu, i0 + 4, in, p + 4, z + i0 + 4, srs);
      } else {
        pval_t<T> p[8];
        load8<T>(P, e0, n, p);
        if (has_dec) {
#pragma unroll
          for (int k = 0; k < 8; ++k) p[k] = pdec(p[k], dec);
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) p[k] = pupd(step, u[k], p[k]);
        store8<T>(P, e0, n, p);
      }
    }
  }

  if constexpr (MODE == 1) {
    const double tot = wg_sum_d(sq, s4d);
    if (lane == 0) gp(ws_dp(const_cast<float*>(ws), W.npart))[wl] = tot;
  }

  if constexpr (MODE != 1 && MK == 3) {
    if (cnt > 0) store8<float>(D.m, e0, n, mn);
  }
  // momentum re-encode: absmax over B_M elements = ML lanes
  if constexpr (MODE != 1 && kHasM && MK != 3) {
    const int wave = lane >> 6;
    float bam = grp_max(__uint_as_float(amaxb), ML < 64 ? ML : 64);
    if (ML > 64) {
      __syncthreads();
      if ((lane & 63) == 0) s4[wave] = bam;
      __syncthreads();
      const int w0 = (lane >> (lbm - 3)) * (ML >> 6);
      bam = s4[w0];
      for (int w = 1; w < (ML >> 6); ++w) bam = fmaxf(bam, s4[w0 + w]);
    }
    if (cnt > 0) {
      const float am = fmaxf(bam, 1e-12f);
      const float ram = fast_rcp(am);
      if (MK == 1) {
        const float kam = 128.0f * ram;
        float r[8];
        bool bad[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) r[k] = uf_round_fast<128>(mn[k], kam, bad[k]);
#pragma unroll
        for (int k = 0; k < 8; ++k)
          if (bad[k]) r[k] = uf_round_exact<128>(mn[k], am);
#pragma unroll
        for (int k = 0; k < 8; ++k) r[k] = uf_clamp<128>(r[k]);
        *gp(reinterpret_cast<u32x2*>(D.m_q + e0)) = u32x2{pack4(r[0], r[1], r[2], r[3]), pack4(r[4], r[5], r[6], r[7])};
      } else if (mk == 2 || mk == 4) {
        uint32_t w = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const uint32_t hi = m_encode(mk, mn[2 * j], am, ram);
          const uint32_t lo = m_encode(mk, mn[2 * j + 1], am, ram);
          w |= ((hi << 4) | lo) << (8 * j);
        }
        *gp(reinterpret_cast<uint32_t*>(D.m_q + (e0 >> 1))) = w;
      } else {
        uint32_t w0 = 0, w1 = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) w0 |= m_encode(mk, mn[k], am, ram) << (8 * k);
#pragma unroll
        for (int k = 0; k < 4; ++k) w1 |= m_encode(mk, mn[k + 4], am, ram) << (8 * k);
        *gp(reinterpret_cast<u32x2*>(D.m_q + e0)) = u32x2{w0, w1};
      }
      if ((lane & (ML - 1)) == 0) gp(D.m_scale)[mb] = am;
    }
  }
}

// k_fupdate for coded momentum whose block size the unit layout cannot take
// (B_M a multiple of 4 in [32, 2^30], not a power of two up to 2048).  One
// workgroup covers h.unit = B_M * ceil(2048 / B_M) elements, a whole number of M
// blocks and at least kUnit, so a tensor takes no more workgroups than its
// W.nunit norm-partial slots; its last workgroup zeroes the slots it does not
// use.  Lanes take quads (a quad never straddles an M block, B_M % 4 == 0); each
// block's absmax meets in LDS (an exact max).  Pass 1 forms M' and u and writes
// the parameter (MODE 1: the partial sum of u^2); pass 2, after the absmaxes,
// forms M' again from the same inputs and writes the codes; the scales follow
// once every lane has read the old ones.  Element for element the arithmetic is
// k_fupdate's.  MK: 0 no momentum (the CAME clip pass), 2 any codec (h.mk).
constexpr int kFGenMaxMB = 64;

template <typename T, int MODE, bool SR, int MK, bool CM>
__global__ __launch_bounds__(256) void k_fupdate_gen(const DescF* __restrict__ table, int ntab, HyperF h) {
  if constexpr (SR) hf_step(h);
  static_assert(MK == 0 || MK == 2, "codes through m_decode / m_encode");
  static_assert(!CM || MK != 0, "CAME needs momentum");
  __shared__ uint32_t s_mab[kFGenMaxMB];
  __shared__ double s4d[4];
  const DescF D = *find_unit(table, ntab, (int64_t)blockIdx.x);
  if (D.tiled) return;
  const FWs W = fws_layout(D.B, D.R, D.C, D.tr);
  const int lane = threadIdx.x;
  const int BM = h.bm, U = h.unit, mpu = U / BM;
  const int64_t wl = (int64_t)blockIdx.x - D.unit_begin;
  const int64_t n = D.numel;
  const int64_t base = wl * U;
  const int64_t mb0 = base / BM, nmb = (n + BM - 1) / BM;
  const int64_t R = D.R, C = D.C;
  float* ws = D.ws;
  const float* invr = ws + W.invr;
  const float* invc = ws + W.invc;
  const float* icr = ws + W.icr;
  const float* icc = ws + W.icc;
  const float* sl = ws + W.scal;
  const T* G = reinterpret_cast<const T*>(D.grad);
  T* P = reinterpret_cast<T*>(D.param);
  const int mk = h.mk;
  const bool nib = mk == 2 || mk == 4;
  const float clip = CM ? gp(sl)[4] : 1.0f;
  if constexpr (MK != 0 && MODE != 1) {
    for (int i = lane; i < mpu; i += 256) s_mab[i] = 0u;
    __syncthreads();
  }

  // M' and u of the quad at unit offset 4q (zero past the tensor)
  auto quad = [&](int q, float* g, float* mn, float* u, int& cnt, int& mb, bool& m_ok) {
    const int64_t i0 = base + 4 * q;
    cnt = i0 >= n ? 0 : (n - i0 >= 4 ? 4 : (int)(n - i0));
    load4n<T>(G, i0, n, g);
#pragma unroll
    for (int k = 0; k < 4; ++k) g[k] = scrub(g[k]);
    mb = (4 * q) / BM;
    m_ok = MK != 0 && mb0 + mb < nmb;   // codes are padded to whole blocks
    float mo[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (m_ok) {
      const float ms = gp(D.m_scale)[mb0 + mb];
      if (nib) {
        const uint32_t w = *gp(reinterpret_cast<const uint16_t*>(D.m_q + (i0 >> 1)));
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const uint32_t byte = (w >> (8 * (k >> 1))) & 0xFFu;
          mo[k] = m_decode(mk, (k & 1) ? (byte & 0x0Fu) : (byte >> 4), ms);
        }
      } else {
        const uint32_t w = *gp(reinterpret_cast<const uint32_t*>(D.m_q + i0));
#pragma unroll
        for (int k = 0; k < 4; ++k) mo[k] = m_decode(mk, (w >> (8 * k)) & 0xFFu, ms);
      }
    }
    int64_t row = i0 / C;
    int64_t c = i0 - row * C;
    int64_t b = row / R;
    int64_t rr = row - b * R;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      mn[k] = 0.0f;
      u[k] = 0.0f;
      if (k < cnt) {
        if constexpr (CM) {
          const float ug = ((g[k] * gp(invr)[row]) * gp(invc)[b * C + c]) / clip;
          mn[k] = lerp_ref(mo[k], ug, h.w_m);
          u[k] = (mn[k] * gp(icr)[row]) * gp(icc)[b * C + c];
        } else {
          if constexpr (MK != 0) mn[k] = lerp_ref(mo[k], g[k], h.w_m);
          const float x = MK != 0 ? mn[k] : g[k];
          u[k] = (x * gp(invr)[row]) * gp(invc)[b * C + c];
        }
      }
      if (++c == C) {
        c = 0;
        ++row;
        if (++rr == R) { rr = 0; ++b; }
      }
    }
  };

  float step = 0.0f, fs = 1.0f, dec = 1.0f;
  if constexpr (MODE != 1) {
    step = (MODE == 0) ? gp(sl)[0] : gp(sl)[1];
    fs = (MODE == 2) ? gp(sl)[2] : 1.0f;
    dec = gp(sl)[3];
  }
  const bool has_dec = h.wd_mode != 0;

  // ---- pass 1
  double sq = 0.0;
  for (int q = lane; q < (U >> 2); q += 256) {
    float g[4], mn[4], u[4];
    int cnt, mb;
    bool m_ok;
    quad(q, g, mn, u, cnt, mb, m_ok);
    const int64_t i0 = base + 4 * q;
    if constexpr (MODE == 1) {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (k < cnt) sq = __builtin_fma((double)u[k], (double)u[k], sq);
    } else {
      if (MODE == 2) {
#pragma unroll
        for (int k = 0; k < 4; ++k) u[k] = u[k] * fs;
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if (k >= cnt) continue;
        if constexpr (SR) {
          const float pv = ld1<T>(P, i0 + k);
          const T r = sr_round<T>((has_dec ? pv * dec : pv) - step * u[k], D.sr_seed, h.sr_step,
                                  (uint64_t)(i0 + k));
          uint16_t bits;
          __builtin_memcpy(&bits, &r, 2);
          gp(reinterpret_cast<uint16_t*>(P))[i0 + k] = bits;
        } else {
          const pval_t<T> pv = ld1<T, pval_t<T>>(P, i0 + k);
          st1<T>(P, i0 + k, pupd(step, u[k], has_dec ? pdec(pv, dec) : pv));
        }
      }
      if constexpr (MK != 0) {
        uint32_t ab = 0u;
#pragma unroll
        for (int k = 0; k < 4; ++k) ab = max(ab, __float_as_uint(mn[k]) & 0x7FFFFFFFu);
        if (m_ok) atomicMax(&s_mab[mb], ab);
      }
    }
  }
  if constexpr (MODE == 1) {
    const double tot = wg_sum_d(sq, s4d);
    const int64_t nu = (n + U - 1) / U;
    if (lane == 0) gp(ws_dp(ws, W.npart))[wl] = tot;
    if (wl == nu - 1)
      for (int64_t k = nu + lane; k < W.nunit; k += 256) gp(ws_dp(ws, W.npart))[k] = 0.0;
    return;
  }
  if constexpr (MK != 0) {
    __syncthreads();
    // ---- pass 2: codes
    for (int q = lane; q < (U >> 2); q += 256) {
      float g[4], mn[4], u[4];
      int cnt, mb;
      bool m_ok;
      quad(q, g, mn, u, cnt, mb, m_ok);
      if (!m_ok) continue;
      const int64_t i0 = base + 4 * q;
      const float am = fmaxf(__uint_as_float(s_mab[mb]), 1e-12f);
      const float ram = fast_rcp(am);
      if (nib) {
        const uint32_t w = ((m_encode(mk, mn[0], am, ram) << 4) | m_encode(mk, mn[1], am, ram)) |
                           (((m_encode(mk, mn[2], am, ram) << 4) | m_encode(mk, mn[3], am, ram)) << 8);
        *gp(reinterpret_cast<uint16_t*>(D.m_q + (i0 >> 1))) = (uint16_t)w;
      } else {
        uint32_t w = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) w |= m_encode(mk, mn[k], am, ram) << (8 * k);
        *gp(reinterpret_cast<uint32_t*>(D.m_q + i0)) = w;
      }
    }
    __syncthreads();   // every lane has read the old scales
    for (int i = lane; i < mpu; i += 256)
      if (mb0 + i < nmb) gp(D.m_scale)[mb0 + i] = fmaxf(__uint_as_float(s_mab[i]), 1e-12f);
  }
}

// Tiled form of k_fupdate for tensors whose columns allow it (C >= 4 and, with coded
// momentum, B_M <= 256 dividing C): the statistics tiles (tr rows x 1024
// columns), each wave walking rows, lanes holding 4 consecutive columns of each
// 256-column chunk (1 KB-contiguous accesses).  The tile's inv_col (and CAME
// inv_conf_col) are staged in LDS once, a row's inv_row arrives through a scalar
// load, and an M block is B_M/4 lanes of one chunk of one row.  Same arithmetic
// and operation order as k_fupdate; MODE 1 writes one partial per tile.
// Pins four values in VGPRs at this point, so the arithmetic that forms them (and
// the waits for its loads) stays ahead of a following lane-conditional store
// instead of being sunk into it; a load left unconsumed on the store-skipping path
// would make the next row's loads wait for every outstanding store.
template <typename V>
__device__ __forceinline__ void keep4(const V* v) {
  asm volatile("" ::"v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]));
}

// Stores columns c0 .. c0 + 3 of a row of C (those inside it), from any element alignment.
template <typename T, typename V>
__device__ __forceinline__ void store4e(T* row, uint32_t c0, uint32_t C, const V* v) {
  if (c0 + 4 <= C) {
    if constexpr (sizeof(T) == 8) {
      A8_G f64x2_e* p = ((A8_G f64x2_e*)(reinterpret_cast<double*>(row) + c0));
      __builtin_nontemporal_store(f64x2{(double)v[0], (double)v[1]}, p);
      __builtin_nontemporal_store(f64x2{(double)v[2], (double)v[3]}, p + 1);
    } else if constexpr (sizeof(T) == 4) {
      __builtin_nontemporal_store(f32x4{v[0], v[1], v[2], v[3]}, ((A8_G f32x4_e*)(row + c0)));
    } else {
      u32x2 a;
      T* h = reinterpret_cast<T*>(&a);
#pragma unroll
      for (int k = 0; k < 4; ++k) h[k] = from_f<T>(v[k]);
      __builtin_nontemporal_store(a, ((A8_G u32x2_e*)(row + c0)));
    }
  } else {
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (c0 + k < C) st1<T, V>(row, c0 + k, v[k]);
  }
}

// CUT: tensors whose column count is no multiple of 4 (a kernel of its own: its window
// moves and partial stores would take the plain update from three waves a SIMD to two).
template <typename T, int MODE, bool SR, int MK, bool CM, bool CUT>
__global__ __launch_bounds__(256) void k_fupdt(const DescF* __restrict__ table, int ntab, HyperF h) {
  if constexpr (SR) hf_step(h);
  static_assert(!CM || MK != 0, "CAME needs momentum");
  __shared__ float s_ic[2 * kTC];
  __shared__ double s4d[4];
  constexpr bool kHasM = MK != 0;
  const DescF D = *find_utile(table, ntab, (int64_t)blockIdx.x);
  if (D.tiled != (CUT ? 2 : 1)) return;   // updated by another launch
  static_assert(!CUT || MK == 0 || MK == 3, "coded momentum: whole M blocks per row");
  const FWs W = fws_layout(D.B, D.R, D.C, D.tr);
  const TilePos q = tile_pos<true>(D, W);
  const int64_t R = D.R, C = D.C, b = q.b, c_base = q.c_base;
  const int lane = threadIdx.x, wl = lane & 63;
  const int wave = __builtin_amdgcn_readfirstlane(lane >> 6);
  float* ws = D.ws;
  for (int k = lane; k < kTC; k += 256) {
    const int64_t c = c_base + k;
    s_ic[k] = c < C ? gp(ws)[W.invc + b * C + c] : 0.0f;
    if constexpr (CM) s_ic[kTC + k] = c < C ? gp(ws)[W.icc + b * C + c] : 0.0f;
  }
  __syncthreads();
  const float* sl = ws + W.scal;
  const int lbm = h.lbm;
  const int G = (1 << lbm) >> 2;          // lanes per M block
  const int mk = (MK == 1) ? 1 : h.mk;
  const float clip = CM ? cp(sl)[4] : 1.0f;
  const float rclip = 1.0f / clip;
  const LerpW lw = lerp_weight(h.w_m);
  float step = 0.0f, fs = 1.0f, dec = 1.0f;
  if constexpr (MODE != 1) {
    step = (MODE == 0) ? cp(sl)[0] : cp(sl)[1];
    fs = (MODE == 2) ? cp(sl)[2] : 1.0f;
    dec = cp(sl)[3];
  }
  const bool has_dec = h.wd_mode != 0;
  const uint64_t sr_z = SR ? sr_base(D.sr_seed, h.sr_step) + 0x9E3779B97F4A7C15ULL : 0u;
  const T* G0 = reinterpret_cast<const T*>(D.grad);
  T* P0 = reinterpret_cast<T*>(D.param);
  // A lane's four 4-column windows (Win); one beyond C is pointed at the tile's first
  // window (a valid address), computed on like the others and never stored.  Loads and
  // their arithmetic are unconditional, so nothing is left in flight across rows.
  const int cut = (int)(C & 3);                     // columns of the window that C cuts
  Win win[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int64_t c0 = c_base + 256 * j + 4 * wl;
    if constexpr (CUT) win[j] = win_at(c0, C, c_base);
    else win[j] = Win{c0 < C ? (uint32_t)c0 : (uint32_t)c_base, c0 < C ? 4 : 0};
  }

  // Rows r, r + 4, r + 8 and r + 12 in one pass for the plain update (the loads
  // of all four in flight together: 2.40 -> 2.33 ms at C2 against two rows); one
  // row per pass with momentum (two rows measured slower there: 172 registers), two with
  // stochastic rounding or cut windows (four: 112 registers and scalar spills)
  // and in the read-only norm pass, where registers are better spent on
  // occupancy.  A row beyond the tile reads the first one again and stores nothing.
  constexpr int NRW = (kHasM || MODE == 1) ? 1 : ((SR || CUT) ? 2 : 4);
  double sq = 0.0;   // sum u^2 (MODE 1), accumulated in double
  for (int64_t r0 = q.r_lo + wave; r0 < q.r_hi; r0 += 4 * NRW) {
    int64_t rowb[NRW];
    bool rv[NRW];
    float irw[NRW], icrw[NRW];
    float gj[NRW][4][4], msj[NRW][4];
    pval_t<T> pj[NRW][4][4];   // double for fp64 parameters
    float mfj[NRW][MK == 3 ? 4 : 1][4];
    uint32_t qj[NRW][4];
#pragma unroll
    for (int rr = 0; rr < NRW; ++rr) {
      rv[rr] = r0 + 4 * rr < q.r_hi;
      const int64_t r = rv[rr] ? r0 + 4 * rr : r0;
      rowb[rr] = (b * R + r) * C;
      irw[rr] = cp(ws)[W.invr + b * R + r];
      icrw[rr] = CM ? cp(ws)[W.icr + b * R + r] : 0.0f;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t cl = win[j].cl;
        const int64_t e = rowb[rr] + cl;
        load4o<T>(G0 + rowb[rr], cl, gj[rr][j]);
        if constexpr (MK == 3) {
          load4o<float>(D.m + rowb[rr], cl, mfj[rr][j]);
        } else if constexpr (kHasM) {
          msj[rr][j] = gp(D.m_scale)[e >> lbm];
          if (MK == 1 || !(mk == 2 || mk == 4)) qj[rr][j] = *gp(reinterpret_cast<const uint32_t*>(D.m_q + e));
          else qj[rr][j] = *gp(reinterpret_cast<const uint16_t*>(D.m_q + (e >> 1)));
        }
        if constexpr (MODE != 1) load4o<T>(P0 + rowb[rr], cl, pj[rr][j]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);   // every load of the pass is issued before its arithmetic
#pragma unroll
    for (int rr = 0; rr < NRW; ++rr)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int q0 = 256 * j + 4 * wl;
      const int64_t e = rowb[rr] + win[j].cl;
      const float ir = irw[rr], icrr = icrw[rr];
      const bool st = rv[rr] && win[j].n > 0;   // this window of this row is stored
      if constexpr (CUT) {
        win_fix(win[j], cut, gj[rr][j]);
        if constexpr (MODE != 1) win_fix(win[j], cut, pj[rr][j]);
        if constexpr (MK == 3) win_fix(win[j], cut, mfj[rr][j]);
      }
      float mo[4] = {0.0f, 0.0f, 0.0f, 0.0f};
      float mn[4] = {0.0f, 0.0f, 0.0f, 0.0f}, u[4];
      pval_t<T>* pv = pj[rr][j];
      if constexpr (MK == 3) {
#pragma unroll
        for (int i = 0; i < 4; ++i) mo[i] = mfj[rr][j][i];
      } else if constexpr (kHasM) {
        const float ms = msj[rr][j];
        const uint32_t qv = qj[rr][j];
        if (MK == 1) {
          const float s128 = ms / 128.0f, b128 = -128.0f * s128;
#pragma unroll
          for (int i = 0; i < 4; ++i) mo[i] = __builtin_fmaf((float)((qv >> (8 * i)) & 0xFFu), s128, b128);
        } else if (mk == 2 || mk == 4) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const uint32_t byte = (qv >> (8 * (i >> 1))) & 0xFFu;
            mo[i] = m_decode(mk, (i & 1) ? (byte & 0x0Fu) : (byte >> 4), ms);
          }
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i) mo[i] = m_decode(mk, (qv >> (8 * i)) & 0xFFu, ms);
        }
      }
      float ugj[4];
      if constexpr (CM) {
        float xs[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) xs[i] = (scrub(gj[rr][j][i]) * ir) * s_ic[q0 + i];
        div_by<4>(ugj, xs, clip, rclip);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float gi = scrub(gj[rr][j][i]);
        const float ic = s_ic[q0 + i];
        if constexpr (CM) {
          mn[i] = lerp_u(mo[i], ugj[i], lw);
          u[i] = (mn[i] * icrr) * s_ic[kTC + q0 + i];
        } else {
          float x = gi;
          if constexpr (kHasM) { mn[i] = lerp_u(mo[i], gi, lw); x = mn[i]; }
          u[i] = (x * ir) * ic;
        }
        if (MODE == 1) {
          const double ud = st ? (double)u[i] : 0.0;
          sq = __builtin_fma(ud, ud, sq);
        }
      }
      if constexpr (MODE != 1) {
        if (MODE == 2) {
#pragma unroll
          for (int i = 0; i < 4; ++i) u[i] = u[i] * fs;
        }
        const uint32_t c0 = (uint32_t)(c_base + q0), cn = (uint32_t)C;
        if constexpr (SR) {
          float x[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) x[i] = (has_dec ? pv[i] * dec : pv[i]) - step * u[i];
          keep4(x);
          // the SR counters of the row's part of the tile, and what they share
          const uint64_t z = sr_z + (uint64_t)rowb[rr];
          const SrUnit srs = sr_unit<kTC>(z + (uint64_t)c_base);
          if (st) sr_store4<T>(P0 + rowb[rr], c0, cn, x, z + c0, srs);
        } else {
          if (has_dec) {
#pragma unroll
            for (int i = 0; i < 4; ++i) pv[i] = pdec(pv[i], dec);
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) pv[i] = pupd(step, u[i], pv[i]);
          keep4(pv);
          if constexpr (CUT) { if (st) store4e<T>(P0 + rowb[rr], c0, cn, pv); }
          else if (st) store4n<T>(P0, e, e + 4, pv);
        }
        if constexpr (MK == 3) {
          keep4(mn);
          if constexpr (CUT) { if (st) store4e<float>(D.m + rowb[rr], c0, cn, mn); }
          else if (st) store4n<float>(D.m, e, e + 4, mn);
        } else if constexpr (kHasM) {
          // momentum re-encode: absmax over the block's G lanes.  C is a multiple
          // of the M block, so a block is wholly inside or wholly beyond C.
          uint32_t ab = 0u;
#pragma unroll
          for (int i = 0; i < 4; ++i) ab = max(ab, st ? (__float_as_uint(mn[i]) & 0x7FFFFFFFu) : 0u);
          const float bam = grp_max_dpp(__uint_as_float(ab), G);
          if (st) {
            const float am = fmaxf(bam, 1e-12f);
            const float ram = fast_rcp(am);
            if (MK == 1) {
              const float kam = 128.0f * ram;
              float rr[4];
              bool bad[4];
#pragma unroll
              for (int i = 0; i < 4; ++i) rr[i] = uf_round_fast<128>(mn[i], kam, bad[i]);
#pragma unroll
              for (int i = 0; i < 4; ++i)
                if (bad[i]) rr[i] = uf_round_exact<128>(mn[i], am);
#pragma unroll
              for (int i = 0; i < 4; ++i) rr[i] = uf_clamp<128>(rr[i]);
              *gp(reinterpret_cast<uint32_t*>(D.m_q + e)) = pack4(rr[0], rr[1], rr[2], rr[3]);
            } else if (mk == 2 || mk == 4) {
              uint32_t w = 0;
#pragma unroll
              for (int k = 0; k < 2; ++k) {
                const uint32_t hi = m_encode(mk, mn[2 * k], am, ram);
                const uint32_t lo = m_encode(mk, mn[2 * k + 1], am, ram);
                w |= ((hi << 4) | lo) << (8 * k);
              }
              *gp(reinterpret_cast<uint16_t*>(D.m_q + (e >> 1))) = (uint16_t)w;
            } else {
              uint32_t w = 0;
#pragma unroll
              for (int i = 0; i < 4; ++i) w |= m_encode(mk, mn[i], am, ram) << (8 * i);
              *gp(reinterpret_cast<uint32_t*>(D.m_q + e)) = w;
            }
            if ((wl & (G - 1)) == 0) gp(D.m_scale)[e >> lbm] = am;
          }
        }
      }
    }
  }
  if constexpr (MODE == 1) {
    const double tot = wg_sum_d(sq, s4d);
    if (lane == 0) gp(ws_dp(ws, W.npart))[q.t] = tot;
  }
}

// ------------------------------------------------------------ norm, Fira, step
// _apply_update_pytorch with Fira (optimizer.py:796-810, 859-875).
__global__ __launch_bounds__(256) void k_fnorm(const DescF* __restrict__ table, HyperF h) {
  __shared__ double sd[4];
  const DescF D = table[blockIdx.x];
  const FWs W = fws_layout(D.B, D.R, D.C, D.tr);
  float* ws = D.ws;
  double s = 0.0;
  const int64_t np = D.tiled ? W.nutile : W.nunit;
  for (int64_t k = threadIdx.x; k < np; k += 256) s += gp(ws_dp(ws, W.npart))[k];
  s = wg_sum_d(s, sd);
  if (threadIdx.x == 0) {
    float* sl = ws + W.scal;
    float nrm = sqrtf((float)s);
    float fs = 1.0f;
    if (h.fira) {
      const bool fin = __builtin_isfinite(nrm);
      if (!fin) nrm = 0.0f;            // u.zero_(); norm.zero_()
      float next = nrm;
      if (D.has_fira_prev) {
        const float p = *gp(D.fira_prev);
        const float ratio = nrm / (p + 1e-8f);
        const float lim = (ratio != ratio ? ratio : fmaxf(ratio, h.margin)) / h.margin;
        const bool reset = p < 1e-6f;
        fs = reset ? 1.0f : 1.0f / lim;
        next = reset ? nrm : nrm * fs;
      }
      *gp(D.fira_prev) = next;
      if (!fin) fs = 0.0f;
    }
    float denom = 1.0f;   // CAME applies its update unclipped (optimizer.py:955)
    if (h.d > 0.0f && !h.came) denom = fmaxf(nrm / (float)(sqrt((double)D.numel) * (double)h.d), 1.0f);
    const float alpha = gp(sl)[0];
    gp(sl)[1] = alpha / denom;
    gp(sl)[2] = fs;
  }
}

// CAME clip factor of U = (g * inv_row) * inv_col (optimizer.py:824-829):
// clip = max((||U|| / sqrt(n)) / d, 1), from the norm pass's unit partials.
__global__ __launch_bounds__(256) void k_fclip(const DescF* __restrict__ table, HyperF h) {
  __shared__ double sd[4];
  const DescF D = table[blockIdx.x];
  const FWs W = fws_layout(D.B, D.R, D.C, D.tr);
  float* ws = D.ws;
  double s = 0.0;
  const int64_t np = D.tiled ? W.nutile : W.nunit;
  for (int64_t k = threadIdx.x; k < np; k += 256) s += gp(ws_dp(ws, W.npart))[k];
  s = wg_sum_d(s, sd);
  if (threadIdx.x == 0) {
    const float rms = sqrtf((float)s) / (float)sqrt((double)D.numel);
    gp(ws)[W.scal + 4] = fmaxf(rms / h.d, 1.0f);
  }
}

hipError_t factored_upload_qmap(const float* q8, const float* q4) { return upload_qmap_tu(q8, q4); }

// ------------------------------------------------------------ launch glue
template <typename T>
static int launch_stats(bool psq, const DescF* tab, int ntab, int64_t ntiles, hipStream_t st) {
  if (psq) hipLaunchKernelGGL((k_fstats<T, true>), dim3((unsigned)ntiles), dim3(256), 0, st, tab, ntab);
  else hipLaunchKernelGGL((k_fstats<T, false>), dim3((unsigned)ntiles), dim3(256), 0, st, tab, ntab);
  return check_launch("k_fstats");
}

// Work split of the update passes: tensors with the tiled layout (k_fupdt,
// over the statistics tiles) and the rest (k_fupdate, over flat units).
struct UpdGrid {
  int64_t ntiles, nunits;
  bool any_tiled, any_cut, any_flat;
};

template <typename T, int MODE, bool SR, bool CM>
static int launch_update_m(int mk, const DescF* tab, int ntab, const UpdGrid& ug, const HyperF& h,
                           hipStream_t st) {
  const dim3 b(256);
  if (ug.any_tiled) {
    const dim3 g((unsigned)ug.ntiles);
    if constexpr (CM) {
      if (mk == 1) hipLaunchKernelGGL((k_fupdt<T, MODE, SR, 1, true, false>), g, b, 0, st, tab, ntab, h);
      else if (mk == kMkFp32) hipLaunchKernelGGL((k_fupdt<T, MODE, SR, 3, true, false>), g, b, 0, st, tab, ntab, h);
      else hipLaunchKernelGGL((k_fupdt<T, MODE, SR, 2, true, false>), g, b, 0, st, tab, ntab, h);
    } else {
      switch (mk) {
        case 0: hipLaunchKernelGGL((k_fupdt<T, MODE, SR, 0, false, false>), g, b, 0, st, tab, ntab, h); break;
        case 1: hipLaunchKernelGGL((k_fupdt<T, MODE, SR, 1, false, false>), g, b, 0, st, tab, ntab, h); break;
        case kMkFp32: hipLaunchKernelGGL((k_fupdt<T, MODE, SR, 3, false, false>), g, b, 0, st, tab, ntab, h); break;
        default: hipLaunchKernelGGL((k_fupdt<T, MODE, SR, 2, false, false>), g, b, 0, st, tab, ntab, h); break;
      }
    }
    int rc = check_launch("k_fupdt");
    if (rc) return rc;
  }
  if (ug.any_cut) {   // no momentum, or fp32 momentum
    const dim3 g((unsigned)ug.ntiles);
    if constexpr (CM) hipLaunchKernelGGL((k_fupdt<T, MODE, SR, 3, true, true>), g, b, 0, st, tab, ntab, h);
    else if (mk == kMkFp32) hipLaunchKernelGGL((k_fupdt<T, MODE, SR, 3, false, true>), g, b, 0, st, tab, ntab, h);
    else hipLaunchKernelGGL((k_fupdt<T, MODE, SR, 0, false, true>), g, b, 0, st, tab, ntab, h);
    int rc = check_launch("k_fupdt");
    if (rc) return rc;
  }
  if (ug.any_flat && h.lbm < 0) {   // general B_M: every tensor is flat, units of h.unit
    const dim3 g((unsigned)ug.nunits);
    if constexpr (CM) hipLaunchKernelGGL((k_fupdate_gen<T, MODE, SR, 2, true>), g, b, 0, st, tab, ntab, h);
    else if (mk == 0) hipLaunchKernelGGL((k_fupdate_gen<T, MODE, SR, 0, false>), g, b, 0, st, tab, ntab, h);
    else hipLaunchKernelGGL((k_fupdate_gen<T, MODE, SR, 2, false>), g, b, 0, st, tab, ntab, h);
    return check_launch("k_fupdate_gen");
  }
  if (ug.any_flat) {
    const dim3 g((unsigned)ug.nunits);
    if constexpr (CM) {
      if (mk == 1) hipLaunchKernelGGL((k_fupdate<T, MODE, SR, 1, true>), g, b, 0, st, tab, ntab, h);
      else if (mk == kMkFp32) hipLaunchKernelGGL((k_fupdate<T, MODE, SR, 3, true>), g, b, 0, st, tab, ntab, h);
      else hipLaunchKernelGGL((k_fupdate<T, MODE, SR, 2, true>), g, b, 0, st, tab, ntab, h);
    } else {
      switch (mk) {
        case 0: hipLaunchKernelGGL((k_fupdate<T, MODE, SR, 0, false>), g, b, 0, st, tab, ntab, h); break;
        case 1: hipLaunchKernelGGL((k_fupdate<T, MODE, SR, 1, false>), g, b, 0, st, tab, ntab, h); break;
        case kMkFp32: hipLaunchKernelGGL((k_fupdate<T, MODE, SR, 3, false>), g, b, 0, st, tab, ntab, h); break;
        default: hipLaunchKernelGGL((k_fupdate<T, MODE, SR, 2, false>), g, b, 0, st, tab, ntab, h); break;
      }
    }
    return check_launch("k_fupdate");
  }
  return 0;
}

template <typename T, bool SR, bool CM>
static int launch_update(int mode, int mk, const DescF* tab, int ntab, const UpdGrid& ug, const HyperF& h,
                         hipStream_t st) {
  switch (mode) {
    case 0: return launch_update_m<T, 0, SR, CM>(mk, tab, ntab, ug, h, st);
    case 1: return launch_update_m<T, 1, false, CM>(mk, tab, ntab, ug, h, st);
    default: return launch_update_m<T, 2, SR, CM>(mk, tab, ntab, ug, h, st);
  }
}

static int launch_colsum(const DescF* tab, int ntab, int64_t ncs, hipStream_t st) {
  if (ncs <= 0) return 0;
  hipLaunchKernelGGL(k_fcolsum, dim3((unsigned)ncs), dim3(256), 0, st, tab, ntab);
  return check_launch("k_fcolsum");
}

template <bool CONF>
static int launch_finish(int bits, const DescF* tab, int ntab, int64_t nfblk, const HyperF& h,
                         hipStream_t st) {
  const dim3 g((unsigned)nfblk), b(256), bb(h.block_size >= 1024 ? 1024 : 256);
  switch (bits) {
    case 8: hipLaunchKernelGGL((k_fblock<8, CONF>), g, bb, 0, st, tab, ntab, h); break;
    case 16: hipLaunchKernelGGL((k_fblock<16, CONF>), g, bb, 0, st, tab, ntab, h); break;
    default: hipLaunchKernelGGL((k_fblock<0, CONF>), g, bb, 0, st, tab, ntab, h); break;
  }
  int rc = check_launch("k_fblock");
  if (rc) return rc;
  hipLaunchKernelGGL((k_frows<CONF>), dim3((unsigned)ntab), b, 0, st, tab, h);
  return check_launch("k_frows");
}

// Launch sequence of one group step.  Plain factored: stats, finish, then the
// update (with a norm pass + k_fnorm first when clipping or Fira is on).  CAME:
// stats, finish, [U norm + k_fclip when d > 0], k_came1, confidence finish,
// [update norm + k_fnorm with Fira], update.
template <typename T, bool SR>
static int run_group(const DescF* tab, int ntab, int64_t ntiles, const UpdGrid& ug, int64_t nfblk, int64_t ncs,
                     int vbits, int cbits, bool clip, const HyperF& h, hipStream_t st) {
  int rc = launch_stats<T>(h.scale_param != 0, tab, ntab, ntiles, st);
  if (rc) return rc;
  if ((rc = launch_colsum(tab, ntab, ncs, st))) return rc;
  if ((rc = launch_finish<false>(vbits, tab, ntab, nfblk, h, st))) return rc;
  if (h.came) {
    if (h.d > 0.0f) {
      if ((rc = launch_update<T, false, false>(1, 0, tab, ntab, ug, h, st))) return rc;
      hipLaunchKernelGGL(k_fclip, dim3((unsigned)ntab), dim3(256), 0, st, tab, h);
      if ((rc = check_launch("k_fclip"))) return rc;
    }
    if (h.mk == 1) hipLaunchKernelGGL((k_came1<T, 1>), dim3((unsigned)ntiles), dim3(256), 0, st, tab, ntab, h);
    else if (h.mk == kMkFp32) hipLaunchKernelGGL((k_came1<T, 3>), dim3((unsigned)ntiles), dim3(256), 0, st, tab, ntab, h);
    else hipLaunchKernelGGL((k_came1<T, 2>), dim3((unsigned)ntiles), dim3(256), 0, st, tab, ntab, h);
    if ((rc = check_launch("k_came1"))) return rc;
    if ((rc = launch_colsum(tab, ntab, ncs, st))) return rc;
    if ((rc = launch_finish<true>(cbits, tab, ntab, nfblk, h, st))) return rc;
    if (!h.fira) return launch_update<T, SR, true>(0, h.mk, tab, ntab, ug, h, st);
    if ((rc = launch_update<T, false, true>(1, h.mk, tab, ntab, ug, h, st))) return rc;
    hipLaunchKernelGGL(k_fnorm, dim3((unsigned)ntab), dim3(256), 0, st, tab, h);
    if ((rc = check_launch("k_fnorm"))) return rc;
    return launch_update<T, SR, true>(2, h.mk, tab, ntab, ug, h, st);
  }
  if (!clip) return launch_update<T, SR, false>(0, h.mk, tab, ntab, ug, h, st);
  if ((rc = launch_update<T, false, false>(1, h.mk, tab, ntab, ug, h, st))) return rc;
  hipLaunchKernelGGL(k_fnorm, dim3((unsigned)ntab), dim3(256), 0, st, tab, h);
  if ((rc = check_launch("k_fnorm"))) return rc;
  return launch_update<T, SR, false>(2, h.mk, tab, ntab, ug, h, st);
}

static int mk_code(int mbits, int mmode) {
  if (mmode == 0) return mbits == 8 ? 1 : 2;
  return mbits == 8 ? 3 : 4;
}

}  // namespace a8

using namespace a8;

extern "C" {

int64_t a8_factored_workspace_floats(int64_t batch, int64_t rows, int64_t cols) {
  return a8_factored_group_workspace_floats(batch, rows, cols, batch * rows * cols);
}

int64_t a8_factored_group_workspace_floats(int64_t batch, int64_t rows, int64_t cols, int64_t total) {
  if (batch <= 0 || rows <= 0 || cols <= 0) return 0;
  return fws_layout(batch, rows, cols, fws_tile_rows(rows, total)).total;
}

int64_t a8_table_bytes_2d(int ntensors) { return (int64_t)sizeof(DescF) * (int64_t)ntensors; }

int a8_factored_step(int dtype, int stochastic, const a8_tensor2d* tensors, int ntensors,
                     void* table_dev, int64_t table_bytes, int upload, double beta_val, float eps1,
                     float eps2, float lr_val, int scale_parameter, int bias_mode, float bias_factor,
                     float weight_decay, int wd_mode, float d, int fira, float fira_margin,
                     float log_floor, int v_bits, int block_size, double beta1, int m_block_size,
                     int m_bits, int m_mode, uint64_t sr_step, int came, double beta3, float eps_came,
                     int c_bits, const void* step_scalars, void* stream) {
  if (ntensors <= 0) return 0;
  if (dtype != A8_F32 && dtype != A8_BF16 && dtype != A8_F16 && dtype != A8_F64)
    return set_error(A8_ERR_DTYPE, "dtype");
  if (v_bits != 0 && v_bits != 8 && v_bits != 16) return set_error(A8_ERR_ARG, "v_bits must be 0, 8 or 16");
  if (came && c_bits != 0 && c_bits != 8 && c_bits != 16) return set_error(A8_ERR_ARG, "c_bits must be 0, 8 or 16");
  if (block_size <= 0) return set_error(A8_ERR_BLOCK, "block_size must be positive");
  if ((int64_t)sizeof(DescF) * ntensors > table_bytes)
    return set_error(A8_ERR_SIZE, "table_dev too small: need a8_table_bytes_2d(ntensors)");
  const bool m32 = tensors[0].m != nullptr;
  const bool has_m = tensors[0].m_q != nullptr || m32;
  int lbm = 5, gbm = 0, gunit = 0;
  if (has_m && !m32) {
    if (!((m_bits == 8 || m_bits == 4) && (m_mode == 0 || m_mode == 1)))
      return set_error(A8_ERR_ARG, "m_bits must be 4/8 and m_mode 0/1");
    if (m_block_size < 32 || m_block_size > (1 << 30) || (m_block_size & 3))
      return set_error(A8_ERR_BLOCK, "m_block_size must be a multiple of 4 in [32, 2^30]");
    if (m_block_size <= kUnit && !(m_block_size & (m_block_size - 1))) {
      lbm = 0;
      while ((1 << lbm) < m_block_size) ++lbm;
    } else {   // k_fupdate_gen: whole M blocks per workgroup, at least kUnit elements
      lbm = -1;
      gbm = m_block_size;
      gunit = m_block_size * ((kUnit + m_block_size - 1) / m_block_size);
    }
  }
  if (came && !has_m) return set_error(A8_ERR_ARG, "CAME needs momentum (m_q or m)");
  if (stochastic && dtype == A8_F32) stochastic = 0;
  std::vector<DescF> tab((size_t)ntensors);
  int64_t tiles = 0, utiles = 0, units = 0, fblks = 0, csw = 0;
  bool any_tiled = false, any_cut = false, any_flat = false;
  int64_t total = 0;
  for (int i = 0; i < ntensors; ++i) total += tensors[i].batch * tensors[i].rows * tensors[i].cols;
  for (int i = 0; i < ntensors; ++i) {
    const a8_tensor2d& t = tensors[i];
    if (t.batch <= 0 || t.rows <= 0 || t.cols <= 0) return set_error(A8_ERR_SIZE, "empty factored tensor");
    if (!t.param || !t.grad || !t.workspace) return set_error(A8_ERR_ARG, "null param/grad/workspace");
    if ((t.m_q != nullptr) != (has_m && !m32) || (t.m != nullptr) != m32)
      return set_error(A8_ERR_ARG, "mixed momentum kinds in one launch");
    if (v_bits ? !(t.row_q && t.col_q && t.row_scale && t.col_scale && t.row_min_log && t.col_min_log)
               : !(t.row_var && t.col_var))
      return set_error(A8_ERR_ARG, "row/column state missing");
    if (fira && !t.fira_prev_norm) return set_error(A8_ERR_ARG, "fira needs fira_prev_norm");
    if (came && (c_bits ? !(t.conf_row_q && t.conf_col_q && t.conf_row_scale && t.conf_col_scale &&
                            t.conf_row_min_log && t.conf_col_min_log)
                        : !(t.conf_row && t.conf_col)))
      return set_error(A8_ERR_ARG, "CAME confidence state missing");
    if (!aligned16(t.param) || !aligned16(t.grad) || (has_m && !aligned16(m32 ? (const void*)t.m : t.m_q)))
      return set_error(A8_ERR_ALIGN, "param/grad/momentum buffers must be 16-byte aligned");
    const int64_t numel = t.batch * t.rows * t.cols;
    if (numel >= ((int64_t)1 << 40)) return set_error(A8_ERR_SIZE, "tensor too large");
    DescF& D = tab[(size_t)i];
    D.param = t.param; D.grad = t.grad; D.m_q = t.m_q; D.m_scale = t.m_scale; D.m = t.m;
    D.row_q = t.row_q; D.row_scale = t.row_scale; D.row_min_log = t.row_min_log; D.row_var = t.row_var;
    D.col_q = t.col_q; D.col_scale = t.col_scale; D.col_min_log = t.col_min_log; D.col_var = t.col_var;
    D.crow_q = t.conf_row_q; D.crow_scale = t.conf_row_scale; D.crow_min_log = t.conf_row_min_log;
    D.crow_var = t.conf_row; D.ccol_q = t.conf_col_q; D.ccol_scale = t.conf_col_scale;
    D.ccol_min_log = t.conf_col_min_log; D.ccol_var = t.conf_col;
    D.ws = t.workspace; D.lr = t.lr; D.fira_prev = t.fira_prev_norm; D.has_fira_prev = t.has_fira_prev;
    D.B = t.batch; D.R = t.rows; D.C = t.cols; D.numel = numel;
    D.sr_seed = t.sr_seed;
    // the tiles' loads take 32-bit byte offsets into a row
    const int64_t esz = dtype == A8_F64 ? 8 : (dtype == A8_F32 || m32 ? 4 : 2);
    D.elem = t.cols < 4 || t.cols * esz > 0xFFFFFFFFll ? 1 : 0;
    // coded momentum: whole M blocks per row (then C % 4 == 0 too)
    D.tiled = !D.elem &&
              (!has_m || m32 || (lbm >= 0 && m_block_size <= 256 && t.cols % m_block_size == 0)) ?
              (t.cols % 4 ? 2 : 1) : 0;
    (D.tiled == 0 ? any_flat : D.tiled == 1 ? any_tiled : any_cut) = true;
    D.tr = (int)fws_tile_rows(t.rows, total);
    const FWs W = fws_layout(t.batch, t.rows, t.cols, D.tr);
    D.tile_begin = tiles;
    D.utile_begin = utiles;
    D.unit_begin = units;
    D.fblk_begin = fblks;
    D.cs_begin = csw;
    D.nbr = (t.batch * t.rows + block_size - 1) / block_size;
    tiles += W.ntile;
    utiles += W.nutile;
    units += lbm >= 0 ? W.nunit : (numel + gunit - 1) / gunit;   // gunit >= kUnit: within W.nunit slots
    fblks += D.nbr + (t.batch * t.cols + block_size - 1) / block_size;
    if (W.nsplit > 1) csw += t.batch * ((t.cols + 255) / 256) * W.nsplit;
  }
  if (tiles > 0x7FFFFFFF || utiles > 0x7FFFFFFF || units > 0x7FFFFFFF || fblks > 0x7FFFFFFF || csw > 0x7FFFFFFF)
    return set_error(A8_ERR_SIZE, "too many workgroups");
  hipStream_t st = (hipStream_t)stream;
  if (upload && upload_table(table_dev, tab.data(), sizeof(DescF) * (size_t)ntensors, st) != hipSuccess)
    return set_error(A8_ERR_HIP, "table upload failed");
  HyperF h{};
  h.bv = (float)beta_val;
  h.eps1 = eps1; h.eps2 = eps2; h.lr_val = lr_val;
  h.bias_factor = bias_factor; h.bias_mode = bias_mode;
  h.scale_param = scale_parameter;
  h.wd = weight_decay; h.wd_mode = wd_mode;
  h.d = d; h.fira = fira; h.margin = (float)(1.0 + (double)fira_margin);
  h.floor_ = log_floor;
  h.w_m = (float)(1.0 - beta1);
  h.came = came ? 1 : 0;
  h.w_c = (float)(1.0 - beta3);
  h.eps_came = eps_came;
  h.block_size = block_size;
  h.mk = m32 ? kMkFp32 : (has_m ? mk_code(m_bits, m_mode) : 0);
  h.lbm = lbm;
  h.bm = gbm;
  h.unit = gunit;
  h.sr_step = sr_step;
  h.dsc = reinterpret_cast<const a8_step_scalars*>(step_scalars);
  const bool clip = d > 0.0f || fira;
  const DescF* dt = reinterpret_cast<const DescF*>(table_dev);
  const UpdGrid ug{utiles, units, any_tiled, any_cut, any_flat};
  switch (dtype) {
    case A8_F32: return run_group<float, false>(dt, ntensors, tiles, ug, fblks, csw, v_bits, c_bits, clip, h, st);
    case A8_BF16:
      return stochastic ? run_group<__hip_bfloat16, true>(dt, ntensors, tiles, ug, fblks, csw, v_bits, c_bits, clip, h, st)
                        : run_group<__hip_bfloat16, false>(dt, ntensors, tiles, ug, fblks, csw, v_bits, c_bits, clip, h, st);
    case A8_F64: return run_group<double, false>(dt, ntensors, tiles, ug, fblks, csw, v_bits, c_bits, clip, h, st);
    default:
      return stochastic ? run_group<__half, true>(dt, ntensors, tiles, ug, fblks, csw, v_bits, c_bits, clip, h, st)
                        : run_group<__half, false>(dt, ntensors, tiles, ug, fblks, csw, v_bits, c_bits, clip, h, st);
  }
}

}  // extern "C"
