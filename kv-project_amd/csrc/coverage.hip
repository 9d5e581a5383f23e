// STRATA coverage statistics on the device (gfx950): coverage_stats, STRATA_KV.py:1225-1298.
//
// For every coverage group g (host-drawn query positions, coverage_groups 1206-1222) and KV head h,
// the rows r = (query head of h, query) attend causally to the keys [0, max position]; their
// probabilities p and outputs o give, for the coded tokens j in [rs, min(re, max position + 1)) read
// at distance >= local: pR = p_j, u = ||v_j - o||^2_M (M the query head's output metric), the drop
// term (pR / max(1 - pR, 1e-6))^2 u, the key term a = pR^2 u and the read mass pR^2, averaged over
// the group's queries and normalised by the group's drop total N (over every head and token); then
// averaged over the live groups, S = sum of alpha q q^T (alpha = a row's key-term mass) normalised
// by sum_j A_j, Mbar = read-weighted mean metric, and every output + floor x its mean.
//
// Rows are laid out per KV head as [group][query head r][query, padded to 16] (row_base of a group in
// the group table); padded rows have position -1 and contribute nothing.  Launches (one stream, no
// host synchronisation, no atomics: every sum has a fixed order):
//   cov_rowstats  per (group, 64-row block, h): logits of 16-key tiles on the matrix cores
//                 (row_tiles.hpp), online max / sum per row -> row max (base 2) and 1 / sum; every
//                 key tile feeds all the block's rows a wavefront holds, the wavefronts split the keys.
//   cov_output    per (group, 64-row block, h, key split): the logits again, p = 2^(s - max) / sum in
//                 registers as the A operand of the PV product (hi + lo parts; the two 16-key tiles
//                 of a 32-key step give every lane 8 keys of its row, in an order the B operand
//                 follows), B = values of the step from an LDS tile; the split's part of o, fp32.
//   cov_metric    x M and x M x for 32 vectors per workgroup with the query head's metric staged in
//                 LDS: the row outputs (the key splits' parts summed in order; o M) and the coded
//                 values (v M v).
//   cov_rowprep   the rows' operands and values as records of 16 rows, in the order cov_terms reads.
//   cov_terms     per (h, chunk of tokens, piece of the groups reaching it): logits and v.(oM) on the
//                 matrix cores, then the per-(row, token) terms, once: the group's drop total, every
//                 row's key-term mass and the read mass per 16 rows as partials per chunk, and the
//                 group's unweighted sums per token.
//   cov_groups    N per group -> weight 1 / N (0 if N = 0), live flag.
//   cov_roww      per row (block): its group's weight x its key-term (read) mass.
//   cov_wsum      the groups' token sums with their weights: A, DD and the read mass W.
//   cov_smat      S = sum over rows of weight * alpha * (scaling q)(scaling q)^T.
//   cov_final     live average, S / sum_j A_j, Mbar, floors (one workgroup for the sums, then all).
#include <algorithm>

#include "common.hpp"
#include "mfma_common.hpp"
#include "row_tiles.hpp"

namespace kvq {
namespace {

constexpr int kCD = 128;
constexpr int kCThreads = 256;
constexpr int kCWaves = 4;
constexpr int kTW = 4;                   // wavefronts of a cov_terms workgroup
constexpr int kChunkTok = 32 * kTW;      // its tokens: two 16-token tiles per wavefront
constexpr int kGT = 8;                  // ints per group-table entry
constexpr int kMetricRows = 32;         // vectors of a cov_metric workgroup
constexpr int kOSplit = 4;              // key splits of cov_output (workgroups per 64-row item)
constexpr int kRowPart = 20;            // its rows' key-term masses, its read mass in four parts
constexpr int kTermsUnits = 1536;       // workgroups of cov_terms worth cutting the groups of a chunk for
constexpr int64_t kStoreFloats = int64_t{1} << 28;   // most floats of the stored token sums (1 GiB)
constexpr int kSSplit = 16;             // row splits of cov_smat (workgroups per 16 rows of S)
constexpr float kCLog2e = 1.4426950408889634f;

// group table entry (kGT ints): row_base, nq, nq_pad, mmax, te, local, 0, 0
struct CovParams {
  const void* qr;                        // (Hkv, NR, d) group query rows (unscaled), DT
  const int32_t* rowpos;                 // (NR): position of each row (-1: padding)
  const int32_t* gtab;                   // (G, kGT)
  const int32_t* items;                  // (n_items, 2): (group, 64-row block)
  const void* k;
  const void* v;
  int64_t k_sh, k_st, v_sh, v_st;        // element strides of the (head, token) axes
  const float* M;                        // (Hq, d, d)
  int Hkv, rep, NR, G, n_items, rs, re, n, n_chunks, T;
  float qscale;                          // scaling * log2(e)
  float scaling, eta;
  float* row_m;                          // (Hkv, NR) row max (base 2)
  float* row_il;                         // (Hkv, NR) 1 / row sum
  float* o;                              // (Hkv, NR, d) o M (cov_metric over the summed outputs)
  float* o_part;                         // (kOSplit, Hkv, NR, d) fp32 outputs of each key split
  float* oMo;                            // (Hkv, NR)
  uint32_t* rec;                         // (Hkv, NR / 16) records of cov_terms (rec_units<DT> u32x4)
  float* vmv;                            // (Hkv, rep, n)
  float* ddpart;                         // (G, Hkv, n_chunks, kTW): drop totals per wavefront
  float* row_part;                       // (Hkv, n_chunks, NR / 16, kRowPart): a 16-row block over a chunk
  float* tsum;                           // (G, Hkv, 3, store_n): a group's key term, drop term, read mass per token
  float* gw;                             // (2 G + 1): 1 / N or 0 per group; [G + 1 + group]: 1 if live
  float* roww;                           // (Hkv, NR): weight * alpha
  float* omega;                          // (Hkv, NR / 16, 4): weight * read mass of a block, in parts
  float* red;                            // finalisation sums
  float* sums;                           // (Hkv, 2 + rep): per-head sums of A, DD, read masses
  float* A;                              // (Hkv, n)
  float* W;                              // (Hkv, n)
  float* DD;                             // (Hkv, n)
  float* S;                              // (Hkv, d, d)
  float* S_part;                         // (kSSplit, Hkv, d, d): each row split's sum
  float* Mbar;                           // (Hkv, d, d)
  // fp32 rows: the powers of two of qr, k and v (rows_scale_kernel, row_tiles.hpp); null otherwise
  const float* xs;
};

// the power of two of fp32 view i (0: qr, 1: k, 2: v); 16-bit rows are exact operands: 1
template <int DT>
__device__ __forceinline__ float cov_xs(const CovParams& p, int i) {
  if constexpr (DT == KVQ_F32) return p.xs[i];
  else return 1.0f;
}

// the rows of head h as a buffer resource covering T token rows (reads past it return zero)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t head_rsrc(const void* base, int64_t sh, int64_t st, int h, int T,
                                                           int esz) {
  const char* b = static_cast<const char*>(base) + static_cast<int64_t>(h) * sh * esz;
  return make_rsrc(b, static_cast<uint32_t>((static_cast<int64_t>(T - 1) * st + kCD) * esz));
}

// Work unit of this block when each XCD (blocks b % 8, dispatched round-robin) takes a contiguous
// range of the units, so neighbouring units, which read overlapping keys and values, share one L2;
// -1 past the last unit (grids are rounded up to a multiple of 8)
__device__ __forceinline__ int xcd_unit(int n_units) {
  const int per = (n_units + 7) / 8;
  const int u = static_cast<int>(blockIdx.x % 8) * per + static_cast<int>(blockIdx.x / 8);
  return u < n_units ? u : -1;
}
inline unsigned xcd_grid(int64_t n_units) { return static_cast<unsigned>(8 * ((n_units + 7) / 8)); }

template <int DT>
__device__ __forceinline__ void zero_ops(u32x4 (&op)[4][TileOps<DT>::NH]) {
#pragma unroll
  for (int ks = 0; ks < 4; ++ks)
#pragma unroll
    for (int hh = 0; hh < TileOps<DT>::NH; ++hh) op[ks][hh] = u32x4{0u, 0u, 0u, 0u};
}

// query operands (B) of the 16 rows starting at row0 of head h; returns this lane's row position
template <int DT>
__device__ __forceinline__ int load_rows(const CovParams& p, int h, int row0, int g, int n,
                                         u32x4 (&qop)[4][TileOps<DT>::NH]) {
  const int row = row0 + n;
  const int pos = row < p.NR ? p.rowpos[row] : -1;
  if (pos >= 0) {
    const int64_t base = (static_cast<int64_t>(h) * p.NR + row) * kCD;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) load_op<DT>(p.qr, base + 32 * ks + 8 * g, qop[ks], cov_xs<DT>(p, 0));
  } else {
    zero_ops<DT>(qop);
  }
  return pos;
}

// A operand (tokens) of the 16-token tile at t0: this lane's token t0 + n
template <int DT>
__device__ __forceinline__ void load_tile(__amdgpu_buffer_rsrc_t rs, int64_t st, int t0, int g, int n,
                                          u32x4 (&op)[4][TileOps<DT>::NH], float sc) {
  const int64_t tok = t0 + n;
#pragma unroll
  for (int ks = 0; ks < 4; ++ks)
    load_op_buf<DT>(rs, static_cast<int>((tok * st + 32 * ks + 8 * g) * TileOps<DT>::ESZ), op[ks], sc);
}

// Every key tile a wavefront loads feeds several of the item's 16-row blocks (16-bit data: all four,
// eight wavefronts (two per SIMD) splitting the keys in eighths; fp32 operands take twice the
// registers: two blocks, four wavefronts in halves), so the workgroup reads its keys once instead of
// once per row block.  The wavefronts' states of a row meet in LDS, split by split in a fixed order.
// The items go in reverse plan order: the groups at the end of the context, whose keys reach
// furthest, start first.
template <int DT>
__global__ __launch_bounds__(DT == KVQ_F32 ? kCThreads : 2 * kCThreads) void cov_rowstats(CovParams p) {
  constexpr int NH = TileOps<DT>::NH;
  constexpr int NW = DT == KVQ_F32 ? kCWaves : 2 * kCWaves;  // wavefronts (16-bit: two per SIMD)
  constexpr int NRB = DT == KVQ_F32 ? 2 : 4;                 // row blocks per wavefront
  constexpr int KS = NW * NRB / 4;                           // key splits (wavefronts sharing blocks)
  __shared__ float st[NW][NRB][16][2];
  const int wave = threadIdx.x / 64, l = threadIdx.x % 64, g = l >> 4, n = l & 15;
  const int unit = xcd_unit(p.Hkv * p.n_items);                // (h, item), h outermost
  if (unit < 0) return;
  const int item = p.n_items - 1 - unit % p.n_items, h = unit / p.n_items;
  const int grp = p.items[2 * item], rb = p.items[2 * item + 1];
  const int32_t* gt = p.gtab + kGT * grp;
  const int rows_g = p.rep * gt[2];
  const int mmax = gt[3];
  const int ks = wave % KS, rgrp = wave / KS;
  u32x4 qop[NRB][4][NH];
  int pos[NRB];
#pragma unroll
  for (int b = 0; b < NRB; ++b) {
    const int rl = 64 * rb + 16 * (rgrp * NRB + b);           // first row of the block in the group
    if (rl < rows_g) {
      pos[b] = load_rows<DT>(p, h, gt[0] + rl, g, n, qop[b]);
    } else {
      pos[b] = -1;
      zero_ops<DT>(qop[b]);
    }
  }
  // this split's keys: whole 16-key tiles
  const int ntile = (mmax + 15) / 16;
  const int k0 = 16 * (ntile * ks / KS), k1 = min(mmax, 16 * (ntile * (ks + 1) / KS));
  const __amdgpu_buffer_rsrc_t rk = head_rsrc(p.k, p.k_sh, p.k_st, h, p.T, TileOps<DT>::ESZ);
  const float qsc = p.qscale / (cov_xs<DT>(p, 0) * cov_xs<DT>(p, 1));   // logit scale of the scaled rows
  float m[NRB], ls[NRB];
#pragma unroll
  for (int b = 0; b < NRB; ++b) {
    m[b] = -INFINITY;
    ls[b] = 0.0f;
  }
  // three key tiles in rotation: two in flight behind the one computed (a tile past the split reads
  // zeros through the buffer resource or in-range keys, masked or never computed)
  u32x4 kt[3][4][NH];
  load_tile<DT>(rk, p.k_st, k0, g, n, kt[0], cov_xs<DT>(p, 1));
  load_tile<DT>(rk, p.k_st, k0 + 16, g, n, kt[1], cov_xs<DT>(p, 1));
  auto tile = [&](int t0, const u32x4 (&kop)[4][NH]) {
#pragma unroll
    for (int b = 0; b < NRB; ++b) {
      const f32x4 d = tile_dots<DT, NH, NH>(kop, qop[b]);
      float sv[4], mt = -INFINITY;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int j = t0 + 4 * g + i;
        sv[i] = (j <= pos[b] && j < mmax) ? d[i] * qsc : -INFINITY;
        mt = fmaxf(mt, sv[i]);
      }
      if (mt > m[b]) {
        ls[b] *= __builtin_amdgcn_exp2f(m[b] - mt);
        m[b] = mt;
      }
      if (m[b] != -INFINITY) {
#pragma unroll
        for (int i = 0; i < 4; ++i) ls[b] += __builtin_amdgcn_exp2f(sv[i] - m[b]);
      }
    }
  };
  for (int t0 = k0; t0 < k1; t0 += 48) {
    load_tile<DT>(rk, p.k_st, t0 + 32, g, n, kt[2], cov_xs<DT>(p, 1));
    tile(t0, kt[0]);
    if (t0 + 16 >= k1) break;
    load_tile<DT>(rk, p.k_st, t0 + 48, g, n, kt[0], cov_xs<DT>(p, 1));
    tile(t0 + 16, kt[1]);
    if (t0 + 32 >= k1) break;
    load_tile<DT>(rk, p.k_st, t0 + 64, g, n, kt[1], cov_xs<DT>(p, 1));
    tile(t0 + 32, kt[2]);
  }
  // lanes (0..3, n) hold disjoint keys of row n: this split's state of the row
#pragma unroll
  for (int b = 0; b < NRB; ++b) {
    const float M = xmax32(xmax16(m[b]));
    const float part = (M == -INFINITY || m[b] == -INFINITY) ? 0.0f : ls[b] * __builtin_amdgcn_exp2f(m[b] - M);
    const float L = xsum32(xsum16(part));
    if (g == 0) {
      st[wave][b][n][0] = M;
      st[wave][b][n][1] = L;
    }
  }
  __syncthreads();
  // thread t < 64: row t % 16 of the item's block t / 16, its splits combined in order
  if (threadIdx.x < 64) {
    const int rbi = threadIdx.x / 16, row = threadIdx.x % 16;
    const int rg = rbi / NRB, b = rbi % NRB;
    float M = -INFINITY;
#pragma unroll
    for (int s = 0; s < KS; ++s) M = fmaxf(M, st[rg * KS + s][b][row][0]);
    float L = 0.0f;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const float ms = st[rg * KS + s][b][row][0];
      if (ms != -INFINITY) L += st[rg * KS + s][b][row][1] * __builtin_amdgcn_exp2f(ms - M);
    }
    const int rl = 64 * rb + 16 * rbi;
    const int r_abs = gt[0] + rl + row;
    if (rl < rows_g && r_abs < p.NR) {
      const int64_t o = static_cast<int64_t>(h) * p.NR + r_abs;
      p.row_m[o] = M == -INFINITY ? 0.0f : M;                // padding rows: every p is masked to 0 below
      p.row_il[o] = L > 0.0f ? 1.0f / L : 0.0f;
    }
  }
}

// values of one 32-key step in LDS: [key][channel].  fp32 rows are padded by 8 bytes against bank
// conflicts; 16-bit rows take 288 bytes (72 words), so that the transposed reads of a channel block
// (16 lanes reading 8 bytes each of 4 keys x 4 channel quads) fall on distinct banks
template <int DT>
constexpr int vrow_words() { return DT == KVQ_F32 ? (kCD * 4 + 8) / 4 : 72; }

typedef short tr16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) tr16x4 lds_tr16x4;

template <int DT>
__global__ __launch_bounds__(kCThreads) void cov_output(CovParams p) {
  constexpr int ESZ = TileOps<DT>::ESZ;
  constexpr int VRW = vrow_words<DT>();
  constexpr int U16 = kCD * ESZ / 16;                        // 16-byte units of a value row
  __shared__ __align__(16) uint32_t vt[32 * VRW];
  const int wave = threadIdx.x / 64, l = threadIdx.x % 64, g = l >> 4, n = l & 15;
  // work units (h, item, key split), h outermost; the items in reverse plan order, so the groups at
  // the end of the context, whose keys reach furthest, start first and the short ones fill the tail
  const int unit = xcd_unit(p.Hkv * kOSplit * p.n_items);
  if (unit < 0) return;
  const int h = unit / (p.n_items * kOSplit), w = unit % (p.n_items * kOSplit);
  const int item = p.n_items - 1 - w / kOSplit, sp = w % kOSplit;
  const int grp = p.items[2 * item], rb = p.items[2 * item + 1];
  const int32_t* gt = p.gtab + kGT * grp;
  const int rows_g = p.rep * gt[2];
  const int row0 = gt[0] + 64 * rb + 16 * wave;
  const bool active = 64 * rb + 16 * wave < rows_g;        // inactive wavefronts still join the barriers
  u32x4 qop[4][TileOps<DT>::NH];
  int pos = -1;
  if (active)
    pos = load_rows<DT>(p, h, row0, g, n, qop);
  else
    zero_ops<DT>(qop);
  const float rm = (active && row0 + n < p.NR) ? p.row_m[static_cast<int64_t>(h) * p.NR + row0 + n] : 0.0f;
  const int mmax = gt[3];
  // this workgroup's keys: split sp of the item's 32-key steps (every split writes its partial,
  // zeros when it holds no keys; the probabilities use the row's global maximum and sum, so the
  // partials add up to o)
  const int nstep = (mmax + 31) / 32;
  const int k0 = 32 * (nstep * sp / kOSplit), k1 = min(mmax, 32 * (nstep * (sp + 1) / kOSplit));
  const __amdgpu_buffer_rsrc_t rk = head_rsrc(p.k, p.k_sh, p.k_st, h, p.T, ESZ);
  const __amdgpu_buffer_rsrc_t rv = head_rsrc(p.v, p.v_sh, p.v_st, h, p.T, ESZ);
  const float qsc = p.qscale / (cov_xs<DT>(p, 0) * cov_xs<DT>(p, 1));   // logit scale of the scaled rows
  const float vsc = cov_xs<DT>(p, 2);
  f32x4 acc[8];
#pragma unroll
  for (int cb = 0; cb < 8; ++cb) acc[cb] = f32x4{0.f, 0.f, 0.f, 0.f};
  // a step's loads: its 32 value rows (this thread's 16-byte units; rows at or past mmax as zeros:
  // p = 0 there must not meet a NaN) and this wavefront's two key tiles.  The next step's loads go
  // out as soon as the current key tiles have entered the logit products.
  constexpr int KU = (32 * U16 + kCThreads - 1) / kCThreads;
  u32x4 vr[KU];
  u32x4 kr[2][4][TileOps<DT>::NH];
  auto load_step = [&](int t0) {
#pragma unroll
    for (int k = 0; k < KU; ++k) {
      const int u = threadIdx.x + kCThreads * k;
      const int key = u / U16, w16 = u % U16;
      vr[k] = u32x4{0u, 0u, 0u, 0u};
      if (u < 32 * U16 && t0 + key < k1)
        vr[k] = __builtin_amdgcn_raw_buffer_load_b128(
            rv, static_cast<int>((static_cast<int64_t>(t0 + key) * p.v_st) * ESZ + 16 * w16), 0, 0);
    }
#pragma unroll
    for (int tau = 0; tau < 2; ++tau) load_tile<DT>(rk, p.k_st, t0 + 16 * tau, g, n, kr[tau], cov_xs<DT>(p, 1));
  };
  if (k0 < k1) load_step(k0);
  for (int t0 = k0; t0 < k1; t0 += 32) {
    // LDS-only barriers: the key tiles of the step stay in flight while its value rows are stored
    block_lds_barrier();                                     // the previous step's value rows are read
#pragma unroll
    for (int k = 0; k < KU; ++k) {
      const int u = threadIdx.x + kCThreads * k;
      if (u < 32 * U16) {
        uint32_t* dst = vt + (u / U16) * VRW + 4 * (u % U16);
        if constexpr (DT == KVQ_F32) {
          dst[0] = vr[k][0];
          dst[1] = vr[k][1];
          dst[2] = vr[k][2];
          dst[3] = vr[k][3];
        } else {
          *reinterpret_cast<u32x4*>(dst) = vr[k];                // 288-byte rows: 16-byte aligned
        }
      }
    }
    block_lds_barrier();
    // probabilities of the two 16-key tiles: lane (g, n) holds keys t0 + 4g + i and t0 + 16 + 4g + i
    // of row n
    f32x4 dd[2];
#pragma unroll
    for (int tau = 0; tau < 2; ++tau) dd[tau] = tile_dots<DT, TileOps<DT>::NH, TileOps<DT>::NH>(kr[tau], qop);
    if (t0 + 32 < k1) load_step(t0 + 32);
    float pr[8];
#pragma unroll
    for (int tau = 0; tau < 2; ++tau) {
      const f32x4 d = dd[tau];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int j = t0 + 16 * tau + 4 * g + i;
        pr[4 * tau + i] = (j <= pos && j < mmax) ? __builtin_amdgcn_exp2f(d[i] * qsc - rm) : 0.0f;
      }
    }
    // A operand: row n, k-index 8g + kk <-> key kk < 4 ? 4g + kk : 16 + 4g + kk - 4 (hi and lo parts)
    u32x4 ph, pl;
    f32_parts<DT>(pr, ph, pl);
    // B operand per 16-channel block cb: lane (g, n) holds the values of those keys at channel 16cb + n
#pragma unroll
    for (int cb = 0; cb < 8; ++cb) {
      const int c = 16 * cb + n;
      if constexpr (DT == KVQ_F32) {
        float x[8];
#pragma unroll
        for (int kk = 0; kk < 8; ++kk) {
          const int key = kk < 4 ? 4 * g + kk : 16 + 4 * g + kk - 4;
          x[kk] = __uint_as_float(vt[key * VRW + c]) * vsc;
        }
        u32x4 vh, vl;
        f32_parts<DT>(x, vh, vl);
        acc[cb] = tile_mfma<DT>(ph, vh, acc[cb]);
        acc[cb] = tile_mfma<DT>(pl, vh, acc[cb]);
        acc[cb] = tile_mfma<DT>(ph, vl, acc[cb]);
      } else {
        // LDS transpose reads (ds_read_b64_tr_b16): within each 16-lane group, lane n receives
        // element n & 3 of the 8-byte loads of lanes (n >> 2) + 4 j, j = 0..3.  Lane (g, q + 4 j)
        // therefore points at key 4g + j (then 16 + 4g + j), channels 16 cb + 4q .. + 3, and lane
        // (g, n) receives keys 4g .. 4g + 3 (16 + 4g ..) of channel 16 cb + n: the B operand
        const int src_key = 4 * g + (n >> 2), src_ch = 16 * cb + 4 * (n & 3);
        const uint32_t* a0 = vt + src_key * VRW + src_ch / 2;
        const tr16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr16x4*)(a0));
        const tr16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr16x4*)(a0 + 16 * VRW));
        const uint2 lw = __builtin_bit_cast(uint2, lo), hw = __builtin_bit_cast(uint2, hi);
        const u32x4 vb = u32x4{lw.x, lw.y, hw.x, hw.y};
        acc[cb] = tile_mfma<DT>(ph, vb, acc[cb]);
        acc[cb] = tile_mfma<DT>(pl, vb, acc[cb]);
      }
    }
  }
  if (!active) return;
  // D lane (g, n) register i: row 4g + i of the block, channel 16cb + n
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = row0 + 4 * g + i;
    if (row >= p.NR) continue;
    const float il = p.row_il[static_cast<int64_t>(h) * p.NR + row] / vsc;   // exact: vsc a power of two
    float* dst = p.o_part + ((static_cast<int64_t>(sp) * p.Hkv + h) * p.NR + row) * kCD + n;
#pragma unroll
    for (int cb = 0; cb < 8; ++cb) dst[16 * cb] = acc[cb][i] * il;
  }
}

// v M v of the coded values on the matrix cores (the row outputs' o M stays on cov_metric): per
// (query head hr = (h, r), kVmvPer values) a workgroup stages that head's metric M transposed in LDS
// as fp16 hi + lo parts of M x 2^(8 - em) (its largest entry brought to [128, 256)); each wavefront
// then takes tiles of 16 values, every value row x scaled by its own power of two the same way and
// split into parts, y = x M by the products hi*hi + hi*lo + lo*hi (fp32 accumulation, about 2^-22
// relative), and x . y by a row sum with x exchanged through the wavefront's LDS into the layout
// of the products' output.
constexpr int kVmvPer = 512;             // values of a cov_vmv workgroup
constexpr int kMtStride = kCD + 8;       // halves per LDS row of M^T (16-byte aligned rows)

template <int DT>
__global__ __launch_bounds__(kCThreads) void cov_vmv(CovParams p) {
  __shared__ __align__(16) uint16_t mt[2][kCD * kMtStride];   // [part][col][k]
  __shared__ __align__(16) float xs[kCWaves][16][kCD + 4];
  __shared__ float red[kCWaves];
  __shared__ int xex[kCWaves][16];
  const int tiles = (p.n + kVmvPer - 1) / kVmvPer;
  const int hr = blockIdx.x / tiles, tile = blockIdx.x % tiles;
  const int h = hr / p.rep;
  const int wave = threadIdx.x / 64, l = threadIdx.x % 64, g = l >> 4, n = l & 15;
  // the metric's largest entry over the workgroup, then its transposed parts
  const float* Mg = p.M + static_cast<int64_t>(hr) * kCD * kCD;
  constexpr int kPer = kCD * kCD / kCThreads;
  float mv[kPer];
  float mx = 0.0f;
#pragma unroll
  for (int e = 0; e < kPer; ++e) {
    mv[e] = Mg[threadIdx.x + kCThreads * e];
    mx = fmaxf(mx, fabsf(mv[e]));
  }
  mx = wave_max(mx);
  if (l == 0) red[wave] = mx;
  __syncthreads();
  mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  int em = 0;
  if (mx > 0.0f) (void)frexpf(mx, &em);
  const float upm = ldexpf(1.0f, 8 - em);
#pragma unroll
  for (int e = 0; e < kPer; ++e) {
    const int idx = threadIdx.x + kCThreads * e, k = idx / kCD, c = idx % kCD;
    const float x = mv[e] * upm;
    const _Float16 hi = static_cast<_Float16>(x);
    const _Float16 lo = static_cast<_Float16>(x - static_cast<float>(hi));
    mt[0][c * kMtStride + k] = __builtin_bit_cast(uint16_t, hi);
    mt[1][c * kMtStride + k] = __builtin_bit_cast(uint16_t, lo);
  }
  __syncthreads();
  for (int t0 = 0; t0 < kVmvPer; t0 += 64) {
    const int j0 = tile * kVmvPer + t0 + 16 * wave;         // this wavefront's 16 values
    const int j = j0 + n;                                   // lane (g, n): value n, channels 32 ks + 8 g ..
    float x[4][8];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      if (j < p.n) {
        load8<DT>(p.v, static_cast<int64_t>(h) * p.v_sh + static_cast<int64_t>(p.rs + j) * p.v_st + 32 * ks + 8 * g,
                  x[ks]);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) x[ks][e] = 0.0f;
      }
    }
    float mxv = 0.0f;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int e = 0; e < 8; ++e) mxv = fmaxf(mxv, fabsf(x[ks][e]));
    mxv = xmax32(xmax16(mxv));                               // over the four lanes of value n
    int ex = 0;
    if (mxv > 0.0f) (void)frexpf(mxv, &ex);
    const float upx = ldexpf(1.0f, 8 - ex);
    u32x4 xh[4], xl[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      float xs8[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) xs8[e] = x[ks][e] * upx;
      f32_parts<KVQ_F16>(xs8, xh[ks], xl[ks]);
      *reinterpret_cast<float4*>(&xs[wave][n][32 * ks + 8 * g]) = make_float4(xs8[0], xs8[1], xs8[2], xs8[3]);
      *reinterpret_cast<float4*>(&xs[wave][n][32 * ks + 8 * g + 4]) = make_float4(xs8[4], xs8[5], xs8[6], xs8[7]);
    }
    if (g == 0) xex[wave][n] = ex;
    wave_lds_fence();
    float dot[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int cb = 0; cb < 8; ++cb) {
      f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        const int o = (16 * cb + n) * kMtStride + 32 * ks + 8 * g;
        const u32x4 bh = *reinterpret_cast<const u32x4*>(&mt[0][o]);
        const u32x4 bl = *reinterpret_cast<const u32x4*>(&mt[1][o]);
        acc = mfma(as_half8(xh[ks]), as_half8(bh), acc);
        acc = mfma(as_half8(xh[ks]), as_half8(bl), acc);
        acc = mfma(as_half8(xl[ks]), as_half8(bh), acc);
      }
      // D lane (g, n) register i: value 4g + i, column 16 cb + n
#pragma unroll
      for (int i = 0; i < 4; ++i) dot[i] = __builtin_fmaf(acc[i], xs[wave][4 * g + i][16 * cb + n], dot[i]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float q = row_sum16(dot[i]);                    // over the 16 columns a lane group holds
      const int jj = j0 + 4 * g + i;
      if (n == 0 && jj < p.n) {
        // x M x = q x 2^(2 ex + em - 24): x and M entered as x 2^(8 - ex) and M 2^(8 - em)
        p.vmv[static_cast<int64_t>(hr) * p.n + jj] = ldexpf(q, 2 * xex[wave][4 * g + i] + em - 24);
      }
    }
    wave_lds_fence();                                       // xs, xex of this tile are read
  }
}

// x M and x M x for 32 vectors per workgroup, M = the metric of query head (h, r) staged in LDS in
// two halves of 64 rows.  ROWS: the row outputs of query head r (o M replaces o, o M o out);
// otherwise the coded values (v M v out).  Grid: (h, r, tile of 32 vectors).
template <int DT, bool ROWS>
__global__ __launch_bounds__(kCThreads) void cov_metric(CovParams p, const int32_t* rlist, int n_rlist) {
  constexpr int XS = kCD + 1;                          // odd stride: the rows' reads hit distinct banks
  __shared__ float Ms[64 * kCD];                       // 32 KiB
  __shared__ float xs[kMetricRows * XS];
  __shared__ float red[kMetricRows][8];
  const int count = ROWS ? n_rlist : p.n;
  const int per = (count + kMetricRows - 1) / kMetricRows;
  const int hr = blockIdx.x / per, tile = blockIdx.x % per;
  const int h = hr / p.rep, r = hr % p.rep;
  const float* Mg = p.M + static_cast<int64_t>(h * p.rep + r) * kCD * kCD;
  const int32_t* rl = ROWS ? rlist + static_cast<int64_t>(r) * n_rlist : nullptr;
  for (int u = threadIdx.x; u < kMetricRows * kCD; u += kCThreads) {
    const int k = u / kCD, c = u % kCD;
    const int idx = kMetricRows * tile + k;
    float x = 0.0f;
    if (idx < count) {
      if constexpr (ROWS) {
        if (rl[idx] >= 0) {                            // the key splits' outputs, summed in order
          const int64_t o = (static_cast<int64_t>(h) * p.NR + rl[idx]) * kCD + c;
          const int64_t split = static_cast<int64_t>(p.Hkv) * p.NR * kCD;
#pragma unroll
          for (int sp = 0; sp < kOSplit; ++sp) x += p.o_part[sp * split + o];
        }
      } else {
        x = load_as_f32<DT>(p.v, static_cast<int64_t>(h) * p.v_sh + static_cast<int64_t>(p.rs + idx) * p.v_st + c);
      }
    }
    xs[k * XS + c] = x;
  }
  // thread: vector k = t / 8, output channels 16 (t % 8) .. + 15
  const int k = threadIdx.x / 8, c8 = threadIdx.x % 8;
  float y[16];
#pragma unroll
  for (int e = 0; e < 16; ++e) y[e] = 0.0f;
  for (int hf = 0; hf < 2; ++hf) {
    __syncthreads();
    for (int u = threadIdx.x; u < 64 * kCD / 4; u += kCThreads)
      reinterpret_cast<float4*>(Ms)[u] = reinterpret_cast<const float4*>(Mg + 64 * hf * kCD)[u];
    __syncthreads();
    for (int d = 0; d < 64; ++d) {
      const float xd = xs[k * XS + 64 * hf + d];
      const float4* mr = reinterpret_cast<const float4*>(Ms + d * kCD + 16 * c8);
#pragma unroll
      for (int e4 = 0; e4 < 4; ++e4) {
        const float4 mv = mr[e4];
        y[4 * e4] = __builtin_fmaf(xd, mv.x, y[4 * e4]);
        y[4 * e4 + 1] = __builtin_fmaf(xd, mv.y, y[4 * e4 + 1]);
        y[4 * e4 + 2] = __builtin_fmaf(xd, mv.z, y[4 * e4 + 2]);
        y[4 * e4 + 3] = __builtin_fmaf(xd, mv.w, y[4 * e4 + 3]);
      }
    }
  }
  float dot = 0.0f;
#pragma unroll
  for (int e = 0; e < 16; ++e) dot = __builtin_fmaf(y[e], xs[k * XS + 16 * c8 + e], dot);
  red[k][c8] = dot;
  __syncthreads();
  const int idx = kMetricRows * tile + k;
  if (idx >= count) return;
  const float tot = ((red[k][0] + red[k][1]) + (red[k][2] + red[k][3])) +
                    ((red[k][4] + red[k][5]) + (red[k][6] + red[k][7]));
  if constexpr (ROWS) {
    if (rl[idx] < 0) return;
    const int64_t rid = static_cast<int64_t>(h) * p.NR + rl[idx];
    float* dst = p.o + rid * kCD + 16 * c8;             // this workgroup staged its rows before any write
#pragma unroll
    for (int e = 0; e < 16; ++e) dst[e] = y[e];
    if (c8 == 0) p.oMo[rid] = tot;
  } else {
    if (c8 == 0) p.vmv[(static_cast<int64_t>(h) * p.rep + r) * p.n + idx] = tot;
  }
}

// Rows of cov_terms in blocks of 16, each one contiguous record: the A operands of its products in lane
// order (part p, k-step ks, lane l at unit (4 p + ks) 64 + l: the row's DT parts, then o M times the power
// of two that brings its largest entry to [128, 256), inside the range of fp16 parts, as hi and lo
// parts), then per row the max, 1 / sum, o M o, -2 x the power of two back, and the last key it counts
// (-1: padding), and the smallest and largest of those keys.  A stage of cov_terms is a plain copy of
// its records and every operand read is 64 consecutive 16-byte units.
template <int DT>
constexpr int rec_ops() { return (TileOps<DT>::NH + 2) * 4 * 64; }            // 16-byte operand units
constexpr int kRecMeta = 32;                                                   // 16-byte units of row values (22 used)
template <int DT>
constexpr int rec_units() { return rec_ops<DT>() + kRecMeta; }

// Once per row (after cov_metric): thread (row, ks, g) converts channels 32 ks + 8 g .. + 7 of its row
template <int DT>
__global__ __launch_bounds__(kCThreads) void cov_rowprep(CovParams p, const int32_t* rowgrp) {
  constexpr int NH = TileOps<DT>::NH;
  __shared__ int lims[16];
  const int nb = p.NR / 16, h = blockIdx.x / nb, block = blockIdx.x % nb;
  const int n = threadIdx.x / 16, sl = threadIdx.x % 16, ks = sl / 4, g = sl % 4;
  const int row = 16 * block + n, pos = p.rowpos[row], grp = rowgrp[row];
  const int64_t rid = static_cast<int64_t>(h) * p.NR + row;
  u32x4* rec = reinterpret_cast<u32x4*>(p.rec) + (static_cast<int64_t>(h) * nb + block) * rec_units<DT>();
  const bool live = pos >= 0 && grp >= 0;
  const float4* src = reinterpret_cast<const float4*>(p.o + rid * kCD + 32 * ks + 8 * g);
  float x[8];
  u32x4 qop[NH];
#pragma unroll
  for (int hh = 0; hh < NH; ++hh) qop[hh] = u32x4{0u, 0u, 0u, 0u};
  if (live) {
    const float4 a = src[0], b = src[1];
    x[0] = a.x; x[1] = a.y; x[2] = a.z; x[3] = a.w;
    x[4] = b.x; x[5] = b.y; x[6] = b.z; x[7] = b.w;
    load_op<DT>(p.qr, rid * kCD + 32 * ks + 8 * g, qop, cov_xs<DT>(p, 0));
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = 0.0f;
  }
  float mx = 0.0f;
#pragma unroll
  for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf(x[e]));
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
  int ex = 0;
  if (mx > 0.0f) (void)frexpf(mx, &ex);
  const float up = ldexpf(1.0f, 8 - ex);
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] *= up;
  u32x4 hi, lo;
  f32_parts<DT>(x, hi, lo);
  const int l = 16 * g + n;
#pragma unroll
  for (int hh = 0; hh < NH; ++hh) rec[(4 * hh + ks) * 64 + l] = qop[hh];
  rec[(4 * NH + ks) * 64 + l] = hi;
  rec[(4 * NH + 4 + ks) * 64 + l] = lo;
  float* meta = reinterpret_cast<float*>(rec + rec_ops<DT>());
  int* lim = reinterpret_cast<int*>(meta) + 64;
  const int last = live ? min(pos - p.gtab[kGT * grp + 5], p.gtab[kGT * grp + 4] - 1) : -1;
  if (sl == 0) {
    meta[n] = live ? p.row_m[rid] : 0.0f;
    meta[16 + n] = live ? p.row_il[rid] : 0.0f;
    meta[32 + n] = live ? p.oMo[rid] : 0.0f;
    meta[48 + n] = -2.0f * ldexpf(1.0f, ex - 8) / cov_xs<DT>(p, 2);       // exact: powers of two
    lim[n] = last;
    lims[n] = last;
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    int m = lims[0];
    for (int i = 1; i < 16; ++i) m = threadIdx.x == 0 ? min(m, lims[i]) : max(m, lims[i]);
    lim[16 + threadIdx.x] = m;
  }
}

// The per-(row, token) terms, once: per (h, 256-token chunk, piece of the groups reaching it) the chunk's
// key and value tiles stay in registers, 32 tokens per wavefront, and the groups' rows stream past them
// through LDS (records of cov_rowprep, a block per stage, two stages, loads one more stage ahead), so
// a group's sums over its rows (key term, drop term, read mass of a token) stay in the lane until its
// last block and no wavefront waits for another within a group.  They go out unweighted, one value per
// (group, h, term, token): a group's weight needs its drop total over every token, and reading them
// back (cov_wsum) costs far less than the logits, exponentials and quotients a second time.  Per block
// the wavefronts' row sums (key-term mass) and read mass meet in LDS, added in wavefront order.
// Bound by the vector ALU and its waits: about 26 issue slots per (row, token) term, the exponential and
// the reciprocal 4 each; 168 registers (three wavefronts per SIMD) hold two tiles -- four tiles (256
// registers) spill and take 950 us, eight wavefronts per workgroup at 128 registers spill and take 1200.
// 8 heads x 4 query heads, 65 groups, 32768 bf16 keys: 705 us and 41 us to read the sums back; the two
// passes before (terms for the totals, then again with the weights, rows in registers and tokens from
// LDS) took 893 and 1287 us.
// R: tokens [store0, store0 + store_n) have their sums stored; `totals`: drop totals, key-term and read
// masses written (the first launch; later ones only fill further token ranges of the store).
struct TermsRange {
  int chunk0, chunks, store0, store_n, pieces;
  bool totals;
};

// lanes 0..31: a over the lane pair (l, l + 32); lanes 32..63: b
__device__ __forceinline__ float add32(float a, float b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// rows of 16 lanes 0 and 2: a over the row pairs (0, 1) and (2, 3); rows 1 and 3: b over them
__device__ __forceinline__ float add16(float a, float b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

template <int DT>
__global__ __launch_bounds__(64 * kTW, DT == KVQ_F32 ? 2 : 3) void cov_terms(CovParams p, TermsRange R) {
  constexpr int NH = TileOps<DT>::NH;
  constexpr int NT = 64 * kTW;
  constexpr int RU = rec_units<DT>();
  constexpr int kPer = rec_ops<DT>() / NT;               // 16-byte operand units per thread and stage
  static_assert(rec_ops<DT>() % NT == 0 && NT % kRecMeta == 0, "whole loads");
  __shared__ u32x4 stage[2][RU];
  __shared__ float vmv_lds[2][kChunkTok];                // v M v of the chunk's tokens with the block's query head
  __shared__ float red[2][kTW][kRowPart];                // a block's 16 row sums, then its read mass in four parts
  const int l = threadIdx.x % 64, g = l >> 4, n = l & 15;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  // Work units u = (h, chunk, piece) in order, a contiguous range per XCD: the pieces and chunks of a
  // head share one L2 for its rows' records.
  const int u = xcd_unit(p.Hkv * R.chunks * R.pieces);
  if (u < 0) return;
  const int ts = u % R.pieces, h = u / R.pieces / R.chunks, chunk = R.chunk0 + u / R.pieces % R.chunks;
  const int c0 = p.rs + chunk * kChunkTok;               // first token of the chunk
  // the groups that reach the chunk lie in [g0, G); this piece of them, and its blocks
  // the group table is only read here: scalar loads
  const auto gtab = reinterpret_cast<const __attribute__((address_space(4))) int32_t*>(reinterpret_cast<uintptr_t>(p.gtab));
  int g0 = p.G;
  for (int x = 0; x < p.G && g0 == p.G; x += 64) {
    const uint64_t hit = __ballot(x + l < p.G && p.gtab[kGT * min(x + l, p.G - 1) + 4] > c0);
    if (hit) g0 = x + __builtin_ctzll(hit);
  }
  const int ga = g0 + (p.G - g0) * ts / R.pieces, gb = g0 + (p.G - g0) * (ts + 1) / R.pieces;
  if (ga == gb) return;
  auto blocks_of = [&](int grp) { return p.rep * (gtab[kGT * grp + 2] / 16); };
  auto first_of = [&](int grp) { return gtab[kGT * grp] / 16; };
  int nb = 0;
  for (int x = ga; x < gb; ++x) nb += blocks_of(x);
  const u32x4* rec = reinterpret_cast<const u32x4*>(p.rec) + static_cast<int64_t>(h) * (p.NR / 16) * RU;
  u32x4 pre[kPer + 1];
  float pre_vmv;
  // the next block to load: its group, blocks left in it and in its query head
  int lg = ga, lleft = blocks_of(ga), lper = gtab[kGT * ga + 2] / 16, lbh = lper;
  const float* const vmv_h = p.vmv + static_cast<int64_t>(h) * p.rep * p.n;
  const float* vmv_r = vmv_h;
  const uint32_t vmv_tok = min(c0 + static_cast<int>(threadIdx.x % kChunkTok), p.re - 1) - p.rs;
  const u32x4* src = rec + static_cast<int64_t>(first_of(ga)) * RU;
  auto load_stage = [&]() {
#pragma unroll
    for (int i = 0; i < kPer; ++i) pre[i] = src[i * NT + threadIdx.x];
    pre[kPer] = src[kPer * NT + threadIdx.x % kRecMeta];   // (every group of threads: no branch)
    pre_vmv = vmv_r[vmv_tok];                              // (a token past the range is masked)
    if (--lleft > 0) {
      src += RU;
      if (--lbh == 0) {
        lbh = lper;
        vmv_r += p.n;
      }
    } else if (++lg < gb) {                                // past the piece: its last block again, not used
      src = rec + static_cast<int64_t>(first_of(lg)) * RU;
      lleft = blocks_of(lg);
      lbh = lper = gtab[kGT * lg + 2] / 16;
      vmv_r = vmv_h;
    }
  };
  auto store_stage = [&](int s) {
#pragma unroll
    for (int i = 0; i < kPer; ++i) stage[s & 1][i * NT + threadIdx.x] = pre[i];
    stage[s & 1][kPer * NT + threadIdx.x % kRecMeta] = pre[kPer];
    vmv_lds[s & 1][threadIdx.x % kChunkTok] = pre_vmv;
  };
  load_stage();
  const int t0 = c0 + 32 * wave;                          // this wavefront's tokens t0 .. t0 + 31
  u32x4 kop[2][4][NH], vop[2][4][NH];
  {
    const __amdgpu_buffer_rsrc_t rk = head_rsrc(p.k, p.k_sh, p.k_st, h, p.T, TileOps<DT>::ESZ);
    const __amdgpu_buffer_rsrc_t rv = head_rsrc(p.v, p.v_sh, p.v_st, h, p.T, TileOps<DT>::ESZ);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      load_tile<DT>(rk, p.k_st, t0 + 16 * t, g, n, kop[t], cov_xs<DT>(p, 1));
      load_tile<DT>(rv, p.v_st, t0 + 16 * t, g, n, vop[t], cov_xs<DT>(p, 2));
    }
  }
  const float qsc = p.qscale / (cov_xs<DT>(p, 0) * cov_xs<DT>(p, 1));   // logit scale of the scaled rows
  store_stage(0);
  load_stage();
  // block `block`'s row sums and read mass, the wavefronts' added in order by one of them
  float* row_part = p.row_part + (static_cast<int64_t>(h) * p.n_chunks + chunk) * (p.NR / 16) * kRowPart;
  auto combine = [&](int s, int block) {
    if (wave != (s & (kTW - 1)) || l >= kRowPart) return;
    float a = 0.0f;
#pragma unroll
    for (int w = 0; w < kTW; ++w) a += red[s & 1][w][l];
    (row_part + static_cast<int64_t>(block) * kRowPart)[static_cast<uint32_t>(l)] = a;
  };
  int grp = ga, left = blocks_of(ga), block = first_of(ga), last = -1;
  int ended = -1;                                          // group whose last block is done, its sums not yet out
  float rA[2] = {0.0f, 0.0f}, rD[2] = {0.0f, 0.0f}, rW[2] = {0.0f, 0.0f};   // this lane's token sums over its rows
  // group ga's token sums over the lane groups' rows, out
  auto flush = [&](int ga) {
    const int te = gtab[kGT * ga + 4];
    float* out = p.tsum + (static_cast<int64_t>(ga) * p.Hkv + h) * 3 * R.store_n;
    float dsum = 0.0f;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      // added over the lane groups and dealt to them at once: group 0 ends with A, 1 with D, 2 with W
      const float z = add16(add32(rA[t], rW[t]), add32(rD[t], rD[t]));
      rA[t] = rD[t] = rW[t] = 0.0f;
      dsum += z;
      const int j = t0 + 16 * t + n, at = j - R.store0;
      if (g < 3 && j < te && at >= 0 && at < R.store_n) out[static_cast<uint32_t>(g * R.store_n + at)] = z;
    }
    if (R.totals) {
      dsum = row_sum16(dsum);
      if (l == 16) p.ddpart[((static_cast<int64_t>(ga) * p.Hkv + h) * p.n_chunks + chunk) * kTW + wave] = dsum;
    }
  };
  for (int s = 0; s < nb; ++s) {
    __syncthreads();                                       // stage s is stored, stage s - 1 read
    store_stage(s + 1);
    load_stage();
    // the results of block s - 1 go out here, a block's work ahead of the next wait for loads
    if (R.totals && last >= 0) combine(s - 1, last);
    if (ended >= 0) flush(ended);
    ended = -1;
    const u32x4* ops = stage[s & 1];
    const float* meta = reinterpret_cast<const float*>(ops + rec_ops<DT>());
    const int* lim = reinterpret_cast<const int*>(meta) + 64;
    const int lim_min = __builtin_amdgcn_readfirstlane(lim[16]), lim_max = __builtin_amdgcn_readfirstlane(lim[17]);
    float alpha[4] = {0.0f, 0.0f, 0.0f, 0.0f}, mass = 0.0f;
    if (t0 <= lim_max) {
      f32x4 sd[2], ov[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) sd[t] = ov[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        u32x4 q[NH];
#pragma unroll
        for (int hh = 0; hh < NH; ++hh) q[hh] = ops[(4 * hh + ks) * 64 + l];
        const u32x4 mh = ops[(4 * NH + ks) * 64 + l], ml = ops[(4 * NH + 4 + ks) * 64 + l];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          sd[t] = tile_mfma<DT>(q[0], kop[t][ks][0], sd[t]);
          ov[t] = tile_mfma<DT>(mh, vop[t][ks][0], ov[t]);
          if constexpr (NH > 1) {
            sd[t] = tile_mfma<DT>(q[0], kop[t][ks][1], sd[t]);
            sd[t] = tile_mfma<DT>(q[1], kop[t][ks][0], sd[t]);
            ov[t] = tile_mfma<DT>(mh, vop[t][ks][1], ov[t]);
          }
          ov[t] = tile_mfma<DT>(ml, vop[t][ks][0], ov[t]);
        }
      }
      // rows 4g + i: their values; lane (g, n) holds the products of those rows with token t0 + 16 t + n
      const float4 m4 = *reinterpret_cast<const float4*>(meta + 4 * g);
      const float4 i4 = *reinterpret_cast<const float4*>(meta + 16 + 4 * g);
      const float4 o4 = *reinterpret_cast<const float4*>(meta + 32 + 4 * g);
      const float4 c4 = *reinterpret_cast<const float4*>(meta + 48 + 4 * g);
      const float rm[4] = {m4.x, m4.y, m4.z, m4.w}, ril[4] = {i4.x, i4.y, i4.z, i4.w};
      const float omo[4] = {o4.x, o4.y, o4.z, o4.w}, msc[4] = {c4.x, c4.y, c4.z, c4.w};
      auto terms = [&](auto edge) {
        int far[4];
        if constexpr (decltype(edge)::value) {
          const int4 f4 = *reinterpret_cast<const int4*>(lim + 4 * g);
          far[0] = f4.x; far[1] = f4.y; far[2] = f4.z; far[3] = f4.w;
        }
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const int tok = 32 * wave + 16 * t + n;
          const float vmv = vmv_lds[s & 1][tok];
          float wt = 0.0f;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            float pr = __builtin_amdgcn_exp2f(__builtin_fmaf(sd[t][i], qsc, -rm[i])) * ril[i];
            float u2 = fmaxf(__builtin_fmaf(ov[t][i], msc[i], vmv) + omo[i], 0.0f);
            if constexpr (decltype(edge)::value) {
              const bool in = c0 + tok <= far[i];
              pr = in ? pr : 0.0f;
              u2 = in ? u2 : 0.0f;
            }
            // pr / b for b = max(1 - pr, 1e-6) in [1e-6, 1]: the reciprocal's quotient and one
            // residual correction (no subnormal, infinite or zero operand can occur)
            const float qb = fmaxf(1.0f - pr, 1e-6f), rb = __builtin_amdgcn_rcpf(qb);
            const float q0 = pr * rb;
            const float qd = __builtin_fmaf(__builtin_fmaf(-qb, q0, pr), rb, q0);
            const float w = pr * pr;
            rD[t] = __builtin_fmaf(qd * qd, u2, rD[t]);
            rA[t] = __builtin_fmaf(w, u2, rA[t]);
            alpha[i] = __builtin_fmaf(w, u2, alpha[i]);
            wt = i == 0 ? w : wt + w;
          }
          rW[t] += wt;
          mass += wt;
        }
      };
      if (t0 + 31 <= lim_min) terms(std::false_type{});
      else terms(std::true_type{});
    }
    if (R.totals) {
      // the block's rows over this wavefront's tokens (the 16 lanes of group g hold them): the four rows
      // are dealt to the lanes of a quad while they are added, lane n ends with row 4g + (n & 3)
      const float a01 = (n & 1 ? alpha[1] : alpha[0]) + dpp<kQuadSwap1>(n & 1 ? alpha[0] : alpha[1]);
      const float a23 = (n & 1 ? alpha[3] : alpha[2]) + dpp<kQuadSwap1>(n & 1 ? alpha[2] : alpha[3]);
      float a = (n & 2 ? a23 : a01) + dpp<kQuadSwap2>(n & 2 ? a01 : a23);
      a += dpp<kRowRor + 4>(a);
      a += dpp<kRowRor + 8>(a);
      mass = row_sum16(mass);
      if (n < 4) red[s & 1][wave][4 * g + n] = a;
      if (n == 0) red[s & 1][wave][16 + g] = mass;
    }
    last = block++;
    if (--left > 0) continue;
    ended = grp;
    if (++grp < gb) {
      left = blocks_of(grp);
      block = first_of(grp);
    }
  }
  flush(ended);
  if (R.totals) {
    __syncthreads();
    combine(nb - 1, last);
  }
}

// chunks that a group's keys reach (its partials exist for those)
__device__ __forceinline__ int reached_chunks(const CovParams& p, int grp) {
  return max(0, min(p.n_chunks, (p.gtab[kGT * grp + 4] - p.rs + kChunkTok - 1) / kChunkTok));
}

// N per group (over heads and chunks) -> weight 1 / N (0 if N = 0) in gw[group], and whether the
// group is live (N > 0) in gw[G + 1 + group]; one workgroup per group
__global__ __launch_bounds__(kCThreads) void cov_groups(CovParams p) {
  __shared__ float red[kCWaves];
  const int grp = blockIdx.x;
  const int rc = reached_chunks(p, grp);
  // the drop total of (group, h, chunk): cov_terms' wavefront partials, in order, over nq
  const float nq = static_cast<float>(p.gtab[kGT * grp + 1]);
  float s = 0.0f;
  for (int u = threadIdx.x; u < p.Hkv * rc; u += kCThreads) {
    const float* d = p.ddpart + ((static_cast<int64_t>(grp) * p.Hkv + u / rc) * p.n_chunks + u % rc) * kTW;
    float t = 0.0f;
#pragma unroll
    for (int w = 0; w < kTW; ++w) t += d[w];
    s += t / nq;
  }
  s = wave_sum(s);
  if (threadIdx.x % 64 == 0) red[threadIdx.x / 64] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    const float N = (red[0] + red[1]) + (red[2] + red[3]);
    p.gw[grp] = N > 0.0f ? 1.0f / N : 0.0f;
    p.gw[p.G + 1 + grp] = N > 0.0f ? 1.0f : 0.0f;
  }
}

// per row: its group's weight x its key-term mass, per block: its group's weight x its read mass (in the
// four parts), summed over the chunks, a quarter of them per wavefront: the loads of one entry are a
// chain of strided reads
__global__ __launch_bounds__(kCThreads) void cov_roww(CovParams p, const int32_t* rowgrp) {
  __shared__ float part[4][64];
  const int nb = p.NR / 16;
  const int64_t t = static_cast<int64_t>(blockIdx.x) * 64 + threadIdx.x % 64;    // (h, block, entry)
  const int qt = threadIdx.x / 64, i = static_cast<int>(t % kRowPart);
  const bool in = t < static_cast<int64_t>(p.Hkv) * nb * kRowPart;
  const int hb = in ? static_cast<int>(t / kRowPart) : 0, h = hb / nb, block = hb % nb, row = 16 * block + (i < 16 ? i : 0);
  const int grp = in && p.rowpos[row] >= 0 ? rowgrp[row] : -1;
  float a = 0.0f;
  if (grp >= 0) {
    const int rc = reached_chunks(p, grp);
    const int e = rc * (qt + 1) / 4;
    const float* src = p.row_part + (static_cast<int64_t>(h) * p.n_chunks * nb + block) * kRowPart + i;
#pragma unroll 8
    for (int c = rc * qt / 4; c < e; ++c) a += src[static_cast<int64_t>(c) * nb * kRowPart];
  }
  part[qt][threadIdx.x % 64] = a;
  __syncthreads();
  if (qt || !in) return;
  const int x = threadIdx.x;
  a = (part[0][x] + part[1][x]) + (part[2][x] + part[3][x]);
  a = grp >= 0 ? a / static_cast<float>(p.gtab[kGT * grp + 1]) * p.gw[grp] : 0.0f;
  if (i < 16) p.roww[static_cast<int64_t>(h) * p.NR + row] = a;
  else p.omega[static_cast<int64_t>(hb) * 4 + i - 16] = a;
}

// the groups' stored token sums with their weights: A, DD and the read mass of the tokens
// [store0, store0 + store_n), one thread per (h, token), groups in order
__global__ __launch_bounds__(kCThreads) void cov_wsum(CovParams p, int store0, int store_n) {
  const int per = (store_n + kCThreads - 1) / kCThreads;
  const int h = blockIdx.x / per, at = blockIdx.x % per * kCThreads + static_cast<int>(threadIdx.x);
  const int j = store0 + at;
  if (at >= store_n || j >= p.re) return;
  float a = 0.0f, dd = 0.0f, w = 0.0f;
#pragma unroll 4
  for (int grp = 0; grp < p.G; ++grp) {
    const float gw = p.gw[grp];
    if (j >= p.gtab[kGT * grp + 4] || gw == 0.0f) continue;   // N = 0: every term of the group is zero
    const float wq = gw / static_cast<float>(p.gtab[kGT * grp + 1]);
    const float* src = p.tsum + (static_cast<int64_t>(grp) * p.Hkv + h) * 3 * store_n + at;
    a = __builtin_fmaf(src[0], wq, a);
    dd = __builtin_fmaf(src[store_n], wq, dd);
    w = __builtin_fmaf(src[2 * static_cast<int64_t>(store_n)], wq, w);
  }
  const int64_t o = static_cast<int64_t>(h) * p.n + (j - p.rs);
  p.A[o] = a;
  p.DD[o] = dd;
  p.W[o] = w;
}

// S[h] = sum over rows of roww * (scaling q)(scaling q)^T: per (h, 16 output rows, row split), 64
// rows per stage staged with 16-byte loads; each split writes its partial sum, cov_smat_sum adds the
// splits in order
template <int DT>
__global__ __launch_bounds__(kCThreads) void cov_smat(CovParams p) {
  constexpr int ESZ = TileOps<DT>::ESZ;
  constexpr int U = kCD * ESZ / 16;                     // 16-byte units of a row
  __shared__ float qs[64][kCD + 4];
  __shared__ float ws[64];
  const int sp = blockIdx.x % kSSplit, c1b = blockIdx.x / kSSplit % (kCD / 16);
  const int h = blockIdx.x / kSSplit / (kCD / 16);
  const int c1 = 16 * c1b + threadIdx.x / 16, c2 = 8 * (threadIdx.x % 16);   // 8 output columns per thread
  const int per = (p.NR + 64 * kSSplit - 1) / (64 * kSSplit) * 64;            // rows of a split, whole stages
  const int rb = sp * per, re = min(p.NR, rb + per);
  float acc[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] = 0.0f;
  for (int r0 = rb; r0 < re; r0 += 64) {
    __syncthreads();
    for (int u = threadIdx.x; u < 64 * U; u += kCThreads) {
      const int k = u / U, w = u % U;
      const int row = r0 + k;
      float x[16 / ESZ];
      const bool live = row < re && p.rowpos[row] >= 0;
      if constexpr (DT == KVQ_F32) {
        const float4 v = live ? *reinterpret_cast<const float4*>(static_cast<const float*>(p.qr) +
                                                                 (static_cast<int64_t>(h) * p.NR + row) * kCD + 4 * w)
                              : make_float4(0.f, 0.f, 0.f, 0.f);
        x[0] = v.x; x[1] = v.y; x[2] = v.z; x[3] = v.w;
      } else {
        if (live) {
          load8<DT>(p.qr, (static_cast<int64_t>(h) * p.NR + row) * kCD + 8 * w, x);
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e) x[e] = 0.0f;
        }
      }
#pragma unroll
      for (int e = 0; e < 16 / ESZ; ++e) qs[k][(16 / ESZ) * w + e] = x[e] * p.scaling;
    }
    if (threadIdx.x < 64)
      ws[threadIdx.x] = r0 + static_cast<int>(threadIdx.x) < re ? p.roww[static_cast<int64_t>(h) * p.NR + r0 + threadIdx.x] : 0.0f;
    __syncthreads();
    for (int k = 0; k < 64; ++k) {
      const float a = ws[k] * qs[k][c1];
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] = __builtin_fmaf(a, qs[k][c2 + e], acc[e]);
    }
  }
  float* dst = p.S_part + ((static_cast<int64_t>(sp) * p.Hkv + h) * kCD + c1) * kCD + c2;
#pragma unroll
  for (int e = 0; e < 8; ++e) dst[e] = acc[e];
}

__global__ __launch_bounds__(kCThreads) void cov_smat_sum(CovParams p) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * kCThreads + threadIdx.x;
  const int64_t total = static_cast<int64_t>(p.Hkv) * kCD * kCD;
  if (t >= total) return;
  float a = 0.0f;
#pragma unroll
  for (int sp = 0; sp < kSSplit; ++sp) a += p.S_part[sp * total + t];
  p.S[t] = a;
}

// finalisation sums: red[0..2] the means of the live-averaged A, DD, W; red[3] the live count;
// red[4 + h rep + r] omega (live-averaged read mass per query head); red[4 + Hkv rep + h] sum_j A
// (live-averaged).  First every per-head sum over the n tokens, one workgroup each (sums[h][0] A,
// [1] DD, [2 + r] the read mass of query head r: its blocks' weighted masses), then one thread combines them in a fixed order.
__global__ __launch_bounds__(1024) void cov_final_sums(CovParams p, const int32_t* rlist, int n_rlist) {
  __shared__ float part[16];
  const int nk = 2 + p.rep;
  const int h = blockIdx.x / nk, kind = blockIdx.x % nk;
  float v = 0.0f;
  if (kind < 2) {
    const float* src = (kind == 0 ? p.A : p.DD) + static_cast<int64_t>(h) * p.n;
    for (int j = threadIdx.x; j < p.n; j += 1024) v += src[j];
  } else {
    // every 16th row of the head's list starts a block (a block's first row is never padding)
    const int32_t* rl = rlist + static_cast<int64_t>(kind - 2) * n_rlist;
    for (int x = threadIdx.x; x < n_rlist / 4; x += 1024)
      v += p.omega[(static_cast<int64_t>(h) * (p.NR / 16) + rl[x / 4 * 16] / 16) * 4 + x % 4];
  }
  v = wave_sum(v);
  if (threadIdx.x % 64 == 0) part[threadIdx.x / 64] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    float t = 0.0f;
    for (int w = 0; w < 16; ++w) t += part[w];
    p.sums[blockIdx.x] = t;
  }
}

__global__ void cov_final_combine(CovParams p) {
  if (threadIdx.x != 0) return;
  float live = 0.0f;                                      // live groups, counted in group order
  for (int g = 0; g < p.G; ++g) live += p.gw[p.G + 1 + g];
  live = fmaxf(live, 1.0f);
  const int nk = 2 + p.rep;
  float gA = 0.0f, gD = 0.0f, gW = 0.0f;
  for (int h = 0; h < p.Hkv; ++h) {
    const float sA = p.sums[h * nk], sD = p.sums[h * nk + 1];
    float sW = 0.0f;
    for (int r = 0; r < p.rep; ++r) {
      const float om = p.sums[h * nk + 2 + r];
      p.red[4 + h * p.rep + r] = om / live;
      sW += om;
    }
    p.red[4 + p.Hkv * p.rep + h] = sA / live;
    gA += sA;
    gD += sD;
    gW += sW;
  }
  const float cnt = static_cast<float>(p.Hkv) * static_cast<float>(p.n);
  p.red[0] = gA / live / cnt;
  p.red[1] = gD / live / cnt;
  p.red[2] = gW / live / cnt;
  p.red[3] = live;
}

__global__ __launch_bounds__(kCThreads) void cov_final(CovParams p) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * kCThreads + threadIdx.x;
  const float live = p.red[3];
  const int64_t nA = static_cast<int64_t>(p.Hkv) * p.n;
  const int64_t nS = static_cast<int64_t>(p.Hkv) * kCD * kCD;
  if (t < nA) {
    p.A[t] = p.A[t] / live + p.eta * p.red[0];
    p.DD[t] = p.DD[t] / live + p.eta * p.red[1];
    p.W[t] = p.W[t] / live + p.eta * p.red[2];
  }
  if (t < nS) {
    const int h = static_cast<int>(t / (kCD * kCD)), e = static_cast<int>(t % (kCD * kCD));
    const float sA = p.red[4 + p.Hkv * p.rep + h];
    p.S[t] = p.S[t] / live / fmaxf(sA, 1e-30f);
    float om = 0.0f, acc = 0.0f, mean = 0.0f;
    for (int r = 0; r < p.rep; ++r) {
      const float o = p.red[4 + h * p.rep + r];
      const float mv = p.M[static_cast<int64_t>(h * p.rep + r) * kCD * kCD + e];
      om += o;
      acc = __builtin_fmaf(o, mv, acc);
      mean += mv;
    }
    p.Mbar[t] = om > 0.0f ? acc / om : mean / static_cast<float>(p.rep);
  }
}

}  // namespace
}  // namespace kvq

using namespace kvq;

// tokens whose per-group sums are stored at once: whole chunks, all of them up to kStoreFloats
static int64_t cov_store_tokens(int64_t Hkv, int64_t n, int64_t G) {
  const int64_t all = (n + kChunkTok - 1) / kChunkTok, fit = kStoreFloats / (3 * G * Hkv * kChunkTok);
  return std::max<int64_t>(1, std::min(all, fit)) * kChunkTok;
}

// workspace layout (floats): row_m, row_il, oMo, roww (Hkv NR each), omega (Hkv NR / 4); o (Hkv NR d); o_part (kOSplit Hkv
// NR d); vmv (Hkv rep n); ddpart (G Hkv n_chunks kTW); gw (2 G + 1); red (4 + Hkv rep + Hkv); tsum (G Hkv 3
// store tokens); row_part (Hkv n_chunks NR / 16 kRowPart), rec (Hkv NR / 16 records, fp32's the larger
// ones), 16-byte aligned; S_part (kSSplit Hkv d d); sums (Hkv (2 + rep));
// fp32 rows: partial maxima and scales (kAmaxFloats)
extern "C" int64_t kvq_coverage_stats_workspace(int64_t Hkv, int64_t rep, int64_t n, int64_t NR, int64_t G) {
  if (Hkv <= 0 || rep <= 0 || n <= 0 || NR <= 0 || G <= 0) return -1;
  const int64_t nch = (n + kChunkTok - 1) / kChunkTok;
  return 4 * Hkv * NR + Hkv * (NR / 4) + (1 + kOSplit) * Hkv * NR * kCD + Hkv * rep * n + G * Hkv * nch * kTW + Hkv * nch * (NR / 16) * kRowPart +
         (2 * G + 1) + (4 + Hkv * rep + Hkv) + G * Hkv * 3 * cov_store_tokens(Hkv, n, G) +
         Hkv * (NR / 16) * rec_units<KVQ_F32>() * 4 + 4 + kSSplit * Hkv * kCD * kCD + Hkv * (2 + rep) + kAmaxFloats;
}

extern "C" int kvq_coverage_stats(const void* qr, int dtype, int64_t NR, const int32_t* rowpos, const int32_t* rowgrp,
                                  const int32_t* rlist, int64_t n_rlist, const int32_t* gtab, int64_t G,
                                  const int32_t* items, int64_t n_items, const void* k, int64_t k_sh, int64_t k_st,
                                  const void* v, int64_t v_sh, int64_t v_st, int64_t T, const float* M, int64_t Hkv,
                                  int64_t rep, int64_t d, int64_t rs, int64_t re, float scaling, float eta, float* A,
                                  float* W, float* DD, float* S, float* Mbar, float* workspace,
                                  int64_t workspace_floats, void* stream) {
  KVQ_REQUIRE(valid_dtype(dtype), "kvq_coverage_stats: bad dtype");
  KVQ_REQUIRE(d == kCD, "kvq_coverage_stats: head_dim must be 128");
  KVQ_REQUIRE(Hkv > 0 && rep > 0 && Hkv * rep <= 1024, "kvq_coverage_stats: bad head counts");
  KVQ_REQUIRE(0 <= rs && rs < re && re <= T && T < (1 << 28), "kvq_coverage_stats: need 0 <= rs < re <= T");
  KVQ_REQUIRE(G > 0 && n_items > 0 && NR > 0 && NR % 16 == 0 && Hkv * NR < (1LL << 31) / kCD && n_rlist > 0 &&
                  n_rlist * rep <= NR,
              "kvq_coverage_stats: bad group plan");
  KVQ_REQUIRE(qr && rowpos && rowgrp && rlist && gtab && items && k && v && M && A && W && DD && S && Mbar && workspace,
              "kvq_coverage_stats: null pointer");
  const int esz = dtype == KVQ_F32 ? 4 : 2;
  KVQ_REQUIRE((k_sh * esz) % 16 == 0 && (k_st * esz) % 16 == 0 && (v_sh * esz) % 16 == 0 && (v_st * esz) % 16 == 0 &&
                  reinterpret_cast<uintptr_t>(k) % 16 == 0 && reinterpret_cast<uintptr_t>(v) % 16 == 0 &&
                  reinterpret_cast<uintptr_t>(qr) % 16 == 0 && reinterpret_cast<uintptr_t>(workspace) % 16 == 0 &&
                  reinterpret_cast<uintptr_t>(M) % 16 == 0 && k_st >= kCD && v_st >= kCD,
              "kvq_coverage_stats: rows must be 16-byte aligned and not overlap");
  KVQ_REQUIRE((T + 48) * std::max(k_st, v_st) * esz < (1LL << 31), "kvq_coverage_stats: one head's rows must span < 2 GiB");
  const int64_t n = re - rs;
  const int64_t need = kvq_coverage_stats_workspace(Hkv, rep, n, NR, G);
  KVQ_REQUIRE(workspace_floats >= need, "kvq_coverage_stats: workspace too small (%lld < %lld floats)",
              (long long)workspace_floats, (long long)need);
  CovParams p{};
  p.qr = qr; p.rowpos = rowpos; p.gtab = gtab; p.items = items;
  p.k = k; p.v = v; p.k_sh = k_sh; p.k_st = k_st; p.v_sh = v_sh; p.v_st = v_st;
  p.M = M;
  p.Hkv = (int)Hkv; p.rep = (int)rep; p.NR = (int)NR; p.G = (int)G; p.n_items = (int)n_items;
  p.rs = (int)rs; p.re = (int)re; p.n = (int)n; p.n_chunks = (int)((n + kChunkTok - 1) / kChunkTok); p.T = (int)T;
  p.scaling = scaling; p.qscale = scaling * kCLog2e; p.eta = eta;
  float* w = workspace;
  p.row_m = w; w += Hkv * NR;
  p.row_il = w; w += Hkv * NR;
  p.oMo = w; w += Hkv * NR;
  p.roww = w; w += Hkv * NR;
  p.omega = w; w += Hkv * (NR / 4);
  p.o = w; w += Hkv * NR * kCD;
  p.o_part = w; w += kOSplit * Hkv * NR * kCD;
  p.vmv = w; w += Hkv * rep * n;
  p.ddpart = w; w += G * Hkv * p.n_chunks * kTW;
  p.gw = w; w += 2 * G + 1;
  p.red = w; w += 4 + Hkv * rep + Hkv;
  const int64_t store_tokens = cov_store_tokens(Hkv, n, G);
  p.tsum = w; w += G * Hkv * 3 * store_tokens;
  w += (4 - (reinterpret_cast<uintptr_t>(w) / 4) % 4) % 4;       // 16-byte alignment
  p.row_part = w; w += Hkv * p.n_chunks * (NR / 16) * kRowPart;
  p.rec = reinterpret_cast<uint32_t*>(w); w += Hkv * (NR / 16) * rec_units<KVQ_F32>() * 4;
  p.S_part = w; w += kSSplit * Hkv * kCD * kCD;
  p.sums = w; w += Hkv * (2 + rep);
  float* amax_part = w;                                       // fp32 rows: partial maxima, then scales
  p.xs = dtype == KVQ_F32 ? w + kAmaxViews * kAmaxBlocks : nullptr;
  p.A = A; p.W = W; p.DD = DD; p.S = S; p.Mbar = Mbar;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const dim3 blk(kCThreads);
  if (dtype == KVQ_F32) {
    // the powers of two that bring the query rows, keys and values into the fp16 parts' range
    const RowView views[3] = {
        RowView{static_cast<const float*>(qr), static_cast<int>(Hkv), static_cast<int>(NR), 1, NR * kCD, kCD, 0},
        RowView{static_cast<const float*>(k), static_cast<int>(Hkv), static_cast<int>(T), 1, k_sh, k_st, 0},
        RowView{static_cast<const float*>(v), static_cast<int>(Hkv), static_cast<int>(T), 1, v_sh, v_st, 0}};
    launch_rows_scales(views, 3, amax_part, const_cast<float*>(p.xs), s);
    KVQ_LAUNCH_CHECK("kvq_coverage_stats(fp32 scales)");
  }
  KVQ_DISPATCH_DTYPE(dtype, hipLaunchKernelGGL((cov_rowstats<DT_>), dim3(xcd_grid(n_items * Hkv)),
                                               dim3(DT_ == KVQ_F32 ? kCThreads : 2 * kCThreads), 0, s, p));
  KVQ_LAUNCH_CHECK("kvq_coverage_stats(rowstats)");
  KVQ_DISPATCH_DTYPE(dtype, hipLaunchKernelGGL((cov_output<DT_>), dim3(xcd_grid(n_items * Hkv * kOSplit)), blk, 0, s, p));
  KVQ_LAUNCH_CHECK("kvq_coverage_stats(output)");
  hipLaunchKernelGGL((cov_metric<KVQ_F32, true>), dim3(Hkv * rep * ((n_rlist + kMetricRows - 1) / kMetricRows)), blk,
                     0, s, p, rlist, (int)n_rlist);
  KVQ_LAUNCH_CHECK("kvq_coverage_stats(o M)");
  KVQ_DISPATCH_DTYPE(dtype, hipLaunchKernelGGL((cov_vmv<DT_>),
                                               dim3(Hkv * rep * ((n + kVmvPer - 1) / kVmvPer)), blk, 0, s, p));
  KVQ_LAUNCH_CHECK("kvq_coverage_stats(v M v)");
  KVQ_DISPATCH_DTYPE(dtype, hipLaunchKernelGGL((cov_rowprep<DT_>), dim3(Hkv * (NR / 16)), blk, 0, s, p, rowgrp));
  KVQ_LAUNCH_CHECK("kvq_coverage_stats(row records)");
  // the terms of every chunk, the sums of the first store_tokens tokens kept; then, where the store
  // holds no more, the further ranges' terms again, each read by cov_wsum before the next
  const int range_chunks = static_cast<int>(store_tokens / kChunkTok);
  for (int c = 0; c < p.n_chunks; c += range_chunks) {
    const bool first = c == 0;
    TermsRange R{c, first ? p.n_chunks : std::min(range_chunks, p.n_chunks - c), p.rs + c * kChunkTok,
                 static_cast<int>(store_tokens), 1, first};
    // a workgroup's start (its key and value tiles, the first record) costs about a block's time, so the
    // groups of a chunk are cut into pieces only while the chip holds more workgroups (three per CU, two
    // rounds, since the chunks' work differs): 8 heads x 32768 tokens, 4 pieces 763 us, 2 pieces 702, 1 705
    while (R.pieces < 8 && Hkv * R.chunks * R.pieces < kTermsUnits) R.pieces *= 2;
    KVQ_DISPATCH_DTYPE(dtype, hipLaunchKernelGGL((cov_terms<DT_>), dim3(xcd_grid(Hkv * R.chunks * R.pieces)), dim3(64 * kTW),
                                                 0, s, p, R));
    KVQ_LAUNCH_CHECK("kvq_coverage_stats(terms)");
    if (first) {
      hipLaunchKernelGGL(cov_groups, dim3(static_cast<unsigned>(G)), blk, 0, s, p);
      KVQ_LAUNCH_CHECK("kvq_coverage_stats(groups)");
      hipLaunchKernelGGL(cov_roww, dim3((Hkv * (NR / 16) * kRowPart + 63) / 64), blk, 0, s, p, rowgrp);
      KVQ_LAUNCH_CHECK("kvq_coverage_stats(row weights)");
    }
    hipLaunchKernelGGL(cov_wsum, dim3(Hkv * ((store_tokens + kCThreads - 1) / kCThreads)), blk, 0, s, p, R.store0, R.store_n);
    KVQ_LAUNCH_CHECK("kvq_coverage_stats(weighted sums)");
  }
  KVQ_DISPATCH_DTYPE(dtype, hipLaunchKernelGGL((cov_smat<DT_>), dim3(Hkv * (kCD / 16) * kSSplit), blk, 0, s, p));
  KVQ_LAUNCH_CHECK("kvq_coverage_stats(S parts)");
  hipLaunchKernelGGL(cov_smat_sum, dim3((Hkv * kCD * kCD + kCThreads - 1) / kCThreads), blk, 0, s, p);
  KVQ_LAUNCH_CHECK("kvq_coverage_stats(S)");
  hipLaunchKernelGGL(cov_final_sums, dim3(static_cast<unsigned>(Hkv * (2 + rep))), dim3(1024), 0, s, p, rlist, (int)n_rlist);
  KVQ_LAUNCH_CHECK("kvq_coverage_stats(sums)");
  hipLaunchKernelGGL(cov_final_combine, dim3(1), dim3(64), 0, s, p);
  KVQ_LAUNCH_CHECK("kvq_coverage_stats(combine)");
  const int64_t nmax = std::max<int64_t>(Hkv * n, Hkv * kCD * kCD);
  hipLaunchKernelGGL(cov_final, dim3((nmax + kCThreads - 1) / kCThreads), blk, 0, s, p);
  KVQ_LAUNCH_CHECK("kvq_coverage_stats(final)");
  return KVQ_OK;
}
