// SnapKV scores on the device (gfx950): the eviction scores of STRATA_KV.py:932-954 (snapkv_scores).
//
// What it computes, per (b, KV head h): the last `w` context queries of each of the rep query heads
// of h (rows r = (head, i), position H - w + i) attend causally to the keys [0, H) (fp32 softmax of
// scaling * q.k); the probabilities of the keys j < H - w are averaged over the rep * w rows
// (mean over the window queries, then over the heads of the group), pooled along j by
// avg_pool1d(kernel, padding kernel / 2, zeros counted), and the w window columns get the global
// maximum + 1.  Output (B, Hkv, H) float32.  Means over rows and pooling along keys are linear along
// different axes, so they are taken in the order that needs one column sum per key.
//
// Passes (one stream, no host synchronisation):
//   1. snap_stats: per (bh, row group, key split) the logits of the group's rows against the split's
//      keys on the matrix cores (v_mfma_f32_16x16x32_{bf16,f16}; fp32 inputs as fp16 hi + lo parts,
//      three products), each lane keeping an online (max, sum) of its rows in base 2; partials out.
//   2. snap_rows: each row's (max, 1 / sum) from the partials.
//   3. snap_cols: per (bh, row group, key split) the logits again, probabilities normalised by the
//      row statistics and summed over the group's rows on the way out of the accumulators.
//   4. snap_pool: sum of the row groups' column sums / (rep * w), the pooling window through LDS,
//      and a maximum per block.
//   5. snap_window: the global maximum + 1 into the w window columns.
// Matrix-core mapping (mfma_common.hpp): A = 16 keys x 32 channels (lane l: key l%16, channels
// 8(l/16)..+7 of the k-step), B = 32 channels x 16 query rows, D lane l register i = logit of key
// 4(l/16) + i for row l%16.
//
// Both logit passes stream their split's keys through LDS (KeyStream): the four wavefronts of a workgroup hold
// the operands of 64 rows each and share every key.  What bounds them: the exp2 of every (row, key)
// pair at a quarter of the vector rate and the products themselves (at 4 x 8 x 65536 bf16 keys and 256 rows
// each, 137 GFLOP and 0.54 GB a pass: statistics 154 us, columns 153 (153 and 152 at best in a trace, 164 and
// 161 on average over 150 passes), 131 without the exponentials; a large
// library product reaches 1.26 PFLOP/s here, which is 109 us).  With each wavefront loading its tiles from
// L2, one ahead, they took 242 and 288.  Eight wavefronts of 32 rows 153 and 157, stages of 128 keys 163
// and 161.
#include <algorithm>

#include "common.hpp"
#include "mfma_common.hpp"
#include "row_tiles.hpp"

namespace kvq {
namespace {

constexpr int kSnapThreads = 256;     // workgroups of the row, pooling and window passes
constexpr int kSnapWaves = 4;
constexpr int kLogitWaves = 4;        // wavefronts of a logit workgroup
constexpr int kLogitThreads = 64 * kLogitWaves;
constexpr int kSnapResident = 2;       // workgroups of a logit pass resident on a CU
constexpr int kSnapPool = 1024;       // keys of a pooling workgroup
constexpr int kSnapMaxPad = 32;       // largest pooling half-width
constexpr float kSnapLog2e = 1.4426950408889634f;

template <int DT>
struct SnapTraits {
  static constexpr int NH = TileOps<DT>::NH;                // operand parts (fp32: fp16 hi, lo)
  static constexpr int NBW = DT == KVQ_F32 ? 2 : 4;         // row blocks of 16 per wavefront
  static constexpr int RG = 16 * NBW * kLogitWaves;         // rows per workgroup
  static constexpr int ESZ = TileOps<DT>::ESZ;
  static constexpr int KT = 64 / NH;                        // keys of a stage
};

struct SnapParams {
  const void* q;
  int64_t q_sb, q_sh, q_st;             // window query rows: (b, head, i) at b*q_sb + head*q_sh + i*q_st
  const void* k;
  int64_t k_sb, k_sh, k_st;             // keys: (b, h, j) at b*k_sb + h*k_sh + j*k_st
  int BH, Hkv, rep, w, H, rows, n_rg, n_split, split_keys, n_pool, kernel;
  float qscale;                         // scaling * log2(e)
  float inv_count;                      // 1 / (rep * w)
  float* part_m;                        // (BH, rows, n_split)
  float* part_l;
  float* row_m;                         // (BH, rows)
  float* row_il;                        // (BH, rows): 1 / row sum
  float* colsum;                        // (BH, n_rg, H - w)
  float* blockmax;                      // (BH, n_pool)
  float* out;                           // (BH, H)
  // fp32 rows: the powers of two of the query rows and the keys (rows_scale_kernel, row_tiles.hpp)
  const float* xs;
};

// the power of two of fp32 view i (0: query rows, 1: keys); 16-bit rows are exact operands: 1
template <int DT>
__device__ __forceinline__ float snap_xs(const SnapParams& p, int i) {
  if constexpr (DT == KVQ_F32) return p.xs[i];
  else return 1.0f;
}

// query operands of this wavefront's row blocks and the position of each lane's row (-1: no row)
template <int DT>
__device__ __forceinline__ void load_queries(const SnapParams& p, int b, int h, int rg, int wave, int g, int n,
                                             u32x4 (&qop)[SnapTraits<DT>::NBW][4][SnapTraits<DT>::NH],
                                             int (&rowpos)[SnapTraits<DT>::NBW], int (&row)[SnapTraits<DT>::NBW]) {
  using T = SnapTraits<DT>;
#pragma unroll
  for (int bw = 0; bw < T::NBW; ++bw) {
    const int r = rg * T::RG + (wave * T::NBW + bw) * 16 + n;
    row[bw] = r;
    if (r < p.rows) {
      const int hq = h * p.rep + r / p.w, i = r % p.w;
      const int64_t base = static_cast<int64_t>(b) * p.q_sb + static_cast<int64_t>(hq) * p.q_sh +
                           static_cast<int64_t>(i) * p.q_st;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) load_op<DT>(p.q, base + 32 * ks + 8 * g, qop[bw][ks], snap_xs<DT>(p, 0));
      rowpos[bw] = p.H - p.w + i;
    } else {
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
#pragma unroll
        for (int hh = 0; hh < T::NH; ++hh) qop[bw][ks][hh] = u32x4{0u, 0u, 0u, 0u};
      rowpos[bw] = -1;
    }
  }
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t key_rsrc(const SnapParams& p, int b, int h, int esz) {
  const char* base = static_cast<const char*>(p.k) +
                     (static_cast<int64_t>(b) * p.k_sb + static_cast<int64_t>(h) * p.k_sh) * esz;
  return make_rsrc(base, static_cast<uint32_t>((static_cast<int64_t>(p.H - 1) * p.k_st + 128) * esz));
}

// The keys of a split in stages of KT, double-buffered in LDS: the loads of a stage go out two stages before
// it is computed (into registers, so that they wait for nothing else), and each 16-byte piece (8
// channels of a key, converted to operand parts where the keys are fp32) is written to LDS once for
// the four wavefronts.  Piece c of key j lies at column c ^ (j % 16) of its row, which puts the 16 keys of
// an operand read on different banks.  Keys past H repeat the last one (their logits are masked).
template <int DT>
struct KeyStream {
  using T = SnapTraits<DT>;
  static constexpr int UNITS = T::KT * 16 / kLogitThreads;   // pieces of a thread and stage
  u32x4 (*lds)[T::NH][T::KT * 16];                          // [2][NH][KT 16]
  __amdgpu_buffer_rsrc_t rk;
  int64_t st;
  int last;                                                 // H - 1
  float xs;
  u32x4 reg[2][UNITS][T::NH];                               // 8 channels: 16 bytes, or 32 of fp32

  __device__ __forceinline__ void load(int k0, u32x4 (&r)[UNITS][T::NH]) {
#pragma unroll
    for (int u = 0; u < UNITS; ++u) {
      const int id = threadIdx.x + kLogitThreads * u;
      const int off = static_cast<int>((min(k0 + id / 16, last) * st + 8 * (id % 16)) * T::ESZ);
#pragma unroll
      for (int e = 0; e < T::NH; ++e) r[u][e] = __builtin_amdgcn_raw_buffer_load_b128(rk, off + 16 * e, 0, 0);
    }
  }
  __device__ __forceinline__ void store(int buf, const u32x4 (&r)[UNITS][T::NH]) {
#pragma unroll
    for (int u = 0; u < UNITS; ++u) {
      const int id = threadIdx.x + kLogitThreads * u;
      const int at = (id / 16) * 16 + ((id % 16) ^ (id / 16 % 16));
      if constexpr (DT == KVQ_F32) {
        float x[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) x[k] = __uint_as_float(r[u][k / 4][k % 4]) * xs;
        u32x4 hi, lo;
        f32_parts<DT>(x, hi, lo);
        lds[buf][0][at] = hi;
        lds[buf][1][at] = lo;
      } else {
        lds[buf][0][at] = r[u][0];
      }
    }
  }
  // the operand of the 16 keys from 16 tt of the stage in buf
  __device__ __forceinline__ void operand(int buf, int tt, int g, int n, u32x4 (&kop)[4][T::NH]) const {
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int hh = 0; hh < T::NH; ++hh) kop[ks][hh] = lds[buf][hh][(16 * tt + n) * 16 + ((4 * ks + g) ^ n)];
  }
  // stage(k, buf) for every stage of [k0, k1), its keys in LDS buffer buf; a barrier lies before each call
  template <class F>
  __device__ __forceinline__ void run(int k0, int k1, F stage) {
    load(k0, reg[0]);
    load(k0 + T::KT, reg[1]);
    store(0, reg[0]);
    block_lds_barrier();
    for (int k = k0; k < k1; k += 2 * T::KT) {
      load(k + 2 * T::KT, reg[0]);
      stage(k, 0);
      store(1, reg[1]);
      block_lds_barrier();
      if (k + T::KT >= k1) break;
      load(k + 3 * T::KT, reg[1]);
      stage(k + T::KT, 1);
      store(0, reg[0]);
      block_lds_barrier();
    }
  }
};

// (bh, row group, split) of a workgroup: the row groups of one split go to one XCD, which reads its keys once
__device__ __forceinline__ bool snap_unit(const SnapParams& p, int* bh, int* rg, int* s) {
  const int k = blockIdx.x / 8;
  const int unit = (k / p.n_rg) * 8 + blockIdx.x % 8;
  *rg = k % p.n_rg;
  *bh = unit / p.n_split;
  *s = unit % p.n_split;
  return *bh < p.BH;
}

constexpr float kSnapNone = -3.0e38f;   // no logit yet (finite, so that a first logit of -inf stays a zero term)
constexpr float kSnapLazy = 8.0f;       // a row's reference is moved when a logit exceeds it by this many octaves

template <int DT>
__global__ __launch_bounds__(kLogitThreads, 2) void snap_stats(SnapParams p) {
  using T = SnapTraits<DT>;
  __shared__ u32x4 keys[2][T::NH][T::KT * 16];
  const int wave = threadIdx.x / 64, l = threadIdx.x % 64, g = l >> 4, n = l & 15;
  int bh, rg, s;
  if (!snap_unit(p, &bh, &rg, &s)) return;
  const int b = bh / p.Hkv, h = bh % p.Hkv;
  u32x4 qop[T::NBW][4][T::NH];
  int rowpos[T::NBW], row[T::NBW];
  load_queries<DT>(p, b, h, rg, wave, g, n, qop, rowpos, row);
  float m[T::NBW], ls[T::NBW];
#pragma unroll
  for (int bw = 0; bw < T::NBW; ++bw) {
    m[bw] = kSnapNone;
    ls[bw] = 0.0f;
  }
  const int k0 = s * p.split_keys, k1 = min(k0 + p.split_keys, p.H);
  const int open = min(k1, p.H - p.w + 1);     // keys below it are in the split and visible to every row
  const float qsc = p.qscale / (snap_xs<DT>(p, 0) * snap_xs<DT>(p, 1));   // logit scale of the scaled rows
  KeyStream<DT> ks{keys, key_rsrc(p, b, h, T::ESZ), p.k_st, p.H - 1, snap_xs<DT>(p, 1)};
  ks.run(k0, k1, [&](int k, int buf) {
#pragma unroll
    for (int tt = 0; tt < T::KT / 16; ++tt) {
      const int t0 = k + 16 * tt;
      if (t0 >= k1) break;
      u32x4 kop[4][T::NH];
      ks.operand(buf, tt, g, n, kop);
      f32x4 acc[T::NBW];
#pragma unroll
      for (int bw = 0; bw < T::NBW; ++bw) acc[bw] = tile_dots<DT, T::NH, T::NH>(kop, qop[bw]);
      const bool edge = t0 + 16 > open;        // the split's end, or keys that some rows do not see
      const float f = edge ? 1.0f : qsc;       // logit = f acc
      if (edge) {
#pragma unroll
        for (int bw = 0; bw < T::NBW; ++bw)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int j = t0 + 4 * g + i;
            acc[bw][i] = (j < k1 && j <= rowpos[bw]) ? acc[bw][i] * qsc : -INFINITY;
          }
      }
#pragma unroll
      for (int bw = 0; bw < T::NBW; ++bw) {
        float a[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) a[i] = __builtin_fmaf(acc[bw][i], f, -m[bw]);
        const float top = fmaxf(fmaxf(a[0], a[1]), fmaxf(a[2], a[3]));
        if (__any(top > kSnapLazy)) {
          const float mn = fmaxf(m[bw], fmaxf(fmaxf(acc[bw][0] * f, acc[bw][1] * f), fmaxf(acc[bw][2] * f, acc[bw][3] * f)));
          ls[bw] *= __builtin_amdgcn_exp2f(m[bw] - mn);
          m[bw] = mn;
#pragma unroll
          for (int i = 0; i < 4; ++i) a[i] = __builtin_fmaf(acc[bw][i], f, -mn);
        }
        ls[bw] += (__builtin_amdgcn_exp2f(a[0]) + __builtin_amdgcn_exp2f(a[1])) +
                  (__builtin_amdgcn_exp2f(a[2]) + __builtin_amdgcn_exp2f(a[3]));
      }
    }
  });
  // the four lanes of a row (xor 16, xor 32) hold disjoint keys of it
#pragma unroll
  for (int bw = 0; bw < T::NBW; ++bw) {
    const float M = xmax32(xmax16(m[bw]));
    const float L = xsum32(xsum16(ls[bw] * __builtin_amdgcn_exp2f(m[bw] - M)));
    if (g == 0 && row[bw] < p.rows) {
      const int64_t o = (static_cast<int64_t>(bh) * p.rows + row[bw]) * p.n_split + s;
      p.part_m[o] = M;
      p.part_l[o] = L;
    }
  }
}

// 16 lanes a row, each over every 16th split
__global__ __launch_bounds__(kSnapThreads) void snap_rows(SnapParams p, int64_t n_rows_all) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * (kSnapThreads / 16) + threadIdx.x / 16;
  const int lane = threadIdx.x % 16;
  const int64_t at = (t < n_rows_all ? t : n_rows_all - 1) * p.n_split;
  float M = kSnapNone;
  for (int s = lane; s < p.n_split; s += 16) M = fmaxf(M, p.part_m[at + s]);
  M = row_max16(M);
  float L = 0.0f;
  for (int s = lane; s < p.n_split; s += 16) L += p.part_l[at + s] * __builtin_amdgcn_exp2f(p.part_m[at + s] - M);
  L = row_sum16(L);
  if (lane == 0 && t < n_rows_all) {
    p.row_m[t] = M;
    p.row_il[t] = 1.0f / L;               // key 0 is visible to every row: L > 0
  }
}

template <int DT>
__global__ __launch_bounds__(kLogitThreads, 2) void snap_cols(SnapParams p) {
  using T = SnapTraits<DT>;
  __shared__ u32x4 keys[2][T::NH][T::KT * 16];
  __shared__ float cols[2][kLogitWaves][T::KT];
  const int wave = threadIdx.x / 64, l = threadIdx.x % 64, g = l >> 4, n = l & 15;
  int bh, rg, s;
  if (!snap_unit(p, &bh, &rg, &s)) return;
  const int b = bh / p.Hkv, h = bh % p.Hkv;
  u32x4 qop[T::NBW][4][T::NH];
  int rowpos[T::NBW], row[T::NBW];
  load_queries<DT>(p, b, h, rg, wave, g, n, qop, rowpos, row);
  // operand roles swapped against snap_stats (A = query rows, B = keys): D lane (g, n) register i
  // is the logit of row 16 (wave NBW + bw) + 4 g + i against key t0 + n, so a column sum over the
  // wavefront's rows is a register sum and two cross-lane steps per tile.  Row statistics per
  // register: the rows of lane group g.
  float rm[T::NBW][4], ril[T::NBW][4];
#pragma unroll
  for (int bw = 0; bw < T::NBW; ++bw) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = rg * T::RG + (wave * T::NBW + bw) * 16 + 4 * g + i;
      const bool ok = r < p.rows;
      rm[bw][i] = ok ? p.row_m[static_cast<int64_t>(bh) * p.rows + r] : 0.0f;
      ril[bw][i] = ok ? p.row_il[static_cast<int64_t>(bh) * p.rows + r] : 0.0f;
    }
  }
  const int nc = p.H - p.w;                 // scored keys: every window row sees all of them
  const int k0 = s * p.split_keys, k1 = min(k0 + p.split_keys, nc);
  const float qsc = p.qscale / (snap_xs<DT>(p, 0) * snap_xs<DT>(p, 1));   // logit scale of the scaled rows
  float* const dst = p.colsum + (static_cast<int64_t>(bh) * p.n_rg + rg) * nc;
  // the wavefronts' sums of a stage meet behind the next barrier
  auto flush = [&](int k, int buf) {
    if (threadIdx.x < T::KT && k + static_cast<int>(threadIdx.x) < k1) {
      const int t = threadIdx.x;
      dst[k + t] = (cols[buf][0][t] + cols[buf][1][t]) + (cols[buf][2][t] + cols[buf][3][t]);
    }
  };
  if (k0 >= k1) return;
  KeyStream<DT> ks{keys, key_rsrc(p, b, h, T::ESZ), p.k_st, p.H - 1, snap_xs<DT>(p, 1)};
  int done = -1, done_buf = 0;
  ks.run(k0, k1, [&](int k, int buf) {
    if (done >= 0) flush(done, done_buf);
#pragma unroll
    for (int tt = 0; tt < T::KT / 16; ++tt) {
      if (k + 16 * tt >= k1) break;
      u32x4 kop[4][T::NH];
      ks.operand(buf, tt, g, n, kop);
      f32x4 acc[T::NBW];
#pragma unroll
      for (int bw = 0; bw < T::NBW; ++bw) acc[bw] = tile_dots<DT, T::NH, T::NH>(qop[bw], kop);
      float colv[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int bw = 0; bw < T::NBW; ++bw)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          colv[i] = __builtin_fmaf(__builtin_amdgcn_exp2f(__builtin_fmaf(acc[bw][i], qsc, -rm[bw][i])), ril[bw][i], colv[i]);
      // the four lane groups hold disjoint rows of key t0 + n
      const float v = xsum32(xsum16((colv[0] + colv[1]) + (colv[2] + colv[3])));
      if (g == 0) cols[buf][wave][16 * tt + n] = v;
    }
    done = k;
    done_buf = buf;
  });
  flush(done, done_buf);                    // run() ends behind a barrier
}

__global__ __launch_bounds__(kSnapThreads) void snap_pool(SnapParams p) {
  __shared__ float sc[kSnapPool + 2 * kSnapMaxPad];
  __shared__ float red[kSnapWaves];
  const int bh = blockIdx.x / p.n_pool, pc = blockIdx.x % p.n_pool;
  const int nc = p.H - p.w;
  const int pad = p.kernel / 2;
  const int j0 = pc * kSnapPool;
  const float* cs = p.colsum + static_cast<int64_t>(bh) * p.n_rg * nc;
  // mean probability of keys j0 - pad .. j0 + kSnapPool + pad (zero outside [0, nc))
  for (int t = threadIdx.x; t < kSnapPool + 2 * pad; t += kSnapThreads) {
    const int j = j0 - pad + t;
    float v = 0.0f;
    if (j >= 0 && j < nc) {
      for (int r = 0; r < p.n_rg; ++r) v += cs[static_cast<int64_t>(r) * nc + j];
      v *= p.inv_count;
    }
    sc[t] = v;
  }
  __syncthreads();
  const float inv_k = 1.0f / static_cast<float>(p.kernel);
  float mx = -INFINITY;
  for (int t = threadIdx.x; t < kSnapPool; t += kSnapThreads) {
    const int j = j0 + t;
    if (j < nc) {
      float v = 0.0f;
      for (int e = 0; e < p.kernel; ++e) v += sc[t + e];
      v *= inv_k;
      p.out[static_cast<int64_t>(bh) * p.H + j] = v;
      mx = fmaxf(mx, v);
    }
  }
  mx = wave_max(mx);
  if (threadIdx.x % 64 == 0) red[threadIdx.x / 64] = mx;
  __syncthreads();
  if (threadIdx.x == 0)
    p.blockmax[blockIdx.x] = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

__global__ __launch_bounds__(kSnapThreads) void snap_window(SnapParams p, int n_blocks) {
  __shared__ float red[kSnapWaves];
  float mx = -INFINITY;
  for (int t = threadIdx.x; t < n_blocks; t += kSnapThreads) mx = fmaxf(mx, p.blockmax[t]);
  mx = wave_max(mx);
  if (threadIdx.x % 64 == 0) red[threadIdx.x / 64] = mx;
  __syncthreads();
  const float top = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3])) + 1.0f;
  for (int t = threadIdx.x; t < p.w; t += kSnapThreads)
    p.out[static_cast<int64_t>(blockIdx.x) * p.H + (p.H - p.w) + t] = top;
}

struct SnapPlan {
  int n_rg, n_split, split_keys, n_pool;
};

SnapPlan snap_plan(int64_t BH, int64_t rows, int64_t w, int64_t H, int dtype) {
  SnapPlan sp{};
  const int64_t RG = dtype == KVQ_F32 ? SnapTraits<KVQ_F32>::RG : SnapTraits<KVQ_BF16>::RG;
  const int64_t KT = dtype == KVQ_F32 ? SnapTraits<KVQ_F32>::KT : SnapTraits<KVQ_BF16>::KT;
  sp.n_rg = static_cast<int>((rows + RG - 1) / RG);
  // one round of resident workgroups (kSnapResident a CU) of key splits, whole stages
  const int64_t want = std::max<int64_t>(1, 256 * kSnapResident / (BH * sp.n_rg));
  const int64_t stages = (H + KT - 1) / KT;
  const int64_t ns = std::min<int64_t>(want, stages);
  sp.split_keys = static_cast<int>(((stages + ns - 1) / ns) * KT);
  sp.n_split = static_cast<int>((H + sp.split_keys - 1) / sp.split_keys);
  sp.n_pool = static_cast<int>((H - w + kSnapPool - 1) / kSnapPool);
  return sp;
}

int64_t snap_ws(int64_t BH, int64_t rows, int64_t w, int64_t H, const SnapPlan& sp, int dtype) {
  return 2 * BH * sp.n_split * rows + 2 * BH * rows + BH * sp.n_rg * (H - w) + BH * sp.n_pool +
         (dtype == KVQ_F32 ? kAmaxFloats : 0);
}

}  // namespace
}  // namespace kvq

using namespace kvq;

extern "C" int64_t kvq_snapkv_scores_workspace(int64_t B, int64_t Hq, int64_t Hkv, int64_t window, int64_t H,
                                               int dtype) {
  if (B <= 0 || Hkv <= 0 || Hq % Hkv != 0 || window <= 0 || H <= window || !valid_dtype(dtype)) return -1;
  const int64_t rows = (Hq / Hkv) * window;
  const SnapPlan sp = snap_plan(B * Hkv, rows, window, H, dtype);
  return snap_ws(B * Hkv, rows, window, H, sp, dtype);
}

extern "C" int kvq_snapkv_scores(const void* q, int dtype, int64_t q_sb, int64_t q_sh, int64_t q_st, const void* k,
                                 int64_t k_sb, int64_t k_sh, int64_t k_st, int64_t B, int64_t Hq, int64_t Hkv,
                                 int64_t d, int64_t window, int64_t H, float scaling, int kernel, float* out,
                                 float* workspace, int64_t workspace_floats, void* stream) {
  KVQ_REQUIRE(valid_dtype(dtype), "kvq_snapkv_scores: bad dtype");
  KVQ_REQUIRE(d == 128, "kvq_snapkv_scores: head_dim must be 128");
  KVQ_REQUIRE(B > 0 && Hkv > 0 && Hq % Hkv == 0 && B * Hkv < 65536, "kvq_snapkv_scores: bad head counts");
  KVQ_REQUIRE(window > 0 && H > window && H < (1LL << 28), "kvq_snapkv_scores: need 0 < window < H");
  KVQ_REQUIRE(kernel >= 1 && kernel % 2 == 1 && kernel / 2 <= kSnapMaxPad,
              "kvq_snapkv_scores: pooling kernel must be odd and at most %d", 2 * kSnapMaxPad + 1);
  KVQ_REQUIRE(q && k && out && workspace, "kvq_snapkv_scores: null pointer");
  const int esz = dtype == KVQ_F32 ? 4 : 2;
  KVQ_REQUIRE((q_sb * esz) % 16 == 0 && (q_sh * esz) % 16 == 0 && (q_st * esz) % 16 == 0 &&
                  reinterpret_cast<uintptr_t>(q) % 16 == 0,
              "kvq_snapkv_scores: query rows must be 16-byte aligned");
  KVQ_REQUIRE((k_sb * esz) % 16 == 0 && (k_sh * esz) % 16 == 0 && (k_st * esz) % 16 == 0 &&
                  reinterpret_cast<uintptr_t>(k) % 16 == 0 && k_st >= 128,
              "kvq_snapkv_scores: key rows must be 16-byte aligned and not overlap");
  // byte offsets of the last tile's keys (up to H + 15 rows) stay below 2^31
  KVQ_REQUIRE((H + 16) * k_st * esz < (1LL << 31), "kvq_snapkv_scores: one head's keys must span < 2 GiB");
  const int64_t BH = B * Hkv, rows = (Hq / Hkv) * window;
  const SnapPlan sp = snap_plan(BH, rows, window, H, dtype);
  const int64_t need = snap_ws(BH, rows, window, H, sp, dtype);
  KVQ_REQUIRE(workspace_floats >= need, "kvq_snapkv_scores: workspace too small (%lld < %lld floats)",
              (long long)workspace_floats, (long long)need);
  SnapParams p{};
  p.q = q; p.q_sb = q_sb; p.q_sh = q_sh; p.q_st = q_st;
  p.k = k; p.k_sb = k_sb; p.k_sh = k_sh; p.k_st = k_st;
  p.Hkv = static_cast<int>(Hkv); p.rep = static_cast<int>(Hq / Hkv); p.w = static_cast<int>(window);
  p.H = static_cast<int>(H); p.rows = static_cast<int>(rows);
  p.BH = static_cast<int>(BH); p.n_rg = sp.n_rg; p.n_split = sp.n_split; p.split_keys = sp.split_keys;
  p.n_pool = sp.n_pool; p.kernel = kernel;
  p.qscale = scaling * kSnapLog2e;
  p.inv_count = 1.0f / static_cast<float>(rows);
  float* ws = workspace;
  p.part_m = ws; ws += BH * sp.n_split * rows;
  p.part_l = ws; ws += BH * sp.n_split * rows;
  p.row_m = ws; ws += BH * rows;
  p.row_il = ws; ws += BH * rows;
  p.colsum = ws; ws += BH * sp.n_rg * (H - window);
  p.blockmax = ws; ws += BH * sp.n_pool;
  p.out = out;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const dim3 blk(kSnapThreads), logit(kLogitThreads), units(static_cast<unsigned>((BH * sp.n_split + 7) / 8 * 8 * sp.n_rg));
  if (dtype == KVQ_F32) {
    // the powers of two that bring the window's query rows and the keys into the fp16 parts' range
    p.xs = ws + kAmaxViews * kAmaxBlocks;
    const RowView views[2] = {
        RowView{static_cast<const float*>(q), static_cast<int>(B), static_cast<int>(Hq), static_cast<int>(window),
                q_sb, q_sh, q_st},
        RowView{static_cast<const float*>(k), static_cast<int>(B), static_cast<int>(Hkv), static_cast<int>(H), k_sb,
                k_sh, k_st}};
    launch_rows_scales(views, 2, ws, const_cast<float*>(p.xs), s);
    KVQ_LAUNCH_CHECK("kvq_snapkv_scores(fp32 scales)");
  }
  KVQ_DISPATCH_DTYPE(dtype, hipLaunchKernelGGL((snap_stats<DT_>), units, logit, 0, s, p));
  KVQ_LAUNCH_CHECK("kvq_snapkv_scores(stats)");
  hipLaunchKernelGGL(snap_rows, dim3((BH * rows + kSnapThreads / 16 - 1) / (kSnapThreads / 16)), blk, 0, s, p, BH * rows);
  KVQ_LAUNCH_CHECK("kvq_snapkv_scores(rows)");
  KVQ_DISPATCH_DTYPE(dtype, hipLaunchKernelGGL((snap_cols<DT_>), units, logit, 0, s, p));
  KVQ_LAUNCH_CHECK("kvq_snapkv_scores(cols)");
  hipLaunchKernelGGL(snap_pool, dim3(BH * sp.n_pool), blk, 0, s, p);
  KVQ_LAUNCH_CHECK("kvq_snapkv_scores(pool)");
  hipLaunchKernelGGL(snap_window, dim3(BH), blk, 0, s, p, static_cast<int>(BH * sp.n_pool));
  KVQ_LAUNCH_CHECK("kvq_snapkv_scores(window)");
  return KVQ_OK;
}
