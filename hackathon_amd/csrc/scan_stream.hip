// Matrix-state scan that streams the tiles, for large launches of short runs
// (see scan_mat.h for the recurrence and launch_mat_scan for the rule that
// takes a launch here).
//
// A slot's tile is S = F B + sum_j a_j b_j g_j^T (B in the state store, the
// sum its pending log). Over a run of up to eight steps with alpha_t,
// sb_t = scale_t beta_t, gamma_t and w_t, the log entries and the run's own
// steps are one list of at most 16 rank-1 entries (b_j, g_j), and
//   out_t = P_t F (w_t . B) + sum_j c_tj (w_t . b_j) g_j,
// with P_t the product of the alphas up to t and c_tj = P_t a_j for a log
// entry, the product of the alphas after s for step s <= t (the sum ends
// there: a step's output never reads a later step's operands). So a
// run that leaves its tile in the store (its steps fit the log) reads the
// tile once and spends one multiply-add per element and step: nothing is
// applied to the tile and nothing of it is kept, where mat_scan_kernel applies
// every entry and step to a resident tile (two to three operations per element
// each). A run that writes the tile back adds one multiply-add per element and
// entry: P F B + sum_j c_j b_j g_j^T.
//
// What bounds it: the read of the tiles. A wave owns 64 tile rows of a
// 256-column tile and streams them one 1 KB row per load, U at a time and two
// such groups in flight; w_t (and b_j where the tile is written) come from
// LDS, four rows per 16-byte read. The waves' sums meet in LDS once per run.
// Measured alone (microseconds, this / mat_scan_kernel; runs of 1, 2, 4 and 8
// steps, logs 0 to 5 entries full, so that most stay, then all full, so that
// every tile is written):
// - 300 runs of 8 512x512 tiles 438 / 480, 488 / 544, 619 / 653, 938 / 1031 (5.8
//   TB/s read at one step); written 1002 / 1046, 1008 / 1071, 1020 / 1114, 1055 /
//   1275 (5.0 TB/s);
// - 64 runs 101 / 114, 111 / 125, 153 / 156, 216 / 249; written 226 / 244 to 252
//   / 305;
// - 300 runs of 8 256x256 tiles 125 / 139, 136 / 158, 183 / 204, 289 / 346;
//   written 272 / 270, 276 / 282, 290 / 310, 339 / 377.
#include <cstdint>

#include "scan_mat.h"

namespace hk {
namespace {

constexpr int kEnt = 2 * kLogCapMax;  // entries of one run: log + steps
static_assert(kLogCapMax == 8, "dispatch on up to eight steps");

// Raw buffer resource word 3 (gfx9: 32-bit data format, no stride, no
// swizzle): an access past the range reads zero and drops its store.
constexpr int kBufWord3 = 0x00020000;

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int CT = 256;            // columns of a work-group
constexpr int TS = kLogCapMax;     // steps of a run
constexpr int TC = 2;              // steps whose sums meet in LDS at once
static_assert(TC * CT <= 64 * kEnt, "the sums fit b's area");

// LDS of a work-group of `waves` waves (floats): g of the run's entries
// [kEnt][CT]; per wave one area for its rows of the entries' b, [kEnt][64],
// and (when the tile is not being updated) its output sums [TC][CT]; per
// wave its rows of w [TS][64]; the waves' dot products [waves][TS][kEnt];
// the coefficients [TS][kEnt + 1].
constexpr int stream_lds(int waves) {
  return kEnt * CT + waves * 64 * (kEnt + TS) + waves * TS * kEnt + TS * (kEnt + 1);
}

// The scalars of one block of steps, lane l of every wave holding entry l's
// and step l's (l < 16).
struct Run {
  int n, ne;      // log entries, all entries
  int ns;         // steps
  int64_t row0;   // request row of step 0
  float f;        // factor of the tile before step 0
  float c;        // lane l: entry l's weight when it enters (log: a_l, steps: 1)
  float sc;       // lane l: factor of entry l's b (steps: scale; 0 past ne)
  float al;       // lane l: alpha of step l (1 past ns)
};

__device__ __forceinline__ float lane_value(float v, int l) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
}

// One (run, head, column tile).
struct Tile {
  static constexpr int NL = 64;  // loads (= rows) of a wave
  const MatScanDesc& d;
  int head, col0, lane, wave, waves, tid;
  int r0, len;
  const float* lh;  // log header
  int64_t le0;      // first log entry
  __amdgpu_buffer_rsrc_t rs;  // this wave's rows, from the tile's first column
  int row_b;        // bytes of a tile row
  int lane_b;       // this lane's columns 4 lane ..
  int rbase;        // this wave's first row within the tile
  float *lg, *lb, *lw, *ldot, *lcd;

  // The wave's slice is a buffer resource: row i at a scalar offset, the
  // lane's four columns at one vector offset.
  __device__ __forceinline__ f32x4 load(int i) const {
    return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, lane_b, i * row_b, 0));
  }
  // (No scalar offset here: the compiler puts the wait between a 16-byte
  // store and the next write of its data registers only on the form without
  // one, and without the wait that write reached the last lanes' data.)
  __device__ __forceinline__ void store(int i, f32x4 v) const {
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), rs, lane_b + i * row_b, 0, 0);
  }
  // Values of rows i .. i + 3 (i a multiple of 4) of a row vector of this
  // wave in LDS (p[64]).
  __device__ __forceinline__ f32x4 rows4(const float* p, int i) const {
    return *reinterpret_cast<const f32x4*>(p + i);
  }
  __device__ __forceinline__ float* wave_w() const { return lw + wave * TS * 64; }
  __device__ __forceinline__ float* wave_b() const { return lb + wave * kEnt * 64; }

  __device__ __forceinline__ Run scalars(int n_log, float f) const {
    const int64_t row0 = r0;
    const int ns = len;
    Run k;
    k.n = n_log;
    k.ns = ns;
    k.ne = n_log + ns;
    k.row0 = row0;
    k.f = f;
    k.al = 1.0f;
    k.c = 1.0f;
    k.sc = 0.0f;
    if (lane < ns)
      k.al = gload(d.alpha.ptr + (row0 + lane) * d.alpha.row_stride + (int64_t)head * d.alpha.head_stride);
    if (lane < n_log) {
      k.c = gload(lh + 2 + lane);
      k.sc = 1.0f;
    } else if (lane < k.ne) {
      k.sc = d.scale.ptr ? gload(d.scale.ptr + (row0 + lane - n_log) * d.scale.row_stride +
                                 (int64_t)head * d.scale.head_stride)
                         : 1.0f;
    }
    return k;
  }

  // w of the run's steps to LDS (this wave's rows, read back by this wave;
  // zero past the run).
  template <int T>
  __device__ __forceinline__ void stage_w(const Run& k) const {
    const float* p = d.w.ptr + k.row0 * d.w.row_stride + (int64_t)head * d.w.head_stride + rbase + lane;
    float w[T];
#pragma unroll
    for (int t = 0; t < T; ++t) w[t] = t < k.ns ? gload(p + t * d.w.row_stride) : 0.0f;
#pragma unroll
    for (int t = 0; t < T; ++t) wave_w()[t * 64 + lane] = w[t];
  }

  // This lane's row of b of the run's first NE entries (NE at least k.ne;
  // zero past k.ne, whose loads repeat the last entry's).
  template <int NE>
  __device__ __forceinline__ void load_b(const Run& k, float (&b)[NE]) const {
    const float* log = d.log_b + le0 * d.rows + rbase;
    const float* st = d.beta.ptr + (k.row0 - k.n) * d.beta.row_stride + (int64_t)head * d.beta.head_stride + rbase;
#pragma unroll
    for (int j = 0; j < NE; ++j) {
      const int q = min(j, k.ne - 1);
      const float* p = q < k.n ? log + (int64_t)q * d.rows : st + (int64_t)q * d.beta.row_stride;
      b[j] = gload(p + lane);
    }
    // (scale * beta): the association the reference uses
#pragma unroll
    for (int j = 0; j < NE; ++j) b[j] = j < k.ne ? lane_value(k.sc, j) * b[j] : 0.0f;
  }
  // Column tile of g of the run's entries to LDS.
  __device__ __forceinline__ void stage_g(const Run& k) const {
    const int c = tid % CT;
    const float* log = d.log_g + le0 * d.cols + col0;
    const float* st = d.gamma.ptr + (k.row0 - k.n) * d.gamma.row_stride + (int64_t)head * d.gamma.head_stride + col0;
    const int j0 = __builtin_amdgcn_readfirstlane(tid / CT);  // CT is whole waves
#pragma unroll 4
    for (int j = j0; j < k.ne; j += 64 * waves / CT) {
      const float* p = j < k.n ? log + (int64_t)j * d.cols : st + (int64_t)j * d.gamma.row_stride;
      lg[j * CT + c] = gload(p + c);
    }
  }

  // This wave's share of w_t . b_j for every step and entry.
  template <int NE>
  __device__ __forceinline__ void dots(const Run& k, const float (&b)[NE]) const {
#pragma unroll 1
    for (int t = 0; t < k.ns; ++t) {
      const float wt = wave_w()[t * 64 + lane];
      float p[NE];
#pragma unroll
      for (int j = 0; j < NE; ++j) p[j] = wt * b[j];
      const float s = transposed_wave_sum<NE>(p);  // lane (64 / NE) j holds entry j
      if (lane % (64 / NE) == 0) ldot[(wave * TS + t) * kEnt + lane / (64 / NE)] = s;
    }
  }

  // c_tj (w_t . b_j) and P_t F of the block to LDS, step t by wave t % waves;
  // between two barriers. NE as the dots were formed.
  template <int NE>
  __device__ __forceinline__ void coefficients(const Run& k) const {
    float c = lane < k.n ? k.c : 0.0f;
    float pf = k.f;
#pragma unroll 1
    for (int t = 0; t < k.ns; ++t) {
      const float a = lane_value(k.al, t);
      pf *= a;
      c = lane == k.n + t ? 1.0f : c * a;
      if (t % waves == wave) {
        float q = 0.0f;
        if (lane < NE)
          for (int v = 0; v < waves; ++v) q += ldot[(v * TS + t) * kEnt + lane];
        if (lane < kEnt) lcd[t * (kEnt + 1) + lane] = c * q;
        if (lane == kEnt) lcd[t * (kEnt + 1) + kEnt] = pf;
      }
    }
  }

  // Lane j: entry j's weight after the run's last step; pf: the tile's.
  __device__ __forceinline__ float final_weights(const Run& k, float& pf) const {
    float c = k.c;
    pf = k.f;
#pragma unroll
    for (int u = 0; u < TS; ++u) {
      const float a = lane_value(k.al, u);
      pf *= a;
      if (u > lane - k.n) c *= a;
    }
    return c;
  }
  // b_j times its final weight to LDS (this wave's rows).
  template <int NE>
  __device__ __forceinline__ void stage_b(const Run& k, float c, const float (&b)[NE]) const {
#pragma unroll
    for (int j = 0; j < NE; ++j)
      if (j < k.ne) wave_b()[j * 64 + lane] = lane_value(c, j) * b[j];
  }

  __device__ __forceinline__ void put_sums(int q, f32x4 a) const {
    *reinterpret_cast<f32x4*>(wave_b() + q * CT + 4 * lane) = a;
  }
  // Outputs of steps t0 .. t0 + m - 1 (their sums are in LDS).
  __device__ __forceinline__ void outputs(const Run& k, int t0, int m) const {
    const int c = tid % CT;
    float* ob = d.out + (int64_t)head * d.out_head_stride + col0 + c;
    for (int q = tid / CT; q < m; q += (64 * waves) / CT) {
      const int t = t0 + q;
      float s = 0.0f;
#pragma unroll 1
      for (int v = 0; v < waves; ++v) s += lb[v * kEnt * 64 + q * CT + c];
      float o = lcd[t * (kEnt + 1) + kEnt] * s;
      // up to the step's own entry: a later one's weight is zero, but zero times
      // an infinity or NaN that came with a later request is not
#pragma unroll 1
      for (int j = 0; j <= k.n + t; ++j) o = fmaf(lcd[t * (kEnt + 1) + j], lg[j * CT + c], o);
      gstore(ob + (k.row0 + t) * d.out_row_stride, o);
    }
  }

  // v (loads i0 .. i0 + U - 1) <- pf v + sum_j b_j g_j
  template <int U>
  __device__ __forceinline__ void update(f32x4 (&v)[U], int i0, int ne, float pf) const {
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] *= pf;
    const float* gl = lg + 4 * lane;
#pragma unroll 1
    for (int j = 0; j < ne; ++j) {
      const f32x4 g = *reinterpret_cast<const f32x4*>(gl + j * CT);
#pragma unroll
      for (int u0 = 0; u0 < U; u0 += 4) {
        const f32x4 bj = rows4(wave_b() + j * 64, i0 + u0);
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int e = 0; e < 4; ++e) v[u0 + u][e] = fmaf(bj[u], g[e], v[u0 + u][e]);
      }
    }
  }
  template <int T, int U>
  __device__ __forceinline__ void accumulate(f32x4 (&acc)[T], const f32x4 (&v)[U], int i0) const {
#pragma unroll
    for (int u0 = 0; u0 < U; u0 += 4)
#pragma unroll
      for (int t = 0; t < T; ++t) {
        const f32x4 wv = rows4(wave_w() + t * 64, i0 + u0);
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[t][e] = fmaf(wv[u], v[u0 + u][e], acc[t][e]);
      }
  }
  // f(i, v) for the tile's loads i .. i + U - 1 in v, two groups (or one) in
  // flight.
  template <int U, int GROUPS = 2, typename Fn>
  __device__ __forceinline__ void for_tile(Fn&& f) const {
    static_assert(NL % (2 * U) == 0, "whole pairs of groups");
    if constexpr (GROUPS == 1) {
#pragma unroll 1
      for (int i = 0; i < NL; i += U) {
        f32x4 v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = load(i + u);
        f(i, v);
      }
      return;
    }
    f32x4 va[U], vb[U];
#pragma unroll
    for (int u = 0; u < U; ++u) va[u] = load(u);
#pragma unroll 1
    for (int i = 0; i < NL; i += 2 * U) {
#pragma unroll
      for (int u = 0; u < U; ++u) vb[u] = load(i + U + u);
      f(i, va);
      if (i + 2 * U < NL)
#pragma unroll
        for (int u = 0; u < U; ++u) va[u] = load(i + 2 * U + u);
      f(i + U, vb);
    }
  }
  template <int T>
  __device__ __forceinline__ void finish(const Run& k, const f32x4 (&acc)[T]) const {
#pragma unroll
    for (int t0 = 0; t0 < T; t0 += TC) {
      if (t0 < k.ns) {
        if (t0 > 0) lds_barrier();  // the earlier sums are read
#pragma unroll
        for (int q = 0; q < TC; ++q)
          if (t0 + q < T) put_sums(q, acc[t0 + q]);
        lds_barrier();
        outputs(k, t0, min(TC, k.ns - t0));
      }
    }
  }

  // A run of at most T <= 8 steps: the tile streams through registers.
  template <int T>
  __device__ __forceinline__ void stream(int n_log, float f) const {
    const Run k = scalars(n_log, f);
    stage_w<T>(k);
    f32x4 acc[T];
#pragma unroll
    for (int t = 0; t < T; ++t) acc[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    if (k.ne <= d.log_cap) {  // the tile stays, the steps join the log
      constexpr int U = T <= 2 ? 8 : 4;  // (register budget: 128)
      for_tile<U>([&](int i, const f32x4(&v)[U]) { accumulate<T, U>(acc, v, i); });
      float b[kLogCapMax];
      load_b(k, b);
      stage_g(k);
      dots(k, b);
      // log entries n .. n + len - 1: column tile 0 writes the wave's rows of
      // b, each column tile (below) its columns of g
      if (blockIdx.x == 0)
#pragma unroll
        for (int j = 0; j < kLogCapMax; ++j)
          if (j >= k.n && j < k.ne) gstore(d.log_b + (le0 + j) * d.rows + rbase + lane, b[j]);
      lds_barrier();
      coefficients<kLogCapMax>(k);
      if (tid < CT)
        for (int j = k.n; j < k.ne; ++j) gstore(d.log_g + (le0 + j) * d.cols + col0 + tid, lg[j * CT + tid]);
    } else {
      float b[kEnt], pf;
      load_b(k, b);
      stage_g(k);
      dots(k, b);
      stage_b(k, final_weights(k, pf), b);
      lds_barrier();
      coefficients<kEnt>(k);
      constexpr int U = 4;
      for_tile<U, T == 8 ? 1 : 2>([&](int i, f32x4(&v)[U]) {
        accumulate<T, U>(acc, v, i);
        update<U>(v, i, k.ne, pf);
#pragma unroll
        for (int u = 0; u < U; ++u) store(i + u, v[u]);
      });
      lds_barrier();  // the sums take b's place
    }
    finish<T>(k, acc);
  }
};

__global__ __launch_bounds__(512, 4) void stream_scan_kernel(MatScanDesc d) {
  extern __shared__ __align__(16) float smem[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int waves = blockDim.x >> 6;
  const int head = blockIdx.y;
  const int run = blockIdx.z;
  const int slot = d.slot_ids[run];
  const int r0 = d.run_off[run];
  Tile k{d};
  k.head = head;
  k.col0 = blockIdx.x * CT;
  k.lane = lane;
  k.wave = wave;
  k.waves = waves;
  k.tid = tid;
  k.r0 = r0;
  k.len = d.run_off[run + 1] - r0;
  k.lh = d.log_hdr + ((int64_t)slot * d.heads + head) * kLogHdr;
  k.le0 = ((int64_t)slot * d.heads + head) * d.log_cap;
  k.rbase = wave * 64;
  k.row_b = 4 * (int)d.row_stride;
  k.lane_b = 16 * lane;
  k.rs = __builtin_amdgcn_make_buffer_rsrc(
      d.state + (int64_t)slot * d.slot_stride + (int64_t)head * d.head_stride +
          (int64_t)k.rbase * d.row_stride + blockIdx.x * CT,
      0, 63 * k.row_b + CT * 4, kBufWord3);
  k.lg = smem;
  k.lb = k.lg + kEnt * CT;
  k.lw = k.lb + waves * 64 * kEnt;
  k.ldot = k.lw + waves * 64 * TS;
  k.lcd = k.ldot + waves * TS * kEnt;
  const int n = (int)k.lh[0];
  const float f = k.lh[1];
  if (k.len == 1)
    k.stream<1>(n, f);
  else if (k.len == 2)
    k.stream<2>(n, f);
  else if (k.len <= 4)
    k.stream<4>(n, f);
  else
    k.stream<8>(n, f);
}

}  // namespace

// Where the lines lie (ticks of equal runs, default widths, bf16, two layers,
// us, streaming / general; 512 work-groups are 32 runs of the mLSTM, 64 of
// RetNet):
// - From 512 work-groups, two per CU: 32 runs of 1, 4 and 8 steps 657 / 671, 812 /
//   838, 1042 / 1106; 64 runs 845 / 880, 1203 / 1269, 1658 / 1823; 96 runs of 8
//   2378 / 2593 (twelve layers, 64 runs 4688 / 4913, 6682 / 7043, 9593 / 10551).
//   Below, in ticks of equal runs, it is ahead as well (24 runs of 1 and 8 steps
//   568 / 579, 898 / 938): the line is on the safe side. The engine keeps the
//   second xLSTM group of a split tick off it longer (group2_runs).
// - Runs of more than eight steps go to mat_scan_kernel in a launch before this
//   one. Taken from 256 short runs: 256 single runs beside two long ones 2336 /
//   2447, 512 4152 / 4329. On the safe side too: streaming 192 would give 1855
//   against 1975, 64 none (twelve layers, 64 and 96 runs 5406 / 5349 and 6699 /
//   6588).
// - Narrower tiles (Mamba2's 128 x 64) read no faster this way (300 runs 151 / 142
//   us alone).
bool stream_scan_takes(const MatScanDesc& d) {
  const int n_short = d.n_runs - d.n_long;
  return d.n_long >= 0 && !d.per_row && d.log_cap == kLogCapMax && d.row_parts == 1 &&
         d.rows % 64 == 0 && d.rows >= 256 && d.rows <= 512 && d.cols % 256 == 0 &&
         d.col_stride == 1 && d.row_stride % 4 == 0 && d.head_stride % 4 == 0 &&
         d.slot_stride % 4 == 0 && (reinterpret_cast<uintptr_t>(d.state) & 15) == 0 &&
         (int64_t)n_short * d.heads * (d.cols / 256) >= 512 && (d.n_long == 0 || n_short >= 256);
}

int launch_stream_scan(const MatScanDesc& d, hipStream_t stream) {
  const int waves = d.rows / 64;
  const size_t lds = stream_lds(waves) * sizeof(float);
  hipLaunchKernelGGL(stream_scan_kernel, dim3(d.cols / CT, d.heads, d.n_runs), dim3(64 * waves), lds,
                     stream, d);
  HK_LAUNCH_CHECK();
  return HK_OK;
}

}  // namespace hk
