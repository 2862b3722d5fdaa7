// Dense projections of the decoder layer on gfx950, at decode batch sizes and
// those of short prefill steps: y = x . w^T, with the layer's RMSNorm in front of it, the
// SwiGLU gate or the residual sum behind it (entry points in
// include/mi_model.h).
//
// What bounds them: w streams once from memory (8.4 MB for a 4096 x 1024
// projection: 1.7 us at the measured copy rate of 4.9 TB/s), but a launch of
// that size is mostly latency -- the launch itself, one memory round trip,
// the sum over the waves -- so the kernels keep everything a wave needs in
// flight at once, and a step's norm, gate and residual sum ride on the
// projections instead of being launches of their own (3.1-3.6 us each).
//
// Two kernels:
//  * linear_kernel (MFMA): a workgroup owns 16 or 32 columns and every row;
//    its waves split k. A operand: 16 weight rows as stored; B operand: 16
//    rows of x. All waves then add the partial sums, wave by wave in order,
//    each wave a share of the tiles.
//  * gemv_kernel (one or two rows): a wave owns whole weight rows, a lane 8 elements
//    of every 512, so a load instruction takes 1 KiB of one row; narrow
//    outputs (1024 columns) then still give all CUs work, where 16-column
//    tiles leave three quarters of them idle.
//
// RMSNorm in front, bf16: y[m] = (1 / rms(x[m])) * (x[m] * weight) . w^T. The
// product x * weight is rounded once to the element type (torch's norm rounds
// twice), 1 / rms scales the float32 sum, so no pass over the row comes first.
// float16: x * weight may lie outside the type's range where the normalised
// row does not (kNormFirst), so the row is normalised first, with the
// additions and roundings of rms_norm_residual_kernel: the result is that
// launch's and the projection's, bit for bit. The pass over the row costs
// (4096 x 1024, us, against scaling the sum) 0.2 at one row, 1.2 at 16, 2.4
// at 64, where the norm's own launch is the cheaper (8.6 against 7.7 in all).
#include "mi_common.h"
#include "mi_model.h"

namespace mi {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

template <typename E>
struct LinMfma;
template <>
struct LinMfma<BF16> {
  using vec8 = bf16x8_t;
  using el = __bf16;
  static __device__ __forceinline__ f32x4_t mma(vec8 a, vec8 b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};
template <>
struct LinMfma<F16> {
  using vec8 = f16x8_t;
  using el = _Float16;
  static __device__ __forceinline__ f32x4_t mma(vec8 a, vec8 b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};

constexpr int kLinMaxRows = 64;
constexpr int kLinMaxFusedRows = 4096;  // mi_linear_fused without a norm
constexpr int kLinStep = 32;  // k per MFMA

struct LinArgs {
  const void* x;
  int64_t xs;
  const void* w;
  int64_t ws;
  void* y;
  int64_t ys;
  int32_t m, n, k;
  int32_t row_groups; // MFMA launches: groups of 16 MT rows
  int32_t inter;      // GLU: rows [0, inter) of w are the gate, the rest up
  const void* norm;   // RMSNorm weight of x (null: x as it is)
  float eps;
  const void* res;    // added to y (null: none)
  int64_t rs;
};

// Whether rows are normalised before they are rounded again. float16 holds
// 6e-8 to 65504: a row with a channel of 6000 under a weight of 12 is finite
// once normalised, its product before that is not.
template <typename E>
constexpr bool kNormFirst = std::is_same<E, F16>::value;

// x[i] * w[i] over an 8-element fragment, rounded once.
template <typename E>
__device__ __forceinline__ Pack<uint16_t, 8> scale8(const Pack<uint16_t, 8>& x,
                                                    const Pack<uint16_t, 8>& w) {
  Pack<uint16_t, 8> r;
#pragma unroll
  for (int i = 0; i < 8; ++i)
    r.v[i] = __builtin_bit_cast(
        uint16_t, static_cast<typename LinMfma<E>::el>(E::load(x.v[i]) * E::load(w.v[i])));
  return r;
}

// round(round(x[i] * inv) * w[i]) over an 8-element fragment.
template <typename E>
__device__ __forceinline__ Pack<uint16_t, 8> norm8(const Pack<uint16_t, 8>& x, float inv,
                                                   const Pack<uint16_t, 8>& w) {
  Pack<uint16_t, 8> r;
#pragma unroll
  for (int i = 0; i < 8; ++i)
    r.v[i] = norm_round<E>(x.v[i], inv, w.v[i]);
  return r;
}

template <typename E>
__device__ __forceinline__ float add_squares(const Pack<uint16_t, 8>& x, float ss) {
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float f = E::load(x.v[i]);
    ss = fmaf(f, f, ss);
  }
  return ss;
}

// 1 / rms of ROWS rows of k elements by a wave, summed in the order of
// rms_norm_residual_kernel: lane i takes the 8-element pieces i, i + 64, ...
template <typename E, int ROWS>
__device__ __forceinline__ void inverse_rms(const uint16_t* const (&row)[ROWS], int k, float eps,
                                            int lane, float (&inv)[ROWS]) {
  constexpr int kAhead = 2;  // pieces of each row in flight
  float ss[ROWS];
#pragma unroll
  for (int r = 0; r < ROWS; ++r) ss[r] = 0.f;
  for (int k0 = 0; k0 < k; k0 += kAhead * 8 * kWave) {
    Pack<uint16_t, 8> x[kAhead][ROWS];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      const int off = k0 + (i * kWave + lane) * 8;
#pragma unroll
      for (int r = 0; r < ROWS; ++r) x[i][r] = load_pack<uint16_t, 8>(row[r] + (off < k ? off : 0));
    }
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      if (k0 + (i * kWave + lane) * 8 < k) {
#pragma unroll
        for (int r = 0; r < ROWS; ++r) ss[r] = add_squares<E>(x[i][r], ss[r]);
      }
    }
  }
#pragma unroll
  for (int r = 0; r < ROWS; ++r)
    inv[r] = rsqrtf(group_sum<kWave>(ss[r]) / static_cast<float>(k) + eps);
}

// acc + sum of x[i] * w[i] over the fragment.
template <typename E>
__device__ __forceinline__ float dot8(const Pack<uint16_t, 8>& x, const Pack<uint16_t, 8>& w,
                                      float acc) {
  const Pack<uint32_t, 4> a = __builtin_bit_cast(Pack<uint32_t, 4>, x);
  const Pack<uint32_t, 4> b = __builtin_bit_cast(Pack<uint32_t, 4>, w);
#pragma unroll
  for (int i = 0; i < 4; ++i) acc = E::dot2(a.v[i], b.v[i], acc);
  return acc;
}

// The residual sum of one element, rounded as a separate launch rounds it.
template <typename E>
__device__ __forceinline__ uint16_t add_residual(uint16_t y, uint16_t res) {
  return E::store(E::load(y) + E::load(res));
}

// ---------------------------------------------------------------------------
// MFMA kernel.
// ---------------------------------------------------------------------------
// NW waves split k by chunks of KC (wave w: a contiguous range); NT 16-column
// tiles per workgroup (GLU: the first half gate columns, the second the
// matching up columns); MT 16-row tiles of x per workgroup, row groups of one
// column tile on one XCD. S LDS slots of one chunk per wave.
//
// A wave stages its chunks of w and x in its own LDS slots with direct
// global->LDS loads, 1 KiB of whole chunk rows per instruction, and reads the
// MFMA fragments from there. Loading the fragments straight into registers
// puts 16 different rows in 16 neighbouring lanes: the address unit was then
// busy 69 cycles per vector memory instruction, 31 as it is (TA_TA_BUSY /
// SQ_INSTS_VMEM of the 4096 x 1024 projection at 64 rows, 8.0 and 4.5 us).
// 16-byte piece c of row r sits at place c ^ swz(r): with rows of 256 bytes
// (KC 128) swz = r & 15, of 128 bytes (KC 64, two rows to a bank cycle)
// (r >> 1) & 7, either of which leaves a fragment read (16 rows, one piece)
// without bank conflicts.
template <typename E, int NW, int NT, int MT, int S, int KC, bool GLU, bool NORM>
__global__ __launch_bounds__(NW* kWave) void linear_kernel(const LinArgs a) {
  using M = LinMfma<E>;
  using vec8 = typename M::vec8;
  using R = uint16_t;
  static_assert(!GLU || NT % 2 == 0, "GLU launches: gate and up tiles");
  constexpr int kOut = GLU ? NT / 2 : NT;  // 16-column tiles of y
  constexpr int kUnits = kOut * MT;        // result tiles to add up and store
  constexpr int kChunkSteps = KC / kLinStep;
  constexpr int kRowBytes = KC * 2;
  constexpr int kTileBytes = 16 * kRowBytes;
  constexpr int kPieces = KC / 8;               // 16-byte pieces of a row
  constexpr int kLoadRows = kWave / kPieces;    // rows per load
  constexpr int kLoads = 16 / kLoadRows;        // loads per tile
  constexpr int kSlot = (NT + MT) * kTileBytes;
  constexpr int kSums = NW * NT * MT * kWave * 16;
  constexpr int kRing = NW * S * kSlot;
  // The ring, then (after every wave has read its last chunk) the sums.
  __shared__ __attribute__((aligned(16))) char s_mem[kRing > kSums ? kRing : kSums];
  constexpr bool kFirst = NORM && kNormFirst<E>;
  constexpr bool kAfter = NORM && !kNormFirst<E>;
  __shared__ float s_ss[kAfter ? NW : 1][MT * 16];  // squares by wave, or the rows' 1 / rms
  const int tid = threadIdx.x;
  const int lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int col = lane % 16;   // weight row (output column) / x row within a tile
  const int quad = lane / 16;  // 8-element group of the k-step
  const int xcd = blockIdx.x % 8, rest = blockIdx.x / 8;
  const int r0 = 16 * MT * (rest % a.row_groups);
  const int n0 = (rest / a.row_groups * 8 + xcd) * (16 * kOut);
  if (n0 >= (GLU ? a.inter : a.n)) return;
  const int chunks = (a.k + KC - 1) / KC;
  const int per_wave = (chunks + NW - 1) / NW;
  const int c_begin = min(wave * per_wave, chunks);
  const int c_end = min(c_begin + per_wave, chunks);

  f32x4_t acc[NT][MT];
  float ss[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    ss[t] = 0.f;
#pragma unroll
    for (int u = 0; u < NT; ++u) acc[u][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }

  // Load i of a tile takes its rows kLoadRows i ..; lane / kPieces is the row
  // of them, lane % kPieces the place in it. n % 16 == 0: a tile's columns
  // exist or none do (then tile 0 is read in its place). Rows of x past m
  // repeat the last one; their results are not stored.
  auto swz = [](int row) { return KC == 128 ? row & 15 : (row >> 1) & 7; };
  const R* src[(NT + MT) * kLoads];
  int piece[kLoads];
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const int row = kLoadRows * i + lane / kPieces;
    piece[i] = (lane % kPieces ^ swz(row)) * 8;
#pragma unroll
    for (int u = 0; u < NT; ++u) {
      const int c = n0 + 16 * (u % kOut);
      const int wr = (c < (GLU ? a.inter : a.n) ? c : n0) + u / kOut * a.inter;
      src[u * kLoads + i] = static_cast<const R*>(a.w) + static_cast<int64_t>(wr + row) * a.ws;
    }
#pragma unroll
    for (int t = 0; t < MT; ++t)
      src[(NT + t) * kLoads + i] = static_cast<const R*>(a.x) +
                                   static_cast<int64_t>(min(r0 + 16 * t + row, a.m - 1)) * a.xs;
  }
  char* ring = s_mem + wave * S * kSlot;
  auto issue = [&](int slot, int c) {
    char* dst = ring + slot * kSlot;
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      // A last chunk may end early: pieces past the row read its start.
      int off = c * KC + piece[i];
      off = off < a.k ? off : 0;
#pragma unroll
      for (int t = 0; t < NT + MT; ++t)
        lds_load16(src[t * kLoads + i] + off, dst + t * kTileBytes + i * 1024);
    }
  };
  auto fragment = [&](const char* tile, int step) {
    return *reinterpret_cast<const Pack<R, 8>*>(tile + col * kRowBytes +
                                                (((4 * step + quad) ^ swz(col)) * 16));
  };
  auto issue_first = [&]() {
#pragma unroll
    for (int s = 0; s < S; ++s)
      if (c_begin + s < c_end) issue(s, c_begin + s);
  };
  const R* nrow = static_cast<const R*>(a.norm) + quad * 8;
  [[maybe_unused]] float inv[MT];
  if constexpr (kFirst) {
    issue_first();
    constexpr int kRows = MT * 16 / NW;
    const R* row[kRows];
    float row_inv[kRows];
#pragma unroll
    for (int i = 0; i < kRows; ++i)
      row[i] = static_cast<const R*>(a.x) +
               static_cast<int64_t>(min(r0 + wave * kRows + i, a.m - 1)) * a.xs;
    inverse_rms<E>(row, a.k, a.eps, lane, row_inv);
#pragma unroll
    for (int i = 0; i < kRows; ++i)
      if (lane == i) s_ss[0][wave * kRows + i] = row_inv[i];
    __syncthreads();
#pragma unroll
    for (int t = 0; t < MT; ++t) inv[t] = s_ss[0][16 * t + col];
  }
  if (c_begin < c_end) {
    if constexpr (!kFirst) issue_first();
    for (int c = c_begin, slot = 0; c < c_end; ++c, slot = slot + 1 == S ? 0 : slot + 1) {
      Pack<R, 8> g[NORM ? kChunkSteps : 1];
      if constexpr (NORM) {
#pragma unroll
        for (int j = 0; j < kChunkSteps; ++j) {
          const int off = c * KC + j * kLinStep;
          g[j] = load_pack<R, 8>(nrow + (off < a.k ? off : 0));
        }
      }
      // Chunk c is in its slot once at most the younger one is in flight
      // (and the norm weights, which were issued last).
      if (!NORM && S > 1 && c + 1 < c_end)
        __builtin_amdgcn_s_waitcnt(vmcnt_only(kLoads * (NT + MT)));
      else
        __builtin_amdgcn_s_waitcnt(vmcnt_only(0));
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      const char* cur = ring + slot * kSlot;
      const int steps = min(kChunkSteps, (a.k - c * KC) / kLinStep);
#pragma unroll
      for (int j = 0; j < kChunkSteps; ++j) {
        if (j >= steps) break;  // uniform
        vec8 wf[NT];
#pragma unroll
        for (int u = 0; u < NT; ++u)
          wf[u] = __builtin_bit_cast(vec8, fragment(cur + u * kTileBytes, j));
#pragma unroll
        for (int t = 0; t < MT; ++t) {
          Pack<R, 8> x = fragment(cur + (NT + t) * kTileBytes, j);
          if constexpr (kFirst) x = norm8<E>(x, inv[t], g[j]);
          if constexpr (kAfter) {
            ss[t] = dot8<E>(x, x, ss[t]);
            x = scale8<E>(x, g[j]);
          }
#pragma unroll
          for (int u = 0; u < NT; ++u)
            acc[u][t] = M::mma(wf[u], __builtin_bit_cast(vec8, x), acc[u][t]);
        }
      }
      if (c + S < c_end) {
        // The fragment reads of this slot have returned.
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        issue(slot, c + S);
      }
    }
  }
  __syncthreads();  // the ring is free

  // acc[u][t][j] = y^T[n0 + 16 u + 4 quad + j][r0 + 16 t + col], this wave's k.
  f32x4_t* sums = reinterpret_cast<f32x4_t*>(s_mem);
  auto sum_at = [&](int w, int tile) -> f32x4_t& {
    return sums[(w * NT * MT + tile) * kWave + lane];
  };
#pragma unroll
  for (int u = 0; u < NT; ++u)
#pragma unroll
    for (int t = 0; t < MT; ++t) sum_at(wave, u * MT + t) = acc[u][t];
  if constexpr (kAfter) {
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const float v = xor_sum<16, kWave>(ss[t]);
      if (lane < 16) s_ss[wave][16 * t + lane] = v;
    }
  }
  __syncthreads();
  R* y = static_cast<R*>(a.y);
#pragma unroll
  for (int i = 0; i < (kUnits + NW - 1) / NW; ++i) {
    const int unit = wave + i * NW;
    if (unit >= kUnits) break;
    const int t = unit % MT, u = unit / MT;
    f32x4_t v = sum_at(0, unit), up = {};
    if constexpr (GLU) up = sum_at(0, kUnits + unit);
#pragma unroll
    for (int wv = 1; wv < NW; ++wv) {
      v += sum_at(wv, unit);
      if constexpr (GLU) up += sum_at(wv, kUnits + unit);
    }
    if constexpr (kAfter) {
      float sum = 0.f;
#pragma unroll
      for (int wv = 0; wv < NW; ++wv) sum += s_ss[wv][16 * t + col];
      const float inv = rsqrtf(sum / static_cast<float>(a.k) + a.eps);
      v *= inv;
      up *= inv;
    }
    const int r = r0 + 16 * t + col;
    const int c = n0 + 16 * u + 4 * quad;
    if (r >= a.m || n0 + 16 * u >= (GLU ? a.inter : a.n)) continue;
    Pack<R, 4> out;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      out.v[j] = GLU ? silu_mul_round<E>(E::store(v[j]), E::store(up[j])) : E::store(v[j]);
    if (a.res != nullptr) {
      const Pack<R, 4> res =
          load_pack<R, 4>(static_cast<const R*>(a.res) + static_cast<int64_t>(r) * a.rs + c);
#pragma unroll
      for (int j = 0; j < 4; ++j) out.v[j] = add_residual<E>(out.v[j], res.v[j]);
    }
    store_pack<R, 4>(y + static_cast<int64_t>(r) * a.ys + c, out);
  }
}

// ---------------------------------------------------------------------------
// One or two rows.
// ---------------------------------------------------------------------------
constexpr int kGemvWaves = 4;
constexpr int kGemvChunk = 8 * kWave;  // elements of a row one load takes

// A wave owns RW weight rows (GLU: one gate row and its up row) and all M rows
// of x; U loads of each row are in flight.
template <typename E, int M, int RW, int U, bool GLU, bool NORM>
__global__ __launch_bounds__(kGemvWaves* kWave) void gemv_kernel(const LinArgs a) {
  using R = uint16_t;
  static_assert(!GLU || RW == 2, "GLU: a gate row and an up row");
  const int lane = threadIdx.x % kWave;
  const int item = __builtin_amdgcn_readfirstlane(blockIdx.x * kGemvWaves + threadIdx.x / kWave);
  const int n0 = GLU ? item : item * RW;
  if (n0 >= (GLU ? a.inter : a.n)) return;
  const R* wrow[RW];
#pragma unroll
  for (int r = 0; r < RW; ++r)
    wrow[r] = static_cast<const R*>(a.w) +
              static_cast<int64_t>(GLU ? n0 + r * a.inter : min(n0 + r, a.n - 1)) * a.ws;
  const R* xrow[M];
#pragma unroll
  for (int i = 0; i < M; ++i)
    xrow[i] = static_cast<const R*>(a.x) + static_cast<int64_t>(min(i, a.m - 1)) * a.xs;
  const R* nrow = static_cast<const R*>(a.norm);

  constexpr bool kFirst = NORM && kNormFirst<E>;
  constexpr bool kAfter = NORM && !kNormFirst<E>;
  float acc[RW][M], ss[M], inv[M];
#pragma unroll
  for (int i = 0; i < M; ++i) {
    ss[i] = inv[i] = 0.f;
#pragma unroll
    for (int r = 0; r < RW; ++r) acc[r][i] = 0.f;
  }
  for (int k0 = 0; k0 < a.k; k0 += U * kGemvChunk) {
    Pack<R, 8> w[U][RW], x[U][M], g[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int off = k0 + u * kGemvChunk + lane * 8;
      const bool in = off < a.k;
      const int at = in ? off : 0;
#pragma unroll
      for (int r = 0; r < RW; ++r) w[u][r] = load_pack<R, 8>(wrow[r] + at);
      if constexpr (NORM) g[u] = load_pack<R, 8>(nrow + at);
#pragma unroll
      for (int i = 0; i < M; ++i) x[u][i] = load_pack<R, 8>(xrow[i] + at);
    }
    if constexpr (kFirst) {
      // A row that is all here needs no loads of its own for its squares.
      if (a.k <= U * kGemvChunk) {
#pragma unroll
        for (int i = 0; i < M; ++i) {
#pragma unroll
          for (int u = 0; u < U; ++u)
            if (u * kGemvChunk + lane * 8 < a.k) ss[i] = add_squares<E>(x[u][i], ss[i]);
          inv[i] = rsqrtf(group_sum<kWave>(ss[i]) / static_cast<float>(a.k) + a.eps);
        }
      } else if (k0 == 0) {
        inverse_rms<E>(xrow, a.k, a.eps, lane, inv);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (k0 + u * kGemvChunk + lane * 8 < a.k) {
#pragma unroll
        for (int i = 0; i < M; ++i) {
          Pack<R, 8> xv = x[u][i];
          if constexpr (kFirst) xv = norm8<E>(xv, inv[i], g[u]);
          if constexpr (kAfter) {
            ss[i] = dot8<E>(xv, xv, ss[i]);
            xv = scale8<E>(xv, g[u]);
          }
#pragma unroll
          for (int r = 0; r < RW; ++r) acc[r][i] = dot8<E>(xv, w[u][r], acc[r][i]);
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < M; ++i) {
    if constexpr (kAfter) {
      const float scale = rsqrtf(group_sum<kWave>(ss[i]) / static_cast<float>(a.k) + a.eps);
#pragma unroll
      for (int r = 0; r < RW; ++r) acc[r][i] = group_sum<kWave>(acc[r][i]) * scale;
    } else {
#pragma unroll
      for (int r = 0; r < RW; ++r) acc[r][i] = group_sum<kWave>(acc[r][i]);
    }
  }
  // Lane i stores row i of x: the wave's columns are neighbours.
#pragma unroll
  for (int i = 0; i < M; ++i) {
    if (lane != i || i >= a.m) continue;
    R* y = static_cast<R*>(a.y) + static_cast<int64_t>(i) * a.ys + n0;
    const R* res = a.res != nullptr
                       ? static_cast<const R*>(a.res) + static_cast<int64_t>(i) * a.rs + n0
                       : nullptr;
    if constexpr (GLU) {
      const R v = silu_mul_round<E>(E::store(acc[0][i]), E::store(acc[1][i]));
      y[0] = res != nullptr ? add_residual<E>(v, res[0]) : v;
    } else {
#pragma unroll
      for (int r = 0; r < RW; ++r) {
        if (n0 + r >= a.n) continue;
        const R v = E::store(acc[r][i]);
        y[r] = res != nullptr ? add_residual<E>(v, res[r]) : v;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Dispatch.
// ---------------------------------------------------------------------------
template <typename E, int NW, int NT, int MT, int S, int KC, bool GLU, bool NORM>
void launch_mfma(LinArgs a, hipStream_t stream) {
  constexpr int kCols = 16 * (GLU ? NT / 2 : NT);
  a.row_groups = (a.m + 16 * MT - 1) / (16 * MT);
  const int col_tiles = ((GLU ? a.inter : a.n) + kCols - 1) / kCols;
  const dim3 grid(static_cast<uint32_t>((col_tiles + 7) / 8 * 8 * a.row_groups));
  linear_kernel<E, NW, NT, MT, S, KC, GLU, NORM><<<grid, NW * kWave, 0, stream>>>(a);
}

// Two slots per wave while every workgroup has a CU to itself (4096 x 1024 at
// 64 rows: 4.5 us, 4.9 with one), else one slot and more workgroups per CU
// (24576 x 4096 at 32 rows: 40.7, 41.6 with two). With the norm, whose weights
// are waited for with the chunk, one slot.
// Past 64 rows four waves always: a launch has workgroups enough.
template <typename E, int NT, int MT, bool GLU, bool NORM>
void launch_tile(const LinArgs& a, bool eight, bool alone, hipStream_t stream) {
  if (eight) {
    if constexpr (MT <= 2) {
      if constexpr (NT == 1 && MT == 1 && !NORM) {
        if (alone) return launch_mfma<E, 8, NT, MT, 2, 128, GLU, NORM>(a, stream);
      }
      return launch_mfma<E, 8, NT, MT, 1, 128, GLU, NORM>(a, stream);
    }
  } else {
    if constexpr (MT <= 2 && !NORM) {
      if (alone) return launch_mfma<E, 4, NT, MT, 2, 128, GLU, NORM>(a, stream);
    }
    return launch_mfma<E, 4, NT, MT, 1, 128, GLU, NORM>(a, stream);
  }
}

// Tile per workgroup (NT 16-column tiles x MT 16-row tiles): a workgroup's
// time goes with the rows of w and x it stages, so the tile with the least
// (workgroups per CU, rounded up) x (NT + MT). Measured against the others
// (us): 4096 x 1024 at 64 rows 2 x 2 4.5, 1 x 1 6.0, 1 x 2 7.0; 2048 x 6144 at
// 48 rows 1 x 2 11.2, 1 x 1 14.7, 2 x 2 15.0; 24576 x 4096 at 48 rows 2 x 3 45,
// 2 x 2 55; past 64 rows, 4096 x 1024 at 128 rows 2 x 2 5.9, 4 x 4 8.6, at 333
// rows 4 x 4 9.7, 2 x 2 12.3.
struct LinTile {
  int nt, mt;
  bool alone;  // at most one workgroup per CU
};
LinTile pick_tile(const LinArgs& a, bool glu, bool eight) {
  static constexpr int kTiles[][2] = {{1, 1}, {2, 1}, {1, 2}, {2, 2}, {2, 3}, {4, 4}};
  const int cus = device_cus(), rows = (a.m + 15) / 16;
  LinTile best{0, 0, false};
  int64_t best_cost = 0;
  for (const auto& t : kTiles) {
    const int nt = t[0], mt = t[1];
    if (mt > rows || (glu && nt < 2) || (!glu && nt == 2 && mt == 1) || (eight && mt == 3) ||
        (nt == 4 && a.m <= kLinMaxRows))
      continue;
    const int64_t cols =
        glu ? (a.inter + 8 * nt - 1) / (8 * nt) : (a.n + 16 * nt - 1) / (16 * nt);
    const int64_t groups = cols * ((rows + mt - 1) / mt);
    const int64_t cost = (groups + cus - 1) / cus * (nt + mt);
    if (best.nt == 0 || cost < best_cost) {
      best = LinTile{nt, mt, groups <= cus};
      best_cost = cost;
    }
  }
  return best;
}

template <typename E, bool GLU, bool NORM>
void launch_many_rows(const LinArgs& a, hipStream_t stream) {
  // Narrow outputs: eight waves per tile (1024 x 3072 at 8 rows: 4.35 us, 4.68
  // with four); wider ones have workgroups enough (4096 x 1024: 3.9, 3.7 with
  // four). By n alone, so that up to 64 rows the fused gate sums as the
  // projection does (past them the tiles split k at other places, unless it is
  // a multiple of 512).
  const bool eight = a.n < 4096 && a.m <= kLinMaxRows;
  const LinTile t = pick_tile(a, GLU, eight);
  if constexpr (!GLU) {
    if (t.nt == 1 && t.mt == 1) return launch_tile<E, 1, 1, GLU, NORM>(a, eight, t.alone, stream);
    if (t.nt == 1) return launch_tile<E, 1, 2, GLU, NORM>(a, eight, t.alone, stream);
  } else if (t.mt == 1) {
    return launch_tile<E, 2, 1, GLU, NORM>(a, eight, t.alone, stream);
  }
  if constexpr (!NORM) {
    // Chunks of 64 and one slot: two workgroups share a CU (4096 x 1024 at 520
    // rows 14.9 us, 20.9 with two slots).
    if (t.mt == 4) return launch_mfma<E, 4, 4, 4, 1, 64, GLU, NORM>(a, stream);
  }
  if (t.mt == 2) return launch_tile<E, 2, 2, GLU, NORM>(a, eight, t.alone, stream);
  return launch_tile<E, 2, 3, GLU, NORM>(a, eight, t.alone, stream);
}

template <typename E, int M, bool GLU, bool NORM>
void launch_gemv(const LinArgs& a, hipStream_t stream) {
  // Rows per wave and loads in flight: one weight row and, past 1024 elements,
  // up to six loads of it; with the norm two rows share the scaled x.
  constexpr int RW = GLU || NORM ? 2 : 1;
  const int items = GLU ? a.inter : (a.n + RW - 1) / RW;
  const dim3 grid(static_cast<uint32_t>((items + kGemvWaves - 1) / kGemvWaves));
  const dim3 block(kGemvWaves * kWave);
  if (GLU || NORM || a.k <= 2 * kGemvChunk)
    gemv_kernel<E, M, RW, 2, GLU, NORM><<<grid, block, 0, stream>>>(a);
  else if (a.k <= 4 * kGemvChunk)
    gemv_kernel<E, M, RW, 4, GLU, NORM><<<grid, block, 0, stream>>>(a);
  else
    gemv_kernel<E, M, RW, 6, GLU, NORM><<<grid, block, 0, stream>>>(a);
}

// One or two rows take the vector kernel (1024 x 2048: 3.1 / 3.2 us, 3.5 / 3.6
// on MFMA; 4096 x 1024 3.6, 3.8; the gate/up 6144 x 1024 4.7 / 5.1, 5.2 / 5.3);
// four take MFMA (3.8 against 3.7, 4.1 against 3.7, 6.6 against 5.3). Two rows
// of a wide, deep weight too, whose waves wait on six pieces of it and of both
// rows at once (151936 x 4096: 275 us, 220 on MFMA; 32768 x 4096 63, 51; 151936
// x 2048 stays: 104, 109; one row 210, 220). By the weight alone, so that all
// forms of a projection sum alike.
template <typename E, bool GLU, bool NORM>
void launch_typed(const LinArgs& a, hipStream_t stream) {
  const bool deep = a.n >= 32768 && a.k >= 4096;
  if (a.m == 1)
    launch_gemv<E, 1, GLU, NORM>(a, stream);
  else if (a.m == 2 && !deep)
    launch_gemv<E, 2, GLU, NORM>(a, stream);
  else
    launch_many_rows<E, GLU, NORM>(a, stream);
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

int32_t linear(const char* who, const LinArgs& a, bool swiglu, int32_t max_rows, int32_t dtype,
               void* stream) {
  clear_error();
  const std::string fn(who);
  if (!valid_dtype(dtype)) return fail(MI_ERR_INVALID_ARGUMENT, fn + ": bad dtype");
  const int out = swiglu ? a.inter : a.n;
  if (a.m < 0 || out <= 0 || a.k <= 0 || out % 16 || a.k % kLinStep)
    return fail(MI_ERR_INVALID_ARGUMENT,
                fn + ": need m >= 0, the output width a positive multiple of 16, k of 32");
  if (dtype == MI_DTYPE_F32) return fail(MI_ERR_UNSUPPORTED, fn + ": 16-bit types only");
  if (a.m > max_rows)
    return fail(MI_ERR_UNSUPPORTED, fn + ": m above " + std::to_string(max_rows));
  if (a.m == 0) return MI_OK;
  if (!a.x || !a.w || !a.y) return fail(MI_ERR_INVALID_ARGUMENT, fn + ": null pointer");
  if (a.xs < a.k || a.ws < a.k || a.ys < out || (a.res && a.rs < out))
    return fail(MI_ERR_INVALID_ARGUMENT, fn + ": row strides below the row lengths");
  if (!aligned16(a.x) || !aligned16(a.w) || !aligned16(a.y) || a.xs % 8 || a.ws % 8 ||
      a.ys % 8 || (a.norm && !aligned16(a.norm)) || (a.res && (!aligned16(a.res) || a.rs % 8)))
    return fail(MI_ERR_INVALID_ARGUMENT,
                fn + ": pointers and row strides must be 16-byte aligned");
  const hipStream_t s = static_cast<hipStream_t>(stream);
  auto go = [&](auto type) {
    using E = decltype(type);
    if (swiglu)
      a.norm ? launch_typed<E, true, true>(a, s) : launch_typed<E, true, false>(a, s);
    else
      a.norm ? launch_typed<E, false, true>(a, s) : launch_typed<E, false, false>(a, s);
  };
  if (dtype == MI_DTYPE_BF16)
    go(BF16{});
  else
    go(F16{});
  return check_launch(who);
}

}  // namespace
}  // namespace mi

extern "C" int32_t mi_linear(const void* x, int64_t x_row_stride, const void* w,
                             int64_t w_row_stride, void* y, int64_t y_row_stride, int32_t m,
                             int32_t n, int32_t k, int32_t dtype, void* stream) {
  mi::LinArgs a{};
  a.x = x;
  a.xs = x_row_stride;
  a.w = w;
  a.ws = w_row_stride;
  a.y = y;
  a.ys = y_row_stride;
  a.m = m;
  a.n = n;
  a.k = k;
  return mi::linear("mi_linear", a, false, mi::kLinMaxRows, dtype, stream);
}

extern "C" int32_t mi_linear_swiglu(const void* x, int64_t x_row_stride, const void* w,
                                    int64_t w_row_stride, void* y, int64_t y_row_stride,
                                    int32_t m, int32_t inter, int32_t k, int32_t dtype,
                                    void* stream) {
  mi::LinArgs a{};
  a.x = x;
  a.xs = x_row_stride;
  a.w = w;
  a.ws = w_row_stride;
  a.y = y;
  a.ys = y_row_stride;
  a.m = m;
  a.n = 2 * inter;
  a.inter = inter;
  a.k = k;
  return mi::linear("mi_linear_swiglu", a, true, mi::kLinMaxRows, dtype, stream);
}

extern "C" int32_t mi_linear_fused(const void* x, int64_t x_row_stride, const void* norm_weight,
                                   float eps, const void* w, int64_t w_row_stride,
                                   const void* residual, int64_t residual_row_stride, void* y,
                                   int64_t y_row_stride, int32_t m, int32_t n, int32_t k,
                                   int32_t swiglu, int32_t dtype, void* stream) {
  mi::LinArgs a{};
  a.x = x;
  a.xs = x_row_stride;
  a.norm = norm_weight;
  a.eps = eps;
  a.w = w;
  a.ws = w_row_stride;
  a.res = residual;
  a.rs = residual_row_stride;
  a.y = y;
  a.ys = y_row_stride;
  a.m = m;
  a.n = n;
  a.inter = n / 2;
  a.k = k;
  if (swiglu && n % 2 != 0) {
    mi::clear_error();
    return mi::fail(MI_ERR_INVALID_ARGUMENT, "mi_linear_fused: gate/up needs an even n");
  }
  return mi::linear("mi_linear_fused", a, swiglu != 0,
                    norm_weight ? mi::kLinMaxRows : mi::kLinMaxFusedRows, dtype, stream);
}
