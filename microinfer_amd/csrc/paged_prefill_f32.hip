// Paged / contiguous varlen attention for float32 with head_dim 128 on the
// float32 MFMA (gfx950).
//
// Covers the float32 rows of _paged_prefill_kernel
// (microinfer/layer/triton_paged_attention.py:134-233) and of the reference
// fallback (microinfer/layer/paged_attention.py:22-67). Inputs, probabilities
// and sums all stay float32: v_mfma_f32_16x16x4_f32 multiplies and adds in it.
//
// What bounds it: the matrix cores (157 TFLOP/s nominal in float32, 137
// measured on a 4096^3 library product). The vector kernel this replaces for
// these shapes spends one 8-wave workgroup on every (query row, KV head), so
// each row streams the whole context for itself.
//
// Design:
//  * Workgroup = 16 rows of one request's flattened (token, query head of the
//    group) rows x one KV head. Its NW waves take the 16-key tiles in turn
//    (wave w: tiles w, w + NW, ...), each with an online softmax of its own,
//    and are merged through LDS once at the end: small chunks still give
//    every SIMD work, and no barrier sits in the loop.
//  * Fragments go from memory straight to the registers in MFMA layout, as
//    16-byte loads, because the contraction index may be numbered freely:
//    S^T = K . Q^T takes k-step (j, e) as dims 16 j + 4 quad + e (lane: key
//    or query row `col`, the float4 at 16 j + 4 quad); O^T = V^T . P^T takes
//    k-step i as keys 4 quad + i -- where S^T left them -- and output block
//    (j, e) as dims 64 j + 4 col + e (lane: V row 4 quad + i, the float4 at
//    64 j + 4 col). Nothing is staged, transposed or shuffled.
//  * A tile's V is issued before its scores, the next tile's K as soon as the
//    scores have used the registers: each half hides the other's loads.
//
// Chunks of 118 / 325 / 210 rows on contexts of 155 / 325 / 359 (16 / 8
// heads), a pass of four layers: 27.3 us a launch, 76.5 on the vector kernel;
// 1000 rows on 1700 keys: 138 us, 71 TFLOP/s. Error against 64 bits, geometric
// mean over 25 cases of 8 to 937 rows on up to 1100 keys: 1.196e-7, the vector
// kernel's 1.201e-7, through short summation chains, a score scaled and its
// maximum subtracted in one rounding, and a division at the end (one chain of
// 16 for a tile's P.V, two roundings and a reciprocal: 1.31e-7).
#include "paged_attention.h"

namespace mi {
namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int kD = 128;
constexpr int kRows = 16;  // query rows per workgroup, keys per tile
constexpr int kOutStride = kD + 4;  // LDS row of a wave's sums: 16 rows hit 16 bank groups
constexpr float kSlack = 8.f;  // the running maximum may lag by 2^8

template <int NW, bool PAGED>
__global__ __launch_bounds__(kWave * NW, 2) void paged_prefill_f32_kernel(const AttnArgs a) {
  __shared__ __attribute__((aligned(16))) float s_o[NW][kRows * kOutStride];
  __shared__ float s_m[NW][kRows];
  __shared__ float s_l[NW][kRows];
  using ConstI32 = __attribute__((address_space(4))) const int32_t;

  const int tid = threadIdx.x;
  const int lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int col = lane % 16;
  const int quad = lane / 16;
  const int head = blockIdx.x % a.num_kv_heads;
  const int G = a.group;

  // Row tile -> (request, tile of it): a scan of the requests' tile counts,
  // 64 at a time. Later tiles (longer contexts) get the earlier workgroups.
  int tile = gridDim.x / a.num_kv_heads - 1 - blockIdx.x / a.num_kv_heads;
  int req = -1;
  for (int r0 = 0; r0 < a.num_seqs; r0 += kWave) {
    const int r = r0 + lane;
    int n = 0;
    if (r < a.num_seqs) n = (max(a.cu_q[r + 1] - a.cu_q[r], 0) * G + kRows - 1) / kRows;
    const int end = wave_inclusive_scan(n, lane);
    const uint64_t past = __ballot(tile < end);
    if (past != 0) {
      const int hit = __ffsll(static_cast<unsigned long long>(past)) - 1;
      tile -= __shfl(end - n, hit, kWave);
      req = r0 + hit;
      break;
    }
    tile -= __shfl(end, kWave - 1, kWave);
  }
  req = __builtin_amdgcn_readfirstlane(req);
  tile = __builtin_amdgcn_readfirstlane(tile);
  if (req < 0) return;  // past the last tile (uniform across the workgroup)

  const int q0 = a.cu_q[req];
  const int q_len = a.cu_q[req + 1] - q0;
  const int ctx = a.cu_k[req + 1] - a.cu_k[req];
  const int rows = q_len * G;
  const int row = tile * kRows + col;  // this lane's query row (MFMA column)
  const bool row_ok = row < rows && q0 + row / G < a.num_rows;
  const int row_c = row_ok ? row : 0;
  // Keys the cache can hold for this request.
  const int64_t key_row0 = PAGED ? 0 : a.cu_k[req];
  const int capacity =
      PAGED ? a.t_width * a.block_size
            : static_cast<int>(max<int64_t>(0, min<int64_t>(a.num_blocks - key_row0, ctx)));
  const int prefix = ctx - q_len;
  const int limit = row_ok ? min(prefix + row_c / G + 1, capacity) : 0;  // keys this row sees
  const int tok_lo = tile * kRows / G;
  const int tok_hi = min(tile * kRows + kRows - 1, rows - 1) / G;
  // Keys any row sees, and keys every row sees.
  const int keys = __builtin_amdgcn_readfirstlane(max(0, min(prefix + tok_hi + 1, capacity)));
  const int keys_all = __builtin_amdgcn_readfirstlane(min(prefix + tok_lo + 1, capacity));
  const int ntiles = (keys + kRows - 1) / kRows;

  const float* kc = static_cast<const float*>(a.kc) + head * a.c_hs;
  const float* vc = static_cast<const float*>(a.vc) + head * a.c_hs;
  const ConstI32* ctab = (const ConstI32*)(PAGED ? a.tables + req * a.t_stride : nullptr);

  // Block id of tile t (a scalar load; its result is used later), then the
  // element offset of its first row and whether it may be read (an invalid
  // block reads block 0 and is masked).
  auto tile_block = [&](int t) -> int { return PAGED ? ctab[(t * kRows) >> a.log2_block] : 0; };
  auto tile_base = [&](int t, int blk, bool& ok) -> int64_t {
    const int p0 = t * kRows;
    ok = !PAGED || (blk >= 0 && blk < a.num_blocks);
    if constexpr (!PAGED) return (key_row0 + p0) * a.c_ts;
    return ok ? blk * a.c_bs + (p0 & (a.block_size - 1)) * a.c_ts : 0;
  };
  // Per-lane offsets from a tile's first row (32 bits over a scalar base).
  // Paged tiles lie in one block; a contiguous request's last tile must not
  // read past its keys, so those rows repeat the last one (masked).
  const uint32_t c_ts = static_cast<uint32_t>(a.c_ts);
  auto in_tile = [&](int t, int r) -> uint32_t {
    return PAGED ? r : min(r, keys - 1 - t * kRows);
  };
  auto load_k = [&](f32x4_t (&kf)[8], int t, int64_t base) {
    const float* p = kc + base;
    const uint32_t off = in_tile(t, col) * c_ts + 4 * quad;
#pragma unroll
    for (int j = 0; j < 8; ++j) kf[j] = *reinterpret_cast<const f32x4_t*>(p + off + 16 * j);
  };

  f32x4_t qf[8];
  {
    const float* p = static_cast<const float*>(a.q) + (q0 + row_c / G) * a.q_ts +
                     (head * G + row_c % G) * a.q_hs + 4 * quad;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const f32x4_t v = *reinterpret_cast<const f32x4_t*>(p + 16 * j);
      qf[j] = row_ok ? v : f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
  }

  f32x4_t o[8];
#pragma unroll
  for (int b = 0; b < 8; ++b) o[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;

  int nonfinite = 0;
  f32x4_t kf[8];
  bool ok = false;
  int64_t base = 0;
  if (wave < ntiles) {
    base = tile_base(wave, tile_block(wave), ok);
    load_k(kf, wave, base);
  }
  for (int t = wave; t < ntiles; t += NW) {
    const int p0 = t * kRows;
    const int next = min(t + NW, ntiles - 1);
    const int next_blk = tile_block(next);
    f32x4_t vf[4][2];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float* p = vc + base + (PAGED ? i * a.c_ts : 0);
      const uint32_t off = (PAGED ? 4 * quad : in_tile(t, 4 * quad + i)) * c_ts + 4 * col;
      vf[i][0] = *reinterpret_cast<const f32x4_t*>(p + off);
      vf[i][1] = *reinterpret_cast<const f32x4_t*>(p + off + 64);
    }
    // The compiler would sink these loads below the products that hide them.
    __builtin_amdgcn_sched_barrier(0);
    // Eight chains of 16 terms, added as a tree: a score's rounding error is
    // that of short sums.
    f32x4_t s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      f32x4_t c[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) c[e] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 4 * h; j < 4 * h + 4; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          c[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[j][e], qf[j][e], c[e], 0, 0, 0);
      s += (c[0] + c[1]) + (c[2] + c[3]);
    }
    // Unconditional (the last round repeats the last tile): the waits below
    // then count these loads as in flight on every path.
    bool next_ok;
    const int64_t next_base = tile_base(next, next_blk, next_ok);
    load_k(kf, next, next_base);
    __builtin_amdgcn_sched_barrier(0);
    // s[i]: key p0 + 4 quad + i, query row `col`.
    const bool masked = !ok || p0 + kRows > keys_all;  // uniform
    const int lim = masked ? (ok ? limit : 0) : INT32_MAX;
    float tmax = -INFINITY;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (p0 + 4 * quad + i >= lim) s[i] = -INFINITY;
      tmax = fmaxf(tmax, s[i] * a.scale_log2);
    }
    tmax = fmaxf(tmax, lane_xor16(tmax, lane));
    tmax = fmaxf(tmax, lane_xor32(tmax, lane));
    if (__ballot(tmax > m + kSlack) != 0) {
      const float mnew = fmaxf(m, tmax);
      const float alpha = mnew == -INFINITY ? 1.f : fast_exp2(m - mnew);
      l *= alpha;
#pragma unroll
      for (int b = 0; b < 8; ++b) o[b] *= alpha;
      m = mnew;
    }
    const float base_m = m == -INFINITY ? 0.f : m;
    float pr[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) pr[i] = fast_exp2(fmaf(s[i], a.scale_log2, -base_m));
    l += (pr[0] + pr[1]) + (pr[2] + pr[3]);
    if (masked) {
      // A key no row sees weighs 0, but 0 * NaN is NaN: its V becomes 0. A
      // non-finite V that only some rows see must not reach the others: the
      // workgroup then takes its rows one by one, below.
      bool odd = false;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const bool seen = ok && p0 + 4 * quad + i < keys;
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float v = seen ? vf[i][j][e] : 0.f;
            vf[i][j][e] = v;
            odd |= !(fabsf(v) < INFINITY);
          }
      }
      if (__ballot(odd) != 0) {
        nonfinite = 1;
        break;
      }
    }
    // The tile's own sums, in two halves, then added to the running ones
    // (short chains again). Two of four blocks at a time: with all four the
    // kernel passes 168 registers, a wave less per SIMD and 15 % more time.
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e0 = 0; e0 < 4; e0 += 2) {
        f32x4_t c[2][2];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int e = 0; e < 2; ++e) c[h][e] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int e = 0; e < 2; ++e)
              c[h][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[2 * h + i][j][e0 + e],
                                                             pr[2 * h + i], c[h][e], 0, 0, 0);
#pragma unroll
        for (int e = 0; e < 2; ++e) o[4 * j + e0 + e] += c[0][e] + c[1][e];
      }
    ok = next_ok;
    base = next_base;
  }

  if (__syncthreads_or(nonfinite)) {
    for (int r = wave; r < kRows; r += NW) {
      const int rr = tile * kRows + r;
      if (rr >= rows || q0 + rr / G >= a.num_rows) continue;
      const int64_t qo = (q0 + rr / G) * a.q_ts + (head * G + rr % G) * a.q_hs + 2 * lane;
      const float qa = static_cast<const float*>(a.q)[qo];
      const float qb = static_cast<const float*>(a.q)[qo + 1];
      const int seen = min(prefix + rr / G + 1, capacity);
      float mr = -INFINITY, lr = 0.f, oa = 0.f, ob = 0.f;
      for (int p = 0; p < seen; ++p) {
        bool ok;
        const int64_t off =
            tile_base(p / kRows, tile_block(p / kRows), ok) + p % kRows * a.c_ts + 2 * lane;
        if (!ok) continue;
        const float sc = xor_sum<1, kWave>(fmaf(qb, kc[off + 1], qa * kc[off])) * a.scale_log2;
        const float mnew = fmaxf(mr, sc);
        const float base_r = mnew == -INFINITY ? 0.f : mnew;  // -inf scores weigh 0
        const float alpha = fast_exp2(mr - base_r);
        const float w = fast_exp2(sc - base_r);
        mr = mnew;
        lr = fmaf(lr, alpha, w);
        oa = fmaf(w, vc[off], oa * alpha);
        ob = fmaf(w, vc[off + 1], ob * alpha);
      }
      const float inv = lr > 0.f ? 1.f / lr : 0.f;
      float* out = static_cast<float*>(a.out) + (q0 + rr / G) * a.o_ts +
                   (head * G + rr % G) * a.o_hs + 2 * lane;
      out[0] = oa * inv;
      out[1] = ob * inv;
    }
    return;
  }

  // Merge the waves. o[4 j + e][i] is dim 64 j + 16 quad + 4 i + e of row `col`.
  l += lane_xor16(l, lane);
  l += lane_xor32(l, lane);
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      *reinterpret_cast<f32x4_t*>(&s_o[wave][col * kOutStride + 64 * j + 16 * quad + 4 * i]) =
          f32x4_t{o[4 * j][i], o[4 * j + 1][i], o[4 * j + 2][i], o[4 * j + 3][i]};
  if (lane < kRows) {
    s_m[wave][lane] = m;
    s_l[wave][lane] = l;
  }
  __syncthreads();
  for (int v = tid; v < kRows * kD / 4; v += kWave * NW) {
    const int r = v / (kD / 4), d = 4 * (v % (kD / 4));
    const int rr = tile * kRows + r;
    if (rr >= rows || q0 + rr / G >= a.num_rows) continue;
    float mx = -INFINITY;
#pragma unroll
    for (int w = 0; w < NW; ++w) mx = fmaxf(mx, s_m[w][r]);
    f32x4_t sum = {0.f, 0.f, 0.f, 0.f};
    float ls = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float mw = s_m[w][r];
      const float f = mw == -INFINITY ? 0.f : fast_exp2(mw - mx);
      ls = fmaf(f, s_l[w][r], ls);
      const f32x4_t part = *reinterpret_cast<const f32x4_t*>(&s_o[w][r * kOutStride + d]);
#pragma unroll
      for (int e = 0; e < 4; ++e) sum[e] = fmaf(f, part[e], sum[e]);
    }
    f32x4_t out;
#pragma unroll
    for (int e = 0; e < 4; ++e) out[e] = ls > 0.f ? sum[e] / ls : 0.f;
    *reinterpret_cast<f32x4_t*>(static_cast<float*>(a.out) + (q0 + rr / G) * a.o_ts +
                                (head * G + rr % G) * a.o_hs + d) = out;
  }
}

template <int NW>
void launch(const AttnArgs& a, uint32_t grid, hipStream_t stream) {
  if (a.tables != nullptr)
    paged_prefill_f32_kernel<NW, true><<<grid, kWave * NW, 0, stream>>>(a);
  else
    paged_prefill_f32_kernel<NW, false><<<grid, kWave * NW, 0, stream>>>(a);
}

}  // namespace

bool prefill_f32_supported(const AttnArgs& a, int32_t dtype) {
  return dtype == MI_DTYPE_F32 && a.varlen && a.head_dim == kD && a.group >= 1 &&
         (a.tables == nullptr || a.block_size >= kRows) && a.c_ts >= 0 &&
         a.c_ts * kRows < (int64_t(1) << 28) &&
         (static_cast<int64_t>(a.num_rows) * a.group / kRows + a.num_seqs) * a.num_kv_heads <
             (int64_t(1) << 31);
}

// Few rows go to the vector kernel: a workgroup per (row, KV head) whose waves
// share the keys fills the chip where tiles of 16 rows leave most of it idle.
// It needs a round per CU's worth of workgroups and reads K and V once for
// each, so its reach falls with the group (heads on one read), the rounds and
// the keys. Measured, us a launch, vector / MFMA, 8 KV heads:
//   one head a group: 8 rows, 256 keys 8.5 / 14.1, 4000 keys 64 / 96; 48 rows
//     128 / 512 / 1024 keys 8.4 / 11.9, 18.7 / 20.9, 31.3 / 32.6, 4000 keys
//     100 / 96; 128 rows 128 / 256 keys 11.4 / 11.9, 18.1 / 15.2;
//   two: 32 rows, 4000 keys 78 / 98; 64 rows 256 / 512 keys 13.9 / 15.2, 22.5
//     / 21.1; 80 rows, 128 keys 12.2 / 11.9;
//   four: 32 rows 256 / 512 keys 14.5 / 15.6, 22.3 / 21.1; 40 rows, 64 keys
//     11.2 / 9.6. Eight: MFMA from 16 keys on (9.4 / 9.3).
// At 2 KV heads, the same workgroups, likewise, except that the rows of a
// request then lie on several XCDs and each reads its K and V for itself: many
// requests of 4 rows and 300 keys, 128 / 192 / 256 / 320 workgroups 11.7 /
// 15.2, 14.3 / 15.3, 16.9 / 15.4, 21 / 15.7 (8 KV heads, 320: 13.7 / 15.8).
// The keys are the most that the table or the rows can hold: the contexts are
// on the device.
bool prefill_f32_preferred(const AttnArgs& a) {
  const int64_t groups = static_cast<int64_t>(a.num_rows) * a.num_kv_heads;
  if (a.num_kv_heads % 8 != 0 && a.num_seqs > 8 && 4 * groups > 3 * device_cus()) return true;
  const int64_t rounds = (groups + device_cus() - 1) / device_cus();
  const int64_t keys = a.tables != nullptr ? static_cast<int64_t>(a.t_width) * a.block_size
                                           : static_cast<int64_t>(a.num_blocks);
  if (a.group == 1) return rounds > 1 && keys > (rounds <= 2 ? 1024 : rounds <= 4 ? 128 : 0);
  if (a.group == 2) return rounds > 1 && keys > (rounds <= 2 ? 256 : 0);
  if (a.group == 4) return rounds > 1 || keys > 256;
  return true;
}

int32_t launch_prefill_f32(const AttnArgs& a, hipStream_t stream) {
  // Every request's rows / 16, rounded up, fit in this many tiles.
  const int64_t tiles = static_cast<int64_t>(a.num_rows) * a.group / kRows + a.num_seqs;
  const uint32_t grid = static_cast<uint32_t>(tiles * a.num_kv_heads);
  // At most a workgroup per CU: eight waves share a tile, so that its keys
  // take half the rounds (two waves then fill each SIMD, and a second
  // workgroup would only wait for them).
  if (static_cast<int64_t>(grid) <= device_cus())
    launch<8>(a, grid, stream);
  else
    launch<4>(a, grid, stream);
  return check_launch("paged prefill (float32)");
}

}  // namespace mi
