// Projections of a few rows: y[rows, n] = x[rows, k] . w[n, k]^T in bf16, the
// shape every projection of a decode step has (rows = running sequences).
//
// Bound by reading the weight once.  One work-group per 16 outputs: its
// wavefronts split k, each lane loads its share of the 16 weight rows in
// 16-byte pieces, up to eight MFMA k-steps before any is used, so that all
// of a work-group's weight bytes (48 KB at k = 1,536) are in flight at once, and the
// partial 16 x 16 tiles are summed over the wavefronts in order through LDS.
// A library GEMM of these shapes walks k in LDS tiles.  us per call at 16 rows,
// weights from HBM, library -> this: 1,536 x 3,968 19.5 -> 10.7, 2,560 x 1,536 9.4 ->
// 5.9, 7,936 x 1,536 11.9 -> 9.6; at 8 rows, in half tiles, 19.3 -> 6.8, 9.4 -> 5.2,
// 11.9 -> 8.1 and 8,384 x 1,536 12.7 -> 8.5.
//
// The tile is W . x^T on v_mfma_f32_16x16x32_bf16 (A = 16 weight rows, B = 16
// rows of x; lanes of rows past the last read the last row, unused): a lane
// ends with four consecutive outputs of one row.  k-steps of 32 are split over
// the wavefronts as whole steps.
//
// The GLU form takes eight gate and the eight matching up columns as the 16
// weight rows, so that the activation (SiTU-GLU, blocks.py:12-27 of
// ml/runtime/model) is formed on the fp32 sums of one tile: the projection is
// neither rounded nor written.
//
// For at most eight rows half of a tile's columns would be empty.  The half-tile
// form puts eight outputs in a tile: A holds their weights at two consecutive
// k-steps (rows 0-7 and 8-15), B the rows of x at the same two, and of the
// product the two diagonal quadrants are the sums over the even and the odd
// steps.  A load then takes whole 128-byte lines of eight weight rows instead of
// half lines of sixteen, x is loaded half as often, and there are twice the
// tiles to spread over the chip (1,536 outputs are 96 tiles of 16 on 256 CUs).
// us per call in a loop of launches, whole tiles -> half: 1,536 x 3,968 7.9 -> 6.0,
// 7,936 x 1,536 with its activation 9.2 -> 7.6, 8,384 x 1,536 14.0 -> 7.5, 2,048 x 384
// 3.8 -> 2.4.
#include "common.hpp"
#include "situ.hpp"

#include "../../include/sophia_decoder.h"

namespace sophia {
namespace {

constexpr int kRlRows = 32;    // most rows of x
constexpr int kCus = 256;      // compute units of the card
constexpr int kHlBatch = 8;    // head_linear: k-steps whose loads are issued together

struct RowLinearArgs {
  const uint16_t *x;
  int64_t x_stride;
  const uint16_t *w;
  int64_t w_stride;
  uint16_t *y;
  int64_t y_stride;
  int rows;
  int64_t hidden;    // GLU: row of w where the up columns begin
  int ksteps;        // k / 32
  int64_t tiles;     // of 16 weight rows
  float rcg, rcu, scale;
};

__device__ __forceinline__ bf8 as_bf8(u4 w) { return __builtin_bit_cast(bf8, w); }

// Sums of a tile's four columns, the partial tiles of the wavefronts, to y.
template <int NW, int NT, int MT, bool GLU, bool CAP4, bool HALF>
__device__ __forceinline__ void store_tile(const RowLinearArgs &a, const f4 (&part)[NW][NT * MT][64], int nt, int mt,
                                           int lane) {
  const int ln = lane & 15, g = lane >> 4;
  const int64_t tile = static_cast<int64_t>(blockIdx.x) * NT + nt;
  if (tile >= a.tiles) return;   // wave-uniform
  f4 sum = part[0][nt * MT + mt][lane];   // weight rows 4 g + i, row 16 mt + ln
#pragma unroll
  for (int p = 1; p < NW; ++p) sum += part[p][nt * MT + mt][lane];
  constexpr int kRows = HALF ? 8 : 16;   // weight rows of a tile
  if constexpr (HALF) {
    // lanes ln < 8, g < 2 hold the even steps' sums, lanes ln + 8, g + 2 the same outputs' of the odd steps
#pragma unroll
    for (int i = 0; i < 4; ++i) sum[i] += lane_xor32(dpp_rotate<0x128>(sum[i]));
  }
  constexpr int kGroups = kRows / 4 / (GLU ? 2 : 1);   // of four outputs
  if constexpr (GLU) {
    // the first half of the tile's weight rows are gate columns, the second their up columns
    f4 up;
#pragma unroll
    for (int i = 0; i < 4; ++i) up[i] = HALF ? lane_xor16(sum[i]) : lane_xor32(sum[i]);
#pragma unroll
    for (int i = 0; i < 4; ++i) sum[i] = situ_value<CAP4>(sum[i], up[i], a.rcg, a.rcu, a.scale);
  }
  const int row = 16 * mt + ln;
  if (g < kGroups && row < a.rows)
    *reinterpret_cast<u2 *>(a.y + row * a.y_stride + 4 * (kGroups * tile + g)) =
        u2{pack_bf16x2(sum[0], sum[1]), pack_bf16x2(sum[2], sum[3])};
}

// NW wavefronts, NT tiles of outputs (sharing the loads of x), MT tiles of 16
// rows of x; loads of BATCH k-steps (HALF: pairs of steps) issued together.
template <int NW, int NT, int MT, int BATCH, bool GLU, bool CAP4, bool HALF>
__global__ __launch_bounds__(NW * 64) void row_linear_kernel(RowLinearArgs a) {
  static_assert(!HALF || MT == 1, "half tiles are for at most eight rows");
  constexpr int kRows = HALF ? 8 : 16;   // weight rows of a tile, rows of x
  __shared__ f4 s_part[NW][NT * MT][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ln = lane & (kRows - 1), g = lane >> 4;
  const int odd = HALF ? (lane >> 3) & 1 : 0;   // this lane's step of a pair
  const uint16_t *wp[NT], *xp[MT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int64_t tile = imin64(static_cast<int64_t>(blockIdx.x) * NT + nt, a.tiles - 1);   // the last again, unused
    constexpr int kCols = kRows / 2;   // GLU: gate and up columns of a tile
    const int64_t wrow = GLU ? (ln < kCols ? kCols * tile + ln : a.hidden + kCols * tile + ln - kCols) : kRows * tile + ln;
    wp[nt] = a.w + wrow * a.w_stride + 8 * g;
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
    xp[mt] = a.x + static_cast<int64_t>(min(16 * mt + ln, a.rows - 1)) * a.x_stride + 8 * g;
  const int units = HALF ? (a.ksteps + 1) / 2 : a.ksteps;   // pairs of steps, or steps
  const int per = (units + NW - 1) / NW;
  const int s0 = wave * per, s1 = min(s0 + per, units);
  f4 acc[NT][MT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[nt][mt] = f4{0.f, 0.f, 0.f, 0.f};
  for (int s = s0; s < s1; s += BATCH) {
    u4 wr[NT][BATCH], xr[MT][BATCH];
#pragma unroll
    for (int i = 0; i < BATCH; ++i) {
      const int unit = min(s + i, s1 - 1);   // past the wave's last: the last again, unused
      const int at = 32 * (HALF ? min(2 * unit + odd, a.ksteps - 1) : unit);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) wr[nt][i] = *reinterpret_cast<const u4 *>(wp[nt] + at);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) xr[mt][i] = *reinterpret_cast<const u4 *>(xp[mt] + at);
    }
    asm volatile("" ::: "memory");   // (the loads stay a batch: none is sunk to its use)
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < BATCH; ++i) {
      if (s + i >= s1) break;   // wave-uniform
      if (HALF && 2 * (s + i) + odd >= a.ksteps) {   // the step that an odd number of them lacks
        xr[0][i] = u4{0, 0, 0, 0};
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) wr[nt][i] = u4{0, 0, 0, 0};
      }
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          acc[nt][mt] =
              __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf8(wr[nt][i]), as_bf8(xr[mt][i]), acc[nt][mt], 0, 0, 0);
    }
  }
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) s_part[wave][nt * MT + mt][lane] = acc[nt][mt];
  __syncthreads();
  for (int t = wave; t < NT * MT; t += NW)   // (wave-uniform)
    store_tile<NW, NT, MT, GLU, CAP4, HALF>(a, s_part, t / MT, t % MT, lane);
}

template <int NW, int NT, int MT, int BATCH, bool GLU, bool CAP4, bool HALF>
int launch(const RowLinearArgs &a, hipStream_t st) {
  hipLaunchKernelGGL((row_linear_kernel<NW, NT, MT, BATCH, GLU, CAP4, HALF>),
                     dim3(static_cast<unsigned>((a.tiles + NT - 1) / NT)), dim3(NW * 64), 0, st, a);
  return check_launch(GLU ? "row_linear_situ_glu" : "row_linear");
}

// The loads of a batch that a wavefront's share of k does not fill are loads of
// the same bytes again, so the batch is the share where one holds it (2,048 x 384
// 3.8 -> 2.4 us, 7,936 x 1,536 9.2 -> 8.6).
template <int NW, int NT, int MT, bool GLU, bool CAP4, bool HALF>
int dispatch_batch(const RowLinearArgs &a, int units, hipStream_t st) {
  const int per = (units + NW - 1) / NW;
  if constexpr (NW == 4 || (HALF && NT > 1)) {   // else k is long: more than four steps each
    if (per <= 1) return launch<NW, NT, MT, 1, GLU, CAP4, HALF>(a, st);
    if (per <= 3) return launch<NW, NT, MT, 3, GLU, CAP4, HALF>(a, st);
  }
  // Past 128 registers of loads in a batch of eight (16 wavefronts have 128 each, two tiles each way take 16 of
  // them per step) they spilled: 32 rows of 8,192 x 3,968 33.3 us with eight, 28.4 with six, x 6,144 57.3 and 35.6.
  if constexpr (NT > 2 || NW * NT * MT > 32) {
    return launch<NW, NT, MT, 6, GLU, CAP4, HALF>(a, st);
  } else {
    if (per <= 6) return launch<NW, NT, MT, 6, GLU, CAP4, HALF>(a, st);
    return launch<NW, NT, MT, 8, GLU, CAP4, HALF>(a, st);
  }
}

// At most eight rows: half tiles, one per work-group while that leaves no CU a
// second one, else two, and five where two per work-group are more work-groups
// than two per CU (8,384 x 1,536: 7.5 us with five on 210 CUs, 8.8 with two,
// 10.1 with four on 262: a second round for six).  Past five per CU the second
// round comes with five too (8 rows: 10,240 x 1,536 8.4 us, 10,256 x 1,536 11.6),
// and a library GEMM is the faster form of most shapes.
template <bool GLU, bool CAP4>
int dispatch_half(RowLinearArgs a, hipStream_t st) {
  a.tiles *= 2;
  const int units = (a.ksteps + 1) / 2;
  if (a.tiles > 4 * kCus) return dispatch_batch<8, 5, 1, GLU, CAP4, true>(a, units, st);
  if (a.tiles > kCus) return dispatch_batch<8, 2, 1, GLU, CAP4, true>(a, units, st);
  if (units <= 32) return dispatch_batch<4, 1, 1, GLU, CAP4, true>(a, units, st);
  return dispatch_batch<8, 1, 1, GLU, CAP4, true>(a, units, st);
}

// Whole tiles: one per work-group while that leaves no CU a second one, else
// two, which share their loads of x (7,936 outputs, k = 1,536, 16 rows: 11.0 us
// with one tile, 9.7 with two, four on 124 CUs 13.8).
template <int NW, int MT, bool GLU, bool CAP4>
int dispatch_tiles(const RowLinearArgs &a, hipStream_t st) {
  if (a.tiles > kCus) return dispatch_batch<NW, 2, MT, GLU, CAP4, false>(a, a.ksteps, st);
  return dispatch_batch<NW, 1, MT, GLU, CAP4, false>(a, a.ksteps, st);
}

// Wavefronts so that one batch holds a wavefront's share of k: 4 up to k =
// 1,024, 8 up to 2,048, 16 beyond.
template <bool GLU, bool CAP4>
int dispatch(const RowLinearArgs &a, hipStream_t st) {
  if (a.rows <= 8) return dispatch_half<GLU, CAP4>(a, st);
  const int need = (a.ksteps + 7) / 8;
  if (a.rows <= 16) {
    if (need <= 4) return dispatch_tiles<4, 1, GLU, CAP4>(a, st);
    if (need <= 8) return dispatch_tiles<8, 1, GLU, CAP4>(a, st);
    return dispatch_tiles<16, 1, GLU, CAP4>(a, st);
  }
  if (need <= 4) return dispatch_tiles<4, 2, GLU, CAP4>(a, st);
  if (need <= 8) return dispatch_tiles<8, 2, GLU, CAP4>(a, st);
  return dispatch_tiles<16, 2, GLU, CAP4>(a, st);
}

// y[row, h, :] = x[row, h, :] . w[h]^T for every head h: MLA's products of the
// decode rows with the per-head blocks of k_up and v_up.  One work-group per
// (16 rows, head, 128 outputs), a wavefront per 16 outputs over all of k, its
// loads eight k-steps at a time.  At 8 rows x 16 heads x 128 x 128 one launch
// of 5 us takes the place of a batched library GEMM (7.8 us) and the two
// transposing copies around it (4.6 us each).  With a gate the output is
// multiplied by its sigmoid (attention.py:655-656), rounded to bf16 before and
// after as two launches round it: a launch of 4.5 us less.
//
// KN: w[h] lies as [k, n], k_up's block as its weight holds it (the product
// contracts over the head's rows).  128 of its rows at a time go to LDS as whole
// lines and come back by transposing reads, four of a column per lane: the same
// operands, steps and sums as over a transposed copy, no copy to keep in step
// with the weight, and whole lines of it (16 heads x 128 x 128 in a loop of
// launches: 8 rows 4.2 us over the copy, 2.4 here; 1,024 rows 16.1 and 6.8).
struct HeadLinearArgs {
  const uint16_t *x;
  int64_t x_row, x_head;
  const uint16_t *w;
  uint16_t *y;
  int64_t y_row, y_head;
  const uint16_t *gate;   // logits like y, or NULL
  int64_t gate_row, gate_head;
  int rows, n, ksteps;
};

constexpr int kHlWaves = 8;
constexpr int kHlCols = 16 * kHlWaves;   // outputs of a work-group
constexpr int kHlK = 128;                // KN: rows of w in LDS at a time
constexpr int kHlLd = kHlCols + 8;       // bf16 row stride there

// KN: rows k0 .. k0 + kHlK - 1 of w[h] (past the last: the last again, unused),
// the columns of this work-group (past the last: the last again, unused).
__device__ __forceinline__ void stage_head_rows(const HeadLinearArgs &a, int h, int col0, int k0, uint16_t *s_w) {
  constexpr int kChunks = kHlCols / 8, kRows = kHlWaves * 64 / kChunks;   // 16-byte chunks of a row, rows at a time
  const int c = threadIdx.x % kChunks, r = threadIdx.x / kChunks;
  const int64_t k = 32 * static_cast<int64_t>(a.ksteps);
  const uint16_t *wp = a.w + static_cast<int64_t>(h) * k * a.n + min(col0 + 8 * c, a.n - 8);
  u4 v[kHlK / kRows];
#pragma unroll
  for (int i = 0; i < kHlK / kRows; ++i)
    v[i] = *reinterpret_cast<const u4 *>(wp + imin64(k0 + r + i * kRows, k - 1) * a.n);
#pragma unroll
  for (int i = 0; i < kHlK / kRows; ++i) *reinterpret_cast<u4 *>(s_w + (r + i * kRows) * kHlLd + 8 * c) = v[i];
}

template <bool KN>
__global__ __launch_bounds__(kHlWaves * 64) void head_linear_kernel(HeadLinearArgs a) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ln = lane & 15, g = lane >> 4;
  const int h = blockIdx.y, n0 = kHlCols * blockIdx.z + 16 * wave;
  if (!KN && n0 >= a.n) return;   // wave-uniform; no barrier below
  const int row = blockIdx.x * 16 + ln;
  const uint16_t *xp = a.x + min(row, a.rows - 1) * a.x_row + h * a.x_head + 8 * g;
  u2 gate = u2{0, 0};
  if (a.gate && n0 < a.n)   // uniform
    gate = *reinterpret_cast<const u2 *>(a.gate + min(row, a.rows - 1) * a.gate_row + h * a.gate_head + n0 + 4 * g);
  f4 acc = f4{0.f, 0.f, 0.f, 0.f};
  if constexpr (KN) {
    __shared__ __attribute__((aligned(16))) uint16_t s_w[kHlK * kHlLd];
    // rows 8 g + ln / 4 of a step (and four on) at this wavefront's columns: A's lane (output ln, k 8 g ..)
    const uint16_t *sp = s_w + (8 * g + (ln >> 2)) * kHlLd + 16 * wave + 4 * (ln & 3);
    constexpr int kSteps = kHlK / 32;
    for (int s = 0; s < a.ksteps; s += kSteps) {
      u4 xr[kSteps];
#pragma unroll
      for (int i = 0; i < kSteps; ++i) xr[i] = *reinterpret_cast<const u4 *>(xp + 32 * min(s + i, a.ksteps - 1));
      if (s > 0) __syncthreads();   // the rows before are read
      stage_head_rows(a, h, kHlCols * blockIdx.z, 32 * s, s_w);
      __syncthreads();
#pragma unroll
      for (int i = 0; i < kSteps; ++i) {
        if (s + i >= a.ksteps) break;   // uniform
        const u2 lo = lds_read_tr(sp + 32 * i * kHlLd), hi = lds_read_tr(sp + (32 * i + 4) * kHlLd);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf8(u4{lo.x, lo.y, hi.x, hi.y}), as_bf8(xr[i]), acc, 0, 0, 0);
      }
    }
    if (n0 >= a.n) return;   // (after the last barrier)
  } else {
    const uint16_t *wp = a.w + (static_cast<int64_t>(h) * a.n + n0 + ln) * (32 * static_cast<int64_t>(a.ksteps)) + 8 * g;
    for (int s = 0; s < a.ksteps; s += kHlBatch) {
      u4 wr[kHlBatch], xr[kHlBatch];
#pragma unroll
      for (int i = 0; i < kHlBatch; ++i) {
        const int at = 32 * min(s + i, a.ksteps - 1);
        wr[i] = *reinterpret_cast<const u4 *>(wp + at);
        xr[i] = *reinterpret_cast<const u4 *>(xp + at);
      }
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < kHlBatch; ++i) {
        if (s + i >= a.ksteps) break;
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf8(wr[i]), as_bf8(xr[i]), acc, 0, 0, 0);
      }
    }
  }
  if (a.gate) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float logit = __uint_as_float(i % 2 ? gate[i / 2] & 0xffff0000u : gate[i / 2] << 16);
      acc[i] = as_dtype(acc[i], SOPHIA_DTYPE_BF16) *
               __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.44269504088896341f * logit));
    }
  }
  if (row < a.rows)
    *reinterpret_cast<u2 *>(a.y + row * a.y_row + h * a.y_head + n0 + 4 * g) =
        u2{pack_bf16x2(acc[0], acc[1]), pack_bf16x2(acc[2], acc[3])};
}

int check(const char *what, const void *x, int64_t x_stride, const void *w, int64_t w_stride, const void *y,
          int64_t y_stride, int64_t rows, int64_t outputs, int64_t weight_rows, int64_t k) {
  SOPHIA_REQUIRE(rows >= 0 && rows <= kRlRows, "%s: rows must be in [0, %d]", what, kRlRows);
  SOPHIA_REQUIRE(k > 0 && k % 32 == 0 && k <= (int64_t{1} << 30), "%s: k must be a positive multiple of 32", what);
  SOPHIA_REQUIRE(weight_rows > 0 && weight_rows % 16 == 0 && weight_rows / 16 <= 0x7fffffff,
                 "%s: n must be a positive multiple of 16", what);
  SOPHIA_REQUIRE(x_stride >= k && w_stride >= k && y_stride >= outputs && x_stride % 8 == 0 && w_stride % 8 == 0 &&
                     y_stride % 4 == 0,
                 "%s: bad strides", what);
  SOPHIA_REQUIRE(rows == 0 || (x && w && y), "%s: NULL pointer", what);
  SOPHIA_REQUIRE(reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0 &&
                     reinterpret_cast<uintptr_t>(y) % 8 == 0,
                 "%s: x and w must be 16-byte and y 8-byte aligned", what);
  return SOPHIA_OK;
}

}  // namespace
}  // namespace sophia

using namespace sophia;

extern "C" int sophia_row_linear(const void *x, int64_t x_stride, const void *w, int64_t w_stride, void *y,
                                 int64_t y_stride, int64_t rows, int64_t n, int64_t k, void *stream) {
  if (const int rc = check("row_linear", x, x_stride, w, w_stride, y, y_stride, rows, n, n, k)) return rc;
  if (rows == 0) return SOPHIA_OK;
  const RowLinearArgs a{static_cast<const uint16_t *>(x), x_stride, static_cast<const uint16_t *>(w), w_stride,
                        static_cast<uint16_t *>(y), y_stride, static_cast<int>(rows), 0, static_cast<int>(k / 32),
                        n / 16, 0.f, 0.f, 0.f};
  return dispatch<false, false>(a, static_cast<hipStream_t>(stream));
}

extern "C" int sophia_row_linear_situ_glu(const void *x, int64_t x_stride, const void *w, int64_t w_stride, void *h,
                                          int64_t h_stride, int64_t rows, int64_t hidden, int64_t k,
                                          float gate_softcap, float up_softcap, void *stream) {
  if (const int rc = check("row_linear_situ_glu", x, x_stride, w, w_stride, h, h_stride, rows, hidden, 2 * hidden, k))
    return rc;
  SOPHIA_REQUIRE(gate_softcap > 0.f && up_softcap > 0.f, "row_linear_situ_glu: soft caps must be positive");
  if (rows == 0) return SOPHIA_OK;
  const RowLinearArgs a{static_cast<const uint16_t *>(x), x_stride, static_cast<const uint16_t *>(w), w_stride,
                        static_cast<uint16_t *>(h), h_stride, static_cast<int>(rows), hidden,
                        static_cast<int>(k / 32), hidden / 8, 1.0f / gate_softcap, 1.0f / up_softcap, gate_softcap * up_softcap};
  if (gate_softcap == 4.0f) return dispatch<true, true>(a, static_cast<hipStream_t>(stream));
  return dispatch<true, false>(a, static_cast<hipStream_t>(stream));
}

namespace {
template <bool KN>
int head_linear(const void *x, int64_t x_row_stride, int64_t x_head_stride, const void *w, void *y, int64_t y_row_stride,
                int64_t y_head_stride, const void *gate, int64_t gate_row_stride, int64_t gate_head_stride, int64_t rows,
                int heads, int n, int k, void *stream) {
  SOPHIA_REQUIRE(rows >= 0 && rows <= 0x7fffffff && heads > 0 && heads <= 65535, "head_linear: bad rows / heads");
  SOPHIA_REQUIRE(k > 0 && k % 32 == 0 && n > 0 && n % 16 == 0 && (n + 127) / 128 <= 65535,
                 "head_linear: k must be a positive multiple of 32 and n of 16");
  SOPHIA_REQUIRE(x_head_stride >= k && y_head_stride >= n && x_row_stride >= (heads - 1) * x_head_stride + k &&
                     y_row_stride >= (heads - 1) * y_head_stride + n && x_row_stride % 8 == 0 && x_head_stride % 8 == 0 &&
                     y_row_stride % 4 == 0 && y_head_stride % 4 == 0,
                 "head_linear: bad strides");
  SOPHIA_REQUIRE(rows == 0 || (x && w && y), "head_linear: NULL pointer");
  SOPHIA_REQUIRE(reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0 &&
                     reinterpret_cast<uintptr_t>(y) % 8 == 0,
                 "head_linear: x and w must be 16-byte and y 8-byte aligned");
  SOPHIA_REQUIRE(!gate || (gate_head_stride >= n && gate_row_stride >= (heads - 1) * gate_head_stride + n &&
                           gate_row_stride % 4 == 0 && gate_head_stride % 4 == 0 &&
                           reinterpret_cast<uintptr_t>(gate) % 8 == 0),
                 "head_linear: bad gate strides or alignment");
  if (rows == 0) return SOPHIA_OK;
  const HeadLinearArgs a{static_cast<const uint16_t *>(x), x_row_stride, x_head_stride, static_cast<const uint16_t *>(w),
                         static_cast<uint16_t *>(y), y_row_stride, y_head_stride, static_cast<const uint16_t *>(gate),
                         gate_row_stride, gate_head_stride, static_cast<int>(rows), n, k / 32};
  const dim3 grid(static_cast<unsigned>((rows + 15) / 16), static_cast<unsigned>(heads),
                  static_cast<unsigned>((n + 127) / 128));
  hipLaunchKernelGGL(head_linear_kernel<KN>, grid, dim3(kHlWaves * 64), 0, static_cast<hipStream_t>(stream), a);
  return check_launch("head_linear");
}
}  // namespace

extern "C" int sophia_head_linear(const void *x, int64_t x_row_stride, int64_t x_head_stride, const void *w, void *y,
                                  int64_t y_row_stride, int64_t y_head_stride, const void *gate,
                                  int64_t gate_row_stride, int64_t gate_head_stride, int64_t rows, int heads, int n, int k,
                                  void *stream) {
  return head_linear<false>(x, x_row_stride, x_head_stride, w, y, y_row_stride, y_head_stride, gate, gate_row_stride,
                            gate_head_stride, rows, heads, n, k, stream);
}

extern "C" int sophia_head_linear_kn(const void *x, int64_t x_row_stride, int64_t x_head_stride, const void *w, void *y,
                                     int64_t y_row_stride, int64_t y_head_stride, int64_t rows, int heads, int n, int k,
                                     void *stream) {
  return head_linear<true>(x, x_row_stride, x_head_stride, w, y, y_row_stride, y_head_stride, nullptr, n,
                           static_cast<int64_t>(heads) * n, rows, heads, n, k, stream);
}
