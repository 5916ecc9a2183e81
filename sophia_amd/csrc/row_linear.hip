// Projections of a few rows: y[rows, n] = x[rows, k] . w[n, k]^T in bf16, the
// shape every projection of a decode step has (rows = running sequences).
//
// Bound by reading the weight once.  One work-group per 16 outputs: its
// wavefronts split k, each lane loads its share of the 16 weight rows in
// 16-byte pieces, eight MFMA k-steps at a time before any is used, so that all
// of a work-group's weight bytes (48 KB at k = 1,536) are in flight at once, and the
// partial 16 x 16 tiles are summed over the wavefronts in order through LDS.
// A library GEMM of these shapes walks k in LDS tiles.  us per call at 8 rows,
// weights from HBM, library -> this: 1,536 x 3,968 15.2 -> 8.1, 1,536 x 2,048 8.2 ->
// 5.2, 2,560 x 1,536 7.2 -> 5.1, 7,936 x 1,536 10.7 -> 8.8 (with its activation, 15.7
// -> 9.4), 2,048 x 128 3.4 -> 3.1.
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
// For at most eight rows half of a tile's columns would be empty, and 1,536
// outputs are 96 tiles on 256 CUs.  The half-tile form puts eight outputs in a
// work-group: A holds their weights over two parts of k (rows 0-7 and 8-15), B
// the rows of x over the same two parts, and of the product the two diagonal
// quadrants are the sums over the parts.  Twice the work-groups, the same bytes
// per load instruction: under the profiler 1,536 x 3,968 9.0 -> 7.3 us, 1,536 x
// 2,048 5.3 -> 4.8.
#include "common.hpp"
#include "situ.hpp"

#include "../../include/sophia_decoder.h"

namespace sophia {
namespace {

constexpr int kRlRows = 32;    // most rows of x
constexpr int kRlBatch = 8;    // k-steps whose loads are issued together

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

// NW wavefronts, NT tiles of outputs (sharing the loads of x), MT tiles of 16
// rows of x.  HALF: eight outputs per tile for at most eight rows, k split over
// 2 NW parts, a lane's part by its half of the 16.
template <int NW, int NT, int MT, bool GLU, bool CAP4, bool HALF>
__global__ __launch_bounds__(NW * 64) void row_linear_kernel(RowLinearArgs a) {
  __shared__ f4 s_part[NW][NT * MT][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ln = lane & 15, g = lane >> 4;
  static_assert(!HALF || (MT == 1 && !GLU), "half tiles: at most eight rows, plain outputs");
  constexpr int kOut = HALF ? 8 : 16;   // outputs per tile
  const uint16_t *wp[NT], *xp[MT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int64_t tile = imin64(static_cast<int64_t>(blockIdx.x) * NT + nt, a.tiles - 1);   // the last again, unused
    const int64_t wrow = GLU ? (ln < 8 ? 8 * tile + ln : a.hidden + 8 * tile + ln - 8) : kOut * tile + ln % kOut;
    wp[nt] = a.w + wrow * a.w_stride + 8 * g;
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
    xp[mt] = a.x + static_cast<int64_t>(min(16 * mt + ln % kOut, a.rows - 1)) * a.x_stride + 8 * g;
  constexpr int kParts = HALF ? 2 * NW : NW;
  const int per = (a.ksteps + kParts - 1) / kParts;
  const int s0 = (HALF ? 2 * wave + ln / 8 : wave) * per, s1 = min(s0 + per, a.ksteps);
  f4 acc[NT][MT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[nt][mt] = f4{0.f, 0.f, 0.f, 0.f};
  // (HALF: the bounds differ between the lanes' halves, the trip count is the
  // same; loads past a part's end are inside the row and replaced by zeros.)
  for (int s = s0; HALF ? s < s0 + per : s < s1; s += kRlBatch) {
    u4 wr[NT][kRlBatch], xr[MT][kRlBatch];
#pragma unroll
    for (int i = 0; i < kRlBatch; ++i) {
      const int at = 32 * min(s + i, (HALF ? a.ksteps : s1) - 1);   // past the wave's last step: the last again, unused
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) wr[nt][i] = *reinterpret_cast<const u4 *>(wp[nt] + at);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) xr[mt][i] = *reinterpret_cast<const u4 *>(xp[mt] + at);
    }
    asm volatile("" ::: "memory");   // (the loads stay a batch: none is sunk to its use)
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < kRlBatch; ++i) {
      if constexpr (HALF) {
        if (s + i >= s0 + per) break;   // wave-uniform (s - s0 is)
        if (s + i >= s1) {
          xr[0][i] = u4{0, 0, 0, 0};
#pragma unroll
          for (int nt = 0; nt < NT; ++nt) wr[nt][i] = u4{0, 0, 0, 0};
        }
      } else {
        if (s + i >= s1) break;   // wave-uniform
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
  static_assert(NT * MT <= NW, "a wavefront sums one tile");
  if (wave >= NT * MT) return;
  f4 sum = s_part[0][wave][lane];   // outputs 16 tile + 4 g + i of row 16 mt + ln
#pragma unroll
  for (int p = 1; p < NW; ++p) sum += s_part[p][wave][lane];
  const int row = 16 * (wave % MT) + ln;
  const int64_t tile = static_cast<int64_t>(blockIdx.x) * NT + wave / MT;
  if (tile >= a.tiles) return;
  if constexpr (HALF) {
    // outputs 8 tile + (4 g + i) % 8: lanes ln < 8, g < 2 hold the sums over the
    // first parts of k, lanes ln + 8, g + 2 the same outputs' over the second
#pragma unroll
    for (int i = 0; i < 4; ++i) sum[i] += lane_xor32(dpp_rotate<0x128>(sum[i]));
    if (g < 2 && row < a.rows)
      *reinterpret_cast<u2 *>(a.y + row * a.y_stride + 8 * tile + 4 * g) =
          u2{pack_bf16x2(sum[0], sum[1]), pack_bf16x2(sum[2], sum[3])};
  } else if constexpr (GLU) {
    // rows 4 g + i of the tile: g < 2 gate columns, g + 2 their up columns
    f4 up;
#pragma unroll
    for (int i = 0; i < 4; ++i) up[i] = lane_xor32(sum[i]);
#pragma unroll
    for (int i = 0; i < 4; ++i) sum[i] = situ_value<CAP4>(sum[i], up[i], a.rcg, a.rcu, a.scale);
    if (g < 2 && row < a.rows)
      *reinterpret_cast<u2 *>(a.y + row * a.y_stride + 8 * tile + 4 * g) =
          u2{pack_bf16x2(sum[0], sum[1]), pack_bf16x2(sum[2], sum[3])};
  } else if (row < a.rows) {
    *reinterpret_cast<u2 *>(a.y + row * a.y_stride + 16 * tile + 4 * g) =
        u2{pack_bf16x2(sum[0], sum[1]), pack_bf16x2(sum[2], sum[3])};
  }
}

template <int NW, int NT, int MT, bool GLU, bool CAP4, bool HALF = false>
int launch(const RowLinearArgs &a, hipStream_t st) {
  hipLaunchKernelGGL((row_linear_kernel<NW, NT, MT, GLU, CAP4, HALF>), dim3(static_cast<unsigned>((a.tiles + NT - 1) / NT)),
                     dim3(NW * 64), 0, st, a);
  return check_launch(GLU ? "row_linear_situ_glu" : "row_linear");
}

// One tile of outputs per work-group while that leaves no CU a second one, else
// two, which share their loads of x (7,936 outputs, k = 1,536, 16 rows: 11.0 us
// with one tile, 9.7 with two, four on 124 CUs 13.8).
template <int NW, int MT, bool GLU, bool CAP4>
int dispatch_tiles(const RowLinearArgs &a, hipStream_t st) {
  if (a.tiles > 256) return launch<NW, 2, MT, GLU, CAP4>(a, st);
  return launch<NW, 1, MT, GLU, CAP4>(a, st);
}

// Wavefronts so that one batch holds a wavefront's share of k: 4 up to k =
// 1,024, 8 up to 2,048, 16 beyond.
template <bool GLU, bool CAP4>
int dispatch(const RowLinearArgs &a, hipStream_t st) {
  const int need = (a.ksteps + kRlBatch - 1) / kRlBatch;
  // Half tiles while they are at most one per CU; past that whole tiles fill
  // the chip.  k over 8 parts up to 2,048, over 16 beyond.
  if constexpr (!GLU) {
    if (a.rows <= 8 && a.tiles <= 128) {
      RowLinearArgs half = a;
      half.tiles = 2 * a.tiles;
      if (need <= 8) return launch<4, 1, 1, false, false, true>(half, st);
      return launch<8, 1, 1, false, false, true>(half, st);
    }
  }
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
// transposing copies around it (4.6 us each).
struct HeadLinearArgs {
  const uint16_t *x;
  int64_t x_row, x_head;
  const uint16_t *w;
  uint16_t *y;
  int64_t y_row, y_head;
  int rows, n, ksteps;
};

constexpr int kHlWaves = 8;

__global__ __launch_bounds__(kHlWaves * 64) void head_linear_kernel(HeadLinearArgs a) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ln = lane & 15, g = lane >> 4;
  const int h = blockIdx.y, n0 = 16 * (blockIdx.z * kHlWaves + wave);
  if (n0 >= a.n) return;   // wave-uniform; no barrier below
  const int row = blockIdx.x * 16 + ln;
  const int64_t k = 32 * static_cast<int64_t>(a.ksteps);
  const uint16_t *wp = a.w + (static_cast<int64_t>(h) * a.n + n0 + ln) * k + 8 * g;
  const uint16_t *xp = a.x + min(row, a.rows - 1) * a.x_row + h * a.x_head + 8 * g;
  f4 acc = f4{0.f, 0.f, 0.f, 0.f};
  for (int s = 0; s < a.ksteps; s += kRlBatch) {
    u4 wr[kRlBatch], xr[kRlBatch];
#pragma unroll
    for (int i = 0; i < kRlBatch; ++i) {
      const int at = 32 * min(s + i, a.ksteps - 1);
      wr[i] = *reinterpret_cast<const u4 *>(wp + at);
      xr[i] = *reinterpret_cast<const u4 *>(xp + at);
    }
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < kRlBatch; ++i) {
      if (s + i >= a.ksteps) break;
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf8(wr[i]), as_bf8(xr[i]), acc, 0, 0, 0);
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

extern "C" int sophia_head_linear(const void *x, int64_t x_row_stride, int64_t x_head_stride, const void *w, void *y,
                                  int64_t y_row_stride, int64_t y_head_stride, int64_t rows, int heads, int n, int k,
                                  void *stream) {
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
  if (rows == 0) return SOPHIA_OK;
  const HeadLinearArgs a{static_cast<const uint16_t *>(x), x_row_stride, x_head_stride, static_cast<const uint16_t *>(w),
                         static_cast<uint16_t *>(y), y_row_stride, y_head_stride, static_cast<int>(rows), n, k / 32};
  const dim3 grid(static_cast<unsigned>((rows + 15) / 16), static_cast<unsigned>(heads),
                  static_cast<unsigned>((n + 127) / 128));
  hipLaunchKernelGGL(head_linear_kernel, grid, dim3(kHlWaves * 64), 0, static_cast<hipStream_t>(stream), a);
  return check_launch("head_linear");
}
