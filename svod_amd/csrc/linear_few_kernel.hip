// linear of few rows for gfx950: y = x . w^T (+ bias, + the rope) where all of the output makes few tiles: a decoder
// step's tokens, a query by itself.  The results are linear_kernel's (the epilogue of tk/src/kernels/gemm.rs:604-645,
// 666-716), the sums over k in eight shares.
//
// Such a product is the way of w's and x's bytes into the compute units: one takes in some 80 bytes a nanosecond,
// whatever the rest of the part does, so what counts is how many of them share the bytes, and the latencies in front.
// linear_kernel's 128 x 128 tiles make N / 128 workgroups, each taking in (128 + 128) k elements in stages that meet at
// a barrier: 32 compute units at work at [45, 1024] x [4096, 1024], 10.4 us.  Here a tile is as small as still leaves no
// more workgroups than compute units, and a workgroup's eight waves share k out among themselves: every wave fills
// its own stretch of LDS with its 64 k-columns of the tile's w and x rows (whole 128-byte lines: fragments loaded
// straight into registers take half a line a row, and took 6.2 us there), reads its fragments back, multiplies on
// v_mfma_f32_16x16x32, and the eight partial tiles meet once.  4.0 us; 16 rows 3.6 (10.3 before), 128 rows 4.8 (10.6),
// 256 rows 7.1 (10.9).
//
// A tile's columns are two runs, with the rope half a head apart, so that it holds both halves of every pair it turns.
#include <hip/hip_runtime.h>

#include <atomic>

#include "kernels.h"
#include "launch.h"
#include "matrix.h"

namespace svodk {
namespace {

constexpr int kWaves = 8;
constexpr int kBk = 64;              // k-columns a wave takes at a time: a row of them is one 128-byte line
constexpr int kRowBytes = kBk * 2;

// A workgroup's tile: 16 RB rows x 16 CB columns.
template <int RB_, int CB_>
struct Tile {
  static constexpr int RB = RB_, CB = CB_;
  static constexpr int kBm = 16 * RB, kBn = 16 * CB;
  static constexpr int kChunkBytes = (kBm + kBn) * kRowBytes;  // a wave's stretch of LDS: the w rows, then the x rows
  static constexpr int kPitch = kBn + 4;                       // floats from a row of a partial tile to the next in LDS
  static constexpr int kPartBytes = kBm * kPitch * 4;
  static constexpr int kWaveBytes = kChunkBytes > kPartBytes ? kChunkBytes : kPartBytes;
  static constexpr int kLds = kWaves * kWaveBytes;
};

struct FewCall {
  const uint16_t *x, *w, *bias, *cos, *sin;
  uint16_t *y;
  int64_t y_ld;
  int32_t rows, n, k, seq, heads;
  uint32_t tiles_m;
};

// HD: the head size a turning kernel is built for (64 or 128), 0: no turn.
template <bool F16, int HD, typename T>
__global__ __launch_bounds__(kWaves * 64) void linear_few_kernel(const FewCall call) {
#if defined(__HIP_DEVICE_COMPILE__)
  const auto [x, w, bias, cos_t, sin_t, y, y_ld, rows, n, k, seq, heads, tiles_m] = call;
  constexpr int RB = T::RB, CB = T::CB, kBm = T::kBm, kBn = T::kBn, kRun = kBn / 2, kPitch = T::kPitch;
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int tid = (int)__builtin_amdgcn_workitem_id_x(), lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ln = lane & 15, g = lane >> 4;

  // The workgroup's rows and its columns: col0 .. col0 + kRun - 1 and col1 .. col1 + kRun - 1.
  constexpr int kHead = HD > 0 ? HD : 64, kHalf = kHead / 2;
  const uint32_t wg = __builtin_amdgcn_workgroup_id_x();
  const int tn = (int)(wg / tiles_m), row0 = (int)(wg - (uint32_t)tn * tiles_m) * kBm;
  const bool turned = HD > 0 && tn * kBn < heads * HD;
  const int in_head = tn % (kHead / kBn) * kRun;  // of a turned workgroup's first run
  const int col0 = turned ? tn / (kHead / kBn) * kHead + in_head : tn * kBn;
  const int col1 = turned ? col0 + kHalf : col0 + kRun;

  // ---- a wave's fill: 64 k-columns of the tile's w rows and x rows, 8 rows x 128 bytes an instruction, the 16-byte
  // chunks of a row xor-ed with (row / 2) % 8 through the lanes' source addresses, so that a fragment's 16 rows at
  // one logical chunk touch every bank once.  Rows past the operands' ends land zeros.
  const int64_t row_bytes = (int64_t)k * 2;
  const int frow = lane >> 3, place = lane & 7;
  uint8_t *mine = smem + wave * T::kWaveBytes;
  const int lds0 = (int)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)(smem) + wave * T::kWaveBytes;
  constexpr int kInstrs = T::kChunkBytes / 1024;
  auto fill = [&](int c) {
    const int64_t at = (int64_t)c * kRowBytes;
    const i32x4 rx = make_rsrc((const uint8_t *)x + row0 * row_bytes + at, (int64_t)(rows - row0) * row_bytes - at);
    const i32x4 r0 = make_rsrc((const uint8_t *)w + col0 * row_bytes + at, (int64_t)(n - col0) * row_bytes - at);
    const i32x4 r1 = make_rsrc((const uint8_t *)w + col1 * row_bytes + at, (int64_t)(n - col1) * row_bytes - at);
    const bool half = c * kBk + 32 >= k;  // a last chunk of one k-step: its second half lands zeros
#pragma unroll
    for (int j = 0; j < kInstrs; j++) {
      const bool is_x = j >= kBn / 8;
      const int first = is_x ? 8 * j - kBn : (8 * j < kRun ? 8 * j : 8 * j - kRun);  // from the descriptor's first row
      if (is_x && row0 + first >= rows) continue;  // the rest of an x tile that is not there: never stored
      const int chunk = place ^ ((4 * (j & 1) + (frow >> 1)) & 7);
      const int voff = half && chunk >= 4 ? (int)kPastBound : (int)((first + frow) * row_bytes) + chunk * 16;
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                   :
                   : "s"(__builtin_amdgcn_readfirstlane(lds0 + j * 1024)), "v"(voff), "s"(is_x ? rx : (8 * j < kRun ? r0 : r1))
                   : "memory");
    }
  };

  // ---- the wave's share of k.  Fragments: A = w, lane row ln (an output column), chunk 4 ks + g of a row; B = x.
  // The wave's stretch is its own: no barrier until the partial tiles meet.  Its fragments are in registers before
  // the next fill is issued.
  f32x4 acc[RB][CB];
#pragma unroll
  for (int rb = 0; rb < RB; rb++)
#pragma unroll
    for (int cb = 0; cb < CB; cb++) acc[rb][cb] = f32x4{0, 0, 0, 0};
  const int chunks = (k + kBk - 1) / kBk;
  int c = (int)((int64_t)chunks * wave / kWaves);
  const int end = (int)((int64_t)chunks * (wave + 1) / kWaves);
  if (c < end) fill(c);
  const int swz = (ln >> 1) & 7;
  for (; c < end; c++) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    u32x4 wf[2][CB], xf[2][RB];
#pragma unroll
    for (int ks = 0; ks < 2; ks++) {
      const uint8_t *at = mine + ln * kRowBytes + (((4 * ks + g) ^ swz) << 4);
#pragma unroll
      for (int cb = 0; cb < CB; cb++) wf[ks][cb] = *reinterpret_cast<const u32x4 *>(at + cb * 16 * kRowBytes);
#pragma unroll
      for (int rb = 0; rb < RB; rb++) xf[ks][rb] = *reinterpret_cast<const u32x4 *>(at + (kBn + rb * 16) * kRowBytes);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (c + 1 < end) fill(c + 1);
#pragma unroll
    for (int ks = 0; ks < 2; ks++)
#pragma unroll
      for (int cb = 0; cb < CB; cb++)
#pragma unroll
        for (int rb = 0; rb < RB; rb++) acc[rb][cb] = mma<F16>(wf[ks][cb], xf[ks][rb], acc[rb][cb]);
  }

  // ---- the partial tiles meet in LDS, each wave's where its chunks lay.  Accumulator (rb, cb) element e: row
  // 16 rb + ln, the tile's column 16 cb + 4 g + e.
  float *part = reinterpret_cast<float *>(mine);
#pragma unroll
  for (int rb = 0; rb < RB; rb++)
#pragma unroll
    for (int cb = 0; cb < CB; cb++)
      *reinterpret_cast<f32x4 *>(part + (16 * rb + ln) * kPitch + 16 * cb + 4 * g) = acc[rb][cb];
  __syncthreads();
  // A thread finishes four columns of a row, or with a turn four and the four they turn with.
  constexpr int kQuads = kBn / 4;
  auto column = [&](int q) { return (q < kQuads / 2 ? col0 : col1 - kRun) + 4 * q; };
  auto sum_of = [&](int r, int q) {
    f32x4 s = *reinterpret_cast<const f32x4 *>(smem + (r * kPitch + 4 * q) * 4);
#pragma unroll
    for (int v = 1; v < kWaves; v++) s += *reinterpret_cast<const f32x4 *>(smem + v * T::kWaveBytes + (r * kPitch + 4 * q) * 4);
    const int col = column(q);
    if (bias != nullptr && col < n) s += load4<F16>(bias + col);
    return s;
  };
  auto store = [&](int r, int q, const f32x4 &s) {
    const int col = column(q);
    if (col < n)
      *reinterpret_cast<u32x2 *>(y + (int64_t)(row0 + r) * y_ld + col) = u32x2{narrow<F16>(s[0], s[1]), narrow<F16>(s[2], s[3])};
  };
  const int live = min(kBm, rows - row0);
  if (HD > 0 && turned) {
    for (int i = tid; i < live * (kQuads / 2); i += kWaves * 64) {
      const int r = i / (kQuads / 2), q = i % (kQuads / 2);
      const f32x4 a = sum_of(r, q), b = sum_of(r, q + kQuads / 2);
      const int64_t at = (int64_t)((row0 + r) % seq) * kHalf + in_head + 4 * q;  // gemm.rs:685: the token's position
      const f32x4 cs = load4<F16>(cos_t + at), sn = load4<F16>(sin_t + at);
      f32x4 ra, rb;
#pragma unroll
      for (int e = 0; e < 4; e++) {
        // gemm.rs:702-705: x cos, then the partner's product joined by one fused multiply-add.
        const float ac = a[e] * cs[e], bc = b[e] * cs[e];
        ra[e] = __builtin_fmaf(b[e], -sn[e], ac);
        rb[e] = __builtin_fmaf(a[e], sn[e], bc);
      }
      store(r, q, ra);
      store(r, q + kQuads / 2, rb);
    }
  } else {
    for (int i = tid; i < live * kQuads; i += kWaves * 64) store(i / kQuads, i % kQuads, sum_of(i / kQuads, i % kQuads));
  }
#endif
}

template <bool F16, int HD, typename T>
hipError_t launch(const LinearArgs &a, hipStream_t stream) {
  const int64_t tiles_m = (a.rows + T::kBm - 1) / T::kBm, tiles = tiles_m * ((a.n + T::kBn - 1) / T::kBn);
  if (tiles > 0x7fffffffLL) return hipErrorInvalidConfiguration;
  return Launch<linear_few_kernel<F16, HD, T>>::run(
      tiles, kWaves * 64, T::kLds, T::kLds, stream,
      FewCall{(const uint16_t *)a.x, (const uint16_t *)a.w, (const uint16_t *)a.bias, (const uint16_t *)a.cos,
              (const uint16_t *)a.sin, (uint16_t *)a.y, a.y_ld > 0 ? a.y_ld : (int64_t)a.n, (int32_t)a.rows, a.n, a.k, a.seq,
              a.heads, (uint32_t)tiles_m});
}

template <typename T>
hipError_t launch_tile(const LinearArgs &a, hipStream_t stream) {
  const int hd = a.cos != nullptr ? a.head_dim : 0;
  if (a.f16) return hd == 0 ? launch<true, 0, T>(a, stream) : hd == 64 ? launch<true, 64, T>(a, stream) : launch<true, 128, T>(a, stream);
  return hd == 0 ? launch<false, 0, T>(a, stream) : hd == 64 ? launch<false, 64, T>(a, stream) : launch<false, 128, T>(a, stream);
}

}  // namespace

hipError_t launch_linear_few(const LinearArgs &a, hipStream_t stream) {
  if (a.rows < 1 || a.rows > 0x7fffffff || a.k > kLinearFewMaxK) return hipErrorInvalidValue;
  switch (a.tile) {
    case kFew16x16: return launch_tile<Tile<1, 1>>(a, stream);
    case kFew32x16: return launch_tile<Tile<2, 1>>(a, stream);
    case kFew32x32: return launch_tile<Tile<2, 2>>(a, stream);
    case kFew64x32: return launch_tile<Tile<4, 2>>(a, stream);
    case kFew64x64: return launch_tile<Tile<4, 4>>(a, stream);
  }
  return hipErrorInvalidValue;
}

}  // namespace svodk
