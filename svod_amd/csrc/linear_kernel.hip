// linear with the rope epilogue for gfx950 (MI355X): y = x . w^T + bias over x [rows, K] and w [N, K]
// (both K-contiguous), the first `heads` heads of `head_dim` output columns turned by the rotary tables'
// row of the token's position before the one rounding at the store.  The algorithm is the reference GEMM
// kernel's epilogue (tk/src/kernels/gemm.rs:604-645 `finish`, :666-716 `turn`): f32 accumulators, the bias
// added in f32, then per turned column  y = fma(partner, +-sin, x * cos)  with the partner half a head
// along and sin negated over a head's first half, then the cast.  A fused projection's queries and keys
// come out rotated and its values plain, so a model without QK norms needs no prologue pass at all
// (tk/src/ops/linear.rs:47-58).
//
// The mapping onto CDNA4 is this file's own.  A workgroup of 4 x WN waves owns a tile of the output, at its largest
// 256 x 256 by 8 waves of 64 rows x 128 columns.  The product runs transposed, C^T = W . X^T, on
// v_mfma_f32_16x16x32: a lane owns one output ROW of a 16 x 16 block and four CONSECUTIVE columns of it, and the
// rotation's partner column (32 or 64 columns along) is the same lane's register of another block.  The 16 x 16 atom
// and not the 32 x 32 x 16 one because the part holds a higher clock under it: 2.12 PFLOP/s against 1.90 for nothing
// but matrix instructions on live data (it moves half the accumulator registers a flop).
// X and W tiles of 64 k-columns stream through an LDS ring, filled global -> LDS by buffer_load_dwordx4 ... lds.
// What bounds this kernel is the way from L2 into LDS beside the matrix pipe: a compute unit takes in some 80 bytes a
// nanosecond when every fill takes whole 128-byte lines (half lines: two thirds of that), so a 256 x 256 x 64 stage's
// 64 KiB are 0.8 us beside 0.85 us of matrix instructions.  Hence rows of 128 bytes, a whole line each, tiles as large
// as LDS holds where there are enough of them, and fills one at a time between the products: issued together behind
// the barrier they fill the address path's queue and the waves stand there instead of issuing products (130 -> 124 us
// at [16384, 1024] x [4096, 1024]).  A row's eight 16-byte chunks are XOR-swizzled by (row / 2) % 8 through the lanes'
// source addresses so that a ds_read_b128 of 16 rows at one logical chunk touches every bank once.  Rows past the
// operands' ends read as zeros through the buffer descriptors' bounds.  One barrier a stage.
#include <hip/hip_runtime.h>

#include <atomic>

#include "kernels.h"
#include "launch.h"
#include "matrix.h"

namespace svodk {
namespace {

#if !defined(__HIP_DEVICE_COMPILE__)
#pragma clang diagnostic ignored "-Wunused-function"
#pragma clang diagnostic ignored "-Wunused-const-variable"
#endif

constexpr int kXcds = 8;
constexpr int kBk = 64;                 // k-columns a stage: a row of a tile is one 128-byte line
constexpr int kGroup = 8;               // column tiles an XCD's resident workgroups spread over
constexpr int kRowBytes = kBk * 2;      // a tile row in LDS
constexpr int kAhead = 4;               // column blocks between a W fragment's request and its products

// The workgroup's output tile: 4 waves along the rows, 16 RB rows each, x WN waves along the columns, 16 CB columns
// each.  The W tiles of SW stages and the X tiles of SX stages lie in LDS.
template <int RB_, int CB_, int WN_, int SW_, int SX_>
struct Tile {
  static constexpr int RB = RB_, CB = CB_, WN = WN_, SW = SW_, SX = SX_;
  static constexpr int kWaves = 4 * WN;
  static constexpr int kBm = 64 * RB, kBn = 16 * CB * WN;
  static constexpr int kWBytes = kBn * kRowBytes, kXBytes = kBm * kRowBytes;
  static constexpr int kLds = SW * kWBytes + SX * kXBytes;     // the W ring, then the X ring
  static constexpr int kWFills = kWBytes / 1024 / kWaves;      // wave instructions of 1 KiB per wave and stage
  static constexpr int kXFills = kXBytes / 1024 / kWaves;
  static constexpr int kOutPitch = CB * 32 + 16;               // a wave's row of the finished tile in LDS
  static_assert(kWBytes % (1024 * kWaves) == 0 && kXBytes % (1024 * kWaves) == 0, "a tile fills in whole instructions a wave");
  static_assert(kWaves * 32 * kOutPitch <= kLds, "32 rows a wave of the finished tile fit where the ring was");
  static_assert(CB >= kAhead && (2 * CB) % kAhead == 0 && RB % 2 == 0 && RB <= 2 * (kAhead - 1), "the k loop's schedule");
  static_assert(SX >= 2 && (SW == SX || SW == SX + 1), "the k loop's waits");
};
// 256 x 256 by 8 waves (64 rows x 128 columns each), 128 KiB: the tile for a product with tiles enough to fill the part.
// (A third W tile in the ring gives 1 % at k = 4096 and nothing at 1024.)
typedef Tile<4, 8, 2, 2, 2> Large;
// 256 x 192 by 8 waves (64 x 96 each), 136 KiB: where it leaves fewer compute units idle in the last round.
typedef Tile<4, 6, 2, 3, 2> Wide;
// 128 x 128 by 8 waves (32 x 64 each), 80 KiB, two workgroups a compute unit: four times the workgroups, at twice the
// fills a flop.  Its products leave a fill less time to arrive, so the third W tile pays: 139 -> 132 us at [16384, 1024]
// x [4096, 1024].
typedef Tile<2, 4, 2, 3, 2> Mid;
// 128 x 64 by 4 waves (32 x 64 each), 72 KiB: where Mid would leave compute units without any tile.
typedef Tile<2, 4, 1, 3, 3> Narrow;

// Where a wave's column blocks lie in the tile.  A turned head's halves have to meet in one wave: two waves of 64
// columns take 32 columns of each half of a head of 128 instead of a half each.
template <int HD, typename T>
struct Columns {
  static constexpr bool kSplit = HD == 128 && T::CB == 4 && T::WN == 2;
  static_assert(HD == 0 || kSplit || (T::CB * 16) % (HD > 0 ? HD : 1) == 0, "a wave holds whole turned heads");
  static constexpr int kWaveStep = kSplit ? 32 : 16 * T::CB;  // from a wave's columns to the next's
  // Block cb's first column in a wave whose columns start at 0.
  __host__ __device__ static constexpr int at(int cb) { return kSplit ? 64 * (cb >> 1) + 16 * (cb & 1) : 16 * cb; }
  static constexpr int kHalfBlocks = kSplit ? 2 : HD / 32;  // from a block to its partner
  __host__ __device__ static constexpr bool first_half(int cb) { return HD > 0 && at(cb) % (HD > 0 ? HD : 1) < HD / 2; }
};

#if defined(__HIP_DEVICE_COMPILE__)
// HD: the head size a turning kernel is built for (64 or 128), 0: no turn.
template <bool F16, int HD, typename T>
__device__ __forceinline__ void linear_body(uint8_t *smem, const uint16_t *__restrict__ x, const uint16_t *__restrict__ w,
                                            const uint16_t *__restrict__ bias, const uint16_t *__restrict__ cos_t,
                                            const uint16_t *__restrict__ sin_t, uint16_t *__restrict__ y, int64_t y_ld,
                                            int64_t rows, int32_t n, int32_t k, int32_t seq, int32_t heads,
                                            uint32_t tiles_n, uint32_t tiles, uint32_t per_xcd) {
  constexpr int kWaves = T::kWaves, kBm = T::kBm, kBn = T::kBn, kWBytes = T::kWBytes, kXBytes = T::kXBytes;
  constexpr int kLds = T::kLds, kWFills = T::kWFills, kXFills = T::kXFills, kFills = kWFills + kXFills;
  constexpr int SW = T::SW, SX = T::SX, RB = T::RB, CB = T::CB, kXRing = SW * kWBytes;
  typedef Columns<HD, T> Cols;
  const int tid = __builtin_amdgcn_workitem_id_x();
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, ln = lane & 15;
  // Workgroups are dealt to the 8 XCDs in turn, each XCD with an L2 of its own.  The tiles stand in one row: groups
  // of up to kGroup column tiles, row tile after row tile within a group; XCD x takes the x-th eighth of that row.
  // The workgroups resident together on an XCD then share few w tiles and few x tiles, and no XCD has more than one
  // tile more than another: whole bands of row tiles an XCD, the order before, gave XCDs 0..5 36 tiles for their 32
  // compute units and XCD 7 none at [6216, 768] x [2304, 768] (225 tiles: 46 us, two rounds; 26 us in one).
  const uint32_t wg = __builtin_amdgcn_workgroup_id_x();
  const uint32_t turn = wg % kXcds * per_xcd + wg / kXcds;
  if (turn >= tiles) return;
  const uint32_t tiles_m = tiles / tiles_n, full = tiles_m * kGroup;  // workgroups of a full-width group
  const uint32_t ng = turn / full;
  const uint32_t first_tn = ng * kGroup;  // the group's first column tile
  const uint32_t width = min((uint32_t)kGroup, tiles_n - first_tn);
  const uint32_t in_group = turn - ng * full;
  const uint32_t tm = in_group / width, tn = first_tn + (in_group - tm * width);
  const int64_t m0 = (int64_t)tm * kBm;
  const int32_t n0 = (int32_t)tn * kBn;
  const int64_t row_bytes = (int64_t)k * 2;

  // ---- this wave's fills of a stage: 8 rows x 8 chunk places an instruction; a stage is the W tile's and then
  // the X tile's, and wave v takes instructions v, v + waves, ...  Those are a multiple of 32 rows apart and the
  // swizzle's period is 16, so one lane offset serves them all; the descriptors' bases differ.
  const int frow = lane >> 3, place = lane & 7;
  const int src = frow * (int)row_bytes + ((place ^ ((4 * (wave & 1) + (frow >> 1)) & 7)) << 4);
  const int lds0 = (int)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)(smem) + wave * 1024;
  i32x4 rsrc[kFills];  // the W tile's instructions, then the X tile's
#pragma unroll
  for (int f = 0; f < kFills; f++) {
    const bool is_x = f >= kWFills;
    const int64_t first = (is_x ? m0 : (int64_t)n0) + 8 * (wave + kWaves * (is_x ? f - kWFills : f));
    const int64_t limit = is_x ? rows : (int64_t)n;
    rsrc[f] = make_rsrc((const uint8_t *)(is_x ? x : w) + first * row_bytes, (limit - first) * row_bytes);
  }
  // k is a multiple of 32: a last stage may hold one k-step only.  The lanes that would fetch the second
  // half of its rows (the next rows' data) then address past every descriptor's bound and land zeros.
  const int nk = (k + kBk - 1) / kBk;
  const bool short_tail = (k % kBk) != 0;
  const bool second_half = ((place ^ ((4 * (wave & 1) + (frow >> 1)) & 7)) & 4) != 0;
  // Fill `f` of stage `s` of the k loop into slot `slot` of its ring; past the last stage an empty descriptor (zeros
  // land in a slot nothing reads any more) keeps the count of fills in flight the same in every iteration.
  auto fill = [&](int s, int slot, int f) {
    const int voff = (short_tail && s == nk - 1 && second_half) ? (int)kPastBound : src + s * kRowBytes;
    const int at = f < kWFills ? slot * kWBytes + f * kWaves * 1024 : kXRing + slot * kXBytes + (f - kWFills) * kWaves * 1024;
    i32x4 r = rsrc[f];
    if (s >= nk) r[2] = 0;
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                 :
                 : "s"(lds0 + at), "v"(voff), "s"(r)
                 : "memory");
  };

  // ---- the schedule of a stage: two k-steps of 32, each CB column blocks of RB products (W fragment cb against the
  // RB fragments of X).  A W fragment is asked for kAhead blocks before its products, a k-step's X fragments in the
  // last blocks of the k-step before.  Ahead of the last kAhead - 1 blocks of a stage therefore stands its barrier:
  // every wave's fills of the next stage have landed and its reads of this one are back (the last of them asked for
  // two blocks earlier), so the next stage is whole and this stage's slots are free.  The fills follow one by one: X of
  // the stage SX further on beside those last blocks, W of the stage SX + 1 further on (with SW = SX + 1; else SX)
  // beside the next stage's first blocks, from where it has more than a stage to arrive.
  constexpr int kBlocks = 2 * CB, kBarrier = kBlocks - kAhead + 1;
  constexpr int kXPer = (kXFills + kAhead - 2) / (kAhead - 1), kWPer = (kWFills + 3) / 4;  // fills a block
  static_assert((kWFills + kWPer - 1) / kWPer <= kBarrier, "a stage's fills are out before its barrier");
  constexpr int kWLead = SW - 1;  // a stage's first blocks ask for W of the stage this much further on
#pragma unroll
  for (int s = 0; s < SX; s++)
#pragma unroll
    for (int f = s < kWLead ? 0 : kWFills; f < kFills; f++) fill(s, s, f);

  // ---- operand reads: A = W rows (the output's columns), B = X rows (the output's rows); a fragment is 16 rows, its
  // lane (ln, g) reads logical chunk 4 ks + g of row ln.
  const int wave_m = wave & 3, wave_n = wave >> 2;
  const int swz = (ln >> 1) & 7;  // every block starts on a multiple of 16 rows
  int w_read[2], x_read[2];
#pragma unroll
  for (int ks = 0; ks < 2; ks++) {
    const int chunk = ((4 * ks + g) ^ swz) << 4;
    w_read[ks] = (wave_n * Cols::kWaveStep + ln) * kRowBytes + chunk;
    x_read[ks] = kXRing + (wave_m * 16 * RB + ln) * kRowBytes + chunk;
  }
  f32x4 acc[RB][CB];
#pragma unroll
  for (int rb = 0; rb < RB; rb++)
#pragma unroll
    for (int cb = 0; cb < CB; cb++) acc[rb][cb] = f32x4{0, 0, 0, 0};
  u32x4 wf[kAhead], xf[2][RB];
  auto read_w = [&](int slot, int block) {  // block 0 .. kBlocks - 1 of a stage
    wf[block % kAhead] = *reinterpret_cast<const u32x4 *>(smem + slot * kWBytes + w_read[block / CB] + Cols::at(block % CB) * kRowBytes);
  };
  auto read_x = [&](int slot, int ks, int rb) {
    xf[ks][rb] = *reinterpret_cast<const u32x4 *>(smem + slot * kXBytes + x_read[ks] + rb * 16 * kRowBytes);
  };
  // The rotary tables' rows of this tile (16 bytes a lane along the rows, kTables loads a table and lane)
  // are asked for behind the barrier of the last stage but one: they arrive under the last stage's products
  // and are in registers when the epilogue wants them in LDS.
  constexpr int kHalf = (HD > 0 ? HD : 64) / 2, kTChunks = kHalf * 2 / 16, kTables = kBm * kTChunks / (kWaves * 64);
  const bool turning = HD > 0 && n0 < heads * HD;  // the same for the whole workgroup
  u32x4 tc[kTables], ts[kTables];
  const int tables_at = nk > 1 ? nk - 2 : 0;
  auto load_tables = [&]() {
    // gemm.rs:685: the table row of the token's position.  A lane's rows are kWaves * 64 / kTChunks apart.
    const uint32_t useq = (uint32_t)seq, step = (uint32_t)(kWaves * 64 / kTChunks) % useq;
    uint32_t pos = ((uint32_t)(m0 % seq) + (uint32_t)(tid / kTChunks)) % useq;
#pragma unroll
    for (int i = 0; i < kTables; i++) {
      const int64_t at = (int64_t)pos * (kHalf * 2) + tid % kTChunks * 16;
      tc[i] = *reinterpret_cast<const u32x4 *>(reinterpret_cast<const uint8_t *>(cos_t) + at);
      ts[i] = *reinterpret_cast<const u32x4 *>(reinterpret_cast<const uint8_t *>(sin_t) + at);
      pos += step;
      pos = pos >= useq ? pos - useq : pos;
    }
  };

  // In flight behind stage 0 there: X of stages 1 .. SX - 1 and W of stages 1 .. min(SX, kWLead) - 1.
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"((SX - 1) * kXFills + ((SX < kWLead ? SX : kWLead) - 1) * kWFills) : "memory");
  __syncthreads();
#pragma unroll
  for (int rb = 0; rb < RB; rb++) read_x(0, 0, rb);
#pragma unroll
  for (int b = 0; b < kAhead; b++) read_w(0, b);
  int ws = 0, xs = 0, wfill = kWLead;  // the slots of this stage, and of the W tile that its first blocks ask for
  for (int s = 0; s < nk; s++) {
    const int ws_next = ws + 1 == SW ? 0 : ws + 1, xs_next = xs + 1 == SX ? 0 : xs + 1;
#pragma unroll
    for (int b = 0; b < kBlocks; b++) {
      const int ks = b / CB, cb = b % CB;
      if (b == kBarrier) {
        // Stage s + 1 is in: behind it in flight are X of the SX - 2 and W of the kWLead - 1 stages after it.
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((SX - 2) * kXFills + (kWLead - 1) * kWFills) : "memory");
        __syncthreads();
        if (HD > 0 && turning && s == tables_at) load_tables();
      }
#pragma unroll
      for (int rb = 0; rb < RB; rb++) acc[rb][cb] = mma<F16>(wf[b % kAhead], xf[ks][rb], acc[rb][cb]);
      if (b == kBarrier) read_w(ws_next, 0);
      if (b < kBlocks - kAhead)
        read_w(ws, b + kAhead);
      else if (b >= kBarrier)
        read_w(ws_next, b + kAhead - kBlocks);
#pragma unroll
      for (int i = 0; i < 2; i++) {  // two fragments of the next k-step's X a block
        const int xr = 2 * (cb - (CB - kAhead + 1)) + i;
        if (xr >= 0 && xr < RB) read_x(ks == 0 ? xs : xs_next, ks ^ 1, xr);
      }
#pragma unroll
      for (int i = 0; i < kXPer; i++)
        if (b >= kBarrier && (b - kBarrier) * kXPer + i < kXFills) fill(s + SX, xs, kWFills + (b - kBarrier) * kXPer + i);
#pragma unroll
      for (int i = 0; i < kWPer; i++)
        if (b * kWPer + i < kWFills) fill(s + kWLead, wfill, b * kWPer + i);
      __builtin_amdgcn_sched_barrier(0);
    }
    wfill = ws;
    ws = ws_next;
    xs = xs_next;
  }
  // The empty fills still in flight write LDS: they land before the workgroup's LDS is given away.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  // ---- epilogue.  Accumulator (rb, cb) element e: row m0 + 16 RB wave_m + 16 rb + ln, column
  // wave_n0 + Cols::at(cb) + 4 g + e.
  const int wave_n0 = n0 + wave_n * Cols::kWaveStep;
  // The bias, or -0 without one (x + -0 is x): a branch around the whole addition would have the compiler keep a second
  // set of accumulators for where its two ways meet.
#pragma unroll
  for (int cb = 0; cb < CB; cb++) {
    f32x4 b4 = {-0.0f, -0.0f, -0.0f, -0.0f};
    if (bias != nullptr) b4 = load4<F16>(bias + min(wave_n0 + Cols::at(cb) + 4 * g, n - 4));  // columns past the end are not stored
#pragma unroll
    for (int rb = 0; rb < RB; rb++)
#pragma unroll
      for (int e = 0; e < 4; e++) acc[rb][cb][e] += b4[e];
  }
  if (HD > 0 && turning) {
    // The tile's rows of the tables go through LDS (the ring is done with): loaded 16 bytes a lane along the rows,
    // read back 8 bytes a lane down them.  A lane owns a ROW of the output, so reading the tables straight from
    // memory would touch 16 lines an instruction.  Rows of 2 * kHalf + 8 bytes keep the reads off each other's banks.
    constexpr int kPitch = kHalf * 2 + 8;
    uint8_t *cos_lds = smem, *sin_lds = smem + kBm * kPitch;
    __syncthreads();  // every wave's last fragments are read and its last fills have landed
    static_assert(2 * kBm * kPitch <= kLds, "the tables fit where the ring was");
#pragma unroll
    for (int i = 0; i < kTables; i++) {
      const int c = tid + i * kWaves * 64, r = c / kTChunks, ch = c % kTChunks;
      const u32x4 vc = tc[i], vs = ts[i];
      u32x2 *cd = reinterpret_cast<u32x2 *>(cos_lds + r * kPitch + ch * 16);
      u32x2 *sd = reinterpret_cast<u32x2 *>(sin_lds + r * kPitch + ch * 16);
      cd[0] = u32x2{vc[0], vc[1]};
      cd[1] = u32x2{vc[2], vc[3]};
      sd[0] = u32x2{vs[0], vs[1]};
      sd[1] = u32x2{vs[2], vs[3]};
    }
    __syncthreads();
    const int turned = heads * HD;
#pragma unroll
    for (int cb = 0; cb < CB; cb++) {
      if (!Cols::first_half(cb)) continue;  // second halves are turned with their first
      constexpr int hd = HD > 0 ? HD : 64;
      const int pb = cb + Cols::kHalfBlocks < CB ? cb + Cols::kHalfBlocks : cb;  // the partner block (always the first)
      const int col = wave_n0 + Cols::at(cb);
      if (col >= turned) continue;
      const int at = (col & (hd - 1)) + 4 * g;  // index into the table row, < kHalf
#pragma unroll
      for (int rb = 0; rb < RB; rb++) {
        const int r = wave_m * 16 * RB + rb * 16 + ln;
        const f32x4 c4 = load4<F16>(reinterpret_cast<const uint16_t *>(cos_lds + r * kPitch) + at);
        const f32x4 s4 = load4<F16>(reinterpret_cast<const uint16_t *>(sin_lds + r * kPitch) + at);
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const float y1 = acc[rb][cb][e], y2 = acc[rb][pb][e];
          // gemm.rs:702-705: x cos, then the partner's product joined by one fused multiply-add.
          const float y1c = y1 * c4[e], y2c = y2 * c4[e];
          acc[rb][cb][e] = __builtin_fmaf(y2, -s4[e], y1c);
          acc[rb][pb][e] = __builtin_fmaf(y1, s4[e], y2c);
        }
      }
    }
  }
  // ---- the store.  A lane owns rows, not runs of columns: written from the registers an instruction would
  // touch 16 rows with 32 bytes each.  The rounded tile goes through LDS instead (every wave is done with the
  // ring, and with the tables), 32 rows of a wave at a time in a stretch of its own, and leaves as whole row
  // segments, 16 bytes a lane.
  __syncthreads();
  constexpr int kOutPitch = T::kOutPitch, kRowChunks = CB * 2, kRowsPer = 64 / kRowChunks;
  uint8_t *stage = smem + wave * 32 * kOutPitch;
  const int orow = lane / kRowChunks, ochunk = lane % kRowChunks;
  const int col = wave_n0 + Cols::at(ochunk >> 1) + 8 * (ochunk & 1);  // n is a multiple of 8: a run of eight lies inside or outside
#pragma unroll
  for (int half = 0; half < RB / 2; half++) {
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int rb = 2 * half + i;
      uint8_t *srow = stage + (16 * i + ln) * kOutPitch + 8 * g;
#pragma unroll
      for (int cb = 0; cb < CB; cb++) {
        u32x2 out;
        out[0] = narrow<F16>(acc[rb][cb][0], acc[rb][cb][1]);
        out[1] = narrow<F16>(acc[rb][cb][2], acc[rb][cb][3]);
        *reinterpret_cast<u32x2 *>(srow + 32 * cb) = out;
      }
    }
#pragma unroll
    for (int it = 0; it < (32 + kRowsPer - 1) / kRowsPer; it++) {
      const int r = it * kRowsPer + orow;
      const bool mine = (kRowsPer * kRowChunks == 64 && 32 % kRowsPer == 0) || (orow < kRowsPer && r < 32);
      const int64_t row = m0 + wave_m * 16 * RB + half * 32 + r;
      // Streaming stores: the output is not read again here, and left out of L2 it does not push the operands out.
      if (mine && row < rows && col < n)
        __builtin_nontemporal_store(*reinterpret_cast<const u32x4 *>(stage + r * kOutPitch + ochunk * 16),
                                    reinterpret_cast<u32x4 *>(y + row * y_ld + col));
    }
  }
}
#endif  // __HIP_DEVICE_COMPILE__

#if !defined(SVODK_CODE_OBJECT)  // the library's kernel and its launch: not part of a code object build
struct LinearCall {
  const uint16_t *x, *w, *bias, *cos, *sin;
  uint16_t *y;
  int64_t y_ld, rows;
  int32_t n, k, seq, heads;
  uint32_t tiles_n, tiles, per_xcd;
};

template <bool F16, int HD, typename T>
__global__ __launch_bounds__(T::kWaves * 64, T::kLds > 80 * 1024 ? T::kWaves / 4 : T::kWaves / 2) void linear_kernel(
    const LinearCall c) {
#if defined(__HIP_DEVICE_COMPILE__)
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  linear_body<F16, HD, T>(smem, c.x, c.w, c.bias, c.cos, c.sin, c.y, c.y_ld, c.rows, c.n, c.k, c.seq, c.heads, c.tiles_n,
                          c.tiles, c.per_xcd);
#endif
}

template <bool F16, int HD, typename T>
hipError_t launch(const LinearArgs &a, hipStream_t stream) {
  const int64_t tiles_m = (a.rows + T::kBm - 1) / T::kBm, tiles_n = (a.n + T::kBn - 1) / T::kBn;
  const int64_t tiles = tiles_m * tiles_n;
  if (tiles == 0) return hipSuccess;
  const int64_t per_xcd = (tiles + kXcds - 1) / kXcds;
  if (tiles_m * kGroup > 0x7fffffffLL || per_xcd * kXcds > 0x7fffffffLL) return hipErrorInvalidConfiguration;
  return Launch<linear_kernel<F16, HD, T>>::run(
      per_xcd * kXcds, T::kWaves * 64, T::kLds, T::kLds, stream,
      LinearCall{(const uint16_t *)a.x, (const uint16_t *)a.w, (const uint16_t *)a.bias, (const uint16_t *)a.cos,
                 (const uint16_t *)a.sin, (uint16_t *)a.y, a.y_ld > 0 ? a.y_ld : (int64_t)a.n, a.rows, a.n, a.k, a.seq,
                 a.heads, (uint32_t)tiles_n, (uint32_t)tiles, (uint32_t)per_xcd});
}

template <int HD, typename T>
hipError_t launch_hd(const LinearArgs &a, hipStream_t stream) {
  return a.f16 ? launch<true, HD, T>(a, stream) : launch<false, HD, T>(a, stream);
}

}  // namespace
#else  // SVODK_CODE_OBJECT
// The same program as kernels for a loader that takes a code object and a flat argument record
// (device/src/amd/program.rs:403-414, 655-675; device/src/hcq.rs:1262-1285): buffers first, then 4-byte
// scalars, nothing hidden, static LDS, no launch geometry from the dispatch packet.
// Parameters follow the reference GEMM's order (tk/src/kernels/gemm.rs:604-645: the operands, the bias, the
// rotary tables, the output): x, w, bias (address 0: none), cos, sin (unread by the kernels that do not turn),
// y, then rows (batch * seq), n, k, seq, heads (the first heads * head size columns are turned).
// Launch: ceil(rows / 256) * ceil(n / 256) workgroups, rounded up to a multiple of 8, of 512 threads
// (`workgroups` in the manifest); rows < 2^31, n a multiple of 8, k a multiple of 32 are the caller's checks.
template <bool F16, int HD>
__device__ __forceinline__ void linear_entry(uint8_t *smem, const uint16_t *x, const uint16_t *w, const uint16_t *bias,
                                             const uint16_t *cos_t, const uint16_t *sin_t, uint16_t *y, int32_t rows,
                                             int32_t n, int32_t k, int32_t seq, int32_t heads) {
  if (rows <= 0 || n <= 0 || k <= 0) return;
  // The code objects hold the 256 x 256 form, with the library's launch geometry.
  const uint32_t tiles_n = ((uint32_t)n + Large::kBn - 1) / Large::kBn;
  const uint32_t tiles = ((uint32_t)rows + Large::kBm - 1) / Large::kBm * tiles_n;
  linear_body<F16, HD, Large>(smem, x, w, bias, cos_t, sin_t, y, (int64_t)n, (int64_t)rows, n, k, seq > 0 ? seq : 1, heads,
                              tiles_n, tiles, (tiles + kXcds - 1) / kXcds);
}

#define SVODK_LINEAR_ENTRY(NAME, F16, HD)                                                                             \
  extern "C" __global__ __launch_bounds__(Large::kWaves * 64, 2) void NAME(                                                    \
      const uint16_t *__restrict__ x, const uint16_t *__restrict__ w, const uint16_t *__restrict__ bias,              \
      const uint16_t *__restrict__ cos_t, const uint16_t *__restrict__ sin_t, uint16_t *__restrict__ y, int32_t rows, \
      int32_t n, int32_t k, int32_t seq, int32_t heads) {                                                             \
    __shared__ __attribute__((aligned(1024))) uint8_t smem[Large::kLds];                                                     \
    linear_entry<F16, HD>(smem, x, w, bias, cos_t, sin_t, y, rows, n, k, seq, heads);                                 \
  }
SVODK_LINEAR_ENTRY(svodk_linear_bf16, false, 0)
SVODK_LINEAR_ENTRY(svodk_linear_rope64_bf16, false, 64)
SVODK_LINEAR_ENTRY(svodk_linear_rope128_bf16, false, 128)
SVODK_LINEAR_ENTRY(svodk_linear_f16, true, 0)
SVODK_LINEAR_ENTRY(svodk_linear_rope64_f16, true, 64)
SVODK_LINEAR_ENTRY(svodk_linear_rope128_f16, true, 128)
#undef SVODK_LINEAR_ENTRY
}  // namespace
}  // namespace svodk
#endif  // SVODK_CODE_OBJECT

#if !defined(SVODK_CODE_OBJECT)
// A fill's lanes address their rows with 32-bit byte offsets from the descriptor's base: 8 rows of 2 k bytes,
// and the stage's place along them.
bool linear_supports(int64_t n, int64_t k) { return n > 0 && n % 8 == 0 && k >= 32 && k % 32 == 0 && k <= (1 << 25); }

bool linear_turns(int32_t head_dim) { return head_dim == 64 || head_dim == 128; }

namespace {
std::atomic<int> g_linear_tile{0};  // 0: by the shape; 128 or 256: every call
}
int linear_tile(int32_t tile) {
  if (tile == 0 || tile == 128 || tile == 256) g_linear_tile.store(tile, std::memory_order_relaxed);
  return g_linear_tile.load(std::memory_order_relaxed);
}

LinearTile linear_tile_of(int64_t rows, int64_t n, int64_t k, int head_dim, int units) {
  const int named = g_linear_tile.load(std::memory_order_relaxed);
  if (named != 0) return named == 128 ? kTile128x128 : kTile256x256;
  auto tiles = [&](int64_t bm, int64_t bn) { return ((rows + bm - 1) / bm) * ((n + bn - 1) / bn); };
  // A product with fewer than a compute unit's worth of tiles each wants as many compute units as it can get: the
  // smallest tile that does not make more workgroups than there are units ([16, 1024] x [4096, 1024] 3.6 us in 16 x 16
  // tiles, 5.2 in 64 x 64; 256 rows 19.6 and 7.1).  From k = 512 on: eight waves share k out a line at a time, and a
  // shorter loop is all start and store whatever the tile.
  if (k >= 512 && k <= kLinearFewMaxK) {
    if (tiles(16, 16) <= units) return kFew16x16;
    if (tiles(32, 16) <= units) return kFew32x16;
    if (tiles(32, 32) <= units) return kFew32x32;
    if (tiles(64, 32) <= units) return kFew64x32;
    if (tiles(64, 64) <= units) return kFew64x64;
  }
  // A head of 128 does not fit the 64 columns' two halves.
  if (k >= 512 && head_dim != 128 && tiles(128, 64) <= units) return kTile128x64;
  // What is left is priced by rounds of workgroups over the part.  A round took, at k = 1024 and n = 3072 and 4096: 29 us
  // of 256 x 256 tiles, 22 of 256 x 192 (whose 96 columns a wave hold no whole heads to turn), 16 of two 128 x 128 tiles
  // a unit, 10 of one.
  const int64_t large = tiles(256, 256), wide = tiles(256, 192), mid = tiles(128, 128);
  auto rounds = [](int64_t t, int64_t each) { return (t + each - 1) / each; };
  const int64_t cost_large = 58 * rounds(large, units), cost_wide = 44 * rounds(wide, units);
  const int64_t left = mid % (2 * units);
  const int64_t cost_mid = 32 * (mid / (2 * units)) + (left == 0 ? 0 : left <= units ? 20 : 32);
  if (head_dim == 0 && cost_wide < cost_large && cost_wide < cost_mid) return kTile256x192;
  return cost_mid < cost_large ? kTile128x128 : kTile256x256;
}

const char *linear_config(const LinearArgs &a) {
  static const char *const kText[9][2] = {
#define SVODK_GEMM(BM, BN, STAGES, WARPS)                                                                          \
  {"GemmCfg { bm: " #BM ", bn: " #BN ", bk: 64, stages: " STAGES ", warps: " WARPS ", epilogue: { bias } }",        \
   "GemmCfg { bm: " #BM ", bn: " #BN ", bk: 64, stages: " STAGES ", warps: " WARPS ", epilogue: { bias, rope } }"},
      SVODK_GEMM(16, 16, "1", "k8") SVODK_GEMM(32, 16, "1", "k8") SVODK_GEMM(32, 32, "1", "k8")
      SVODK_GEMM(64, 32, "1", "k8") SVODK_GEMM(64, 64, "1", "k8") SVODK_GEMM(128, 64, "3", "[4, 1]")
      SVODK_GEMM(128, 128, "2", "[4, 2]") SVODK_GEMM(256, 192, "2", "[4, 2]") SVODK_GEMM(256, 256, "2", "[4, 2]")
#undef SVODK_GEMM
  };
  return kText[a.tile][a.cos != nullptr ? 1 : 0];
}

hipError_t launch_linear(const LinearArgs &a, hipStream_t stream) {
  if (!linear_supports(a.n, a.k)) return hipErrorInvalidValue;
  if (a.cos != nullptr && (!linear_turns(a.head_dim) || a.seq <= 0 || (int64_t)a.heads * a.head_dim > a.n))
    return hipErrorInvalidValue;
  const int hd = a.cos != nullptr ? a.head_dim : 0;
  switch (a.tile) {
    case kTile128x64:
      if (hd == 128) return hipErrorInvalidValue;
      return hd == 0 ? launch_hd<0, Narrow>(a, stream) : launch_hd<64, Narrow>(a, stream);
    case kTile128x128:
      return hd == 0 ? launch_hd<0, Mid>(a, stream) : hd == 64 ? launch_hd<64, Mid>(a, stream) : launch_hd<128, Mid>(a, stream);
    case kTile256x192:
      return hd == 0 ? launch_hd<0, Wide>(a, stream) : hipErrorInvalidValue;
    case kTile256x256:
      return hd == 0 ? launch_hd<0, Large>(a, stream) : hd == 64 ? launch_hd<64, Large>(a, stream) : launch_hd<128, Large>(a, stream);
    default: return launch_linear_few(a, stream);
  }
}

}  // namespace svodk
#endif  // !SVODK_CODE_OBJECT
