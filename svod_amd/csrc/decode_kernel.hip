// The decoder step of flash attention for gfx950: a call whose (batch, KV head) has at most four query rows
// (one new token, or a few, for the heads of a KV head's group), without a causal or per-row mask or a bias.
//
// Such a call is a stream of K and V past a handful of queries (tk/src/kernels/attention.rs:466-924 is the
// program whose results it reproduces; nothing in it is a matrix product worth a matrix instruction): its time is
// the bytes of K and V over what the memory system delivers, and what it delivers is set by the bytes a compute
// unit has in flight.  The tile kernel holds 48 KiB a compute unit in its LDS rings and waits for each step's
// fills before the next; here every lane loads its 16 bytes of a key row straight into registers, several
// rows ahead, with no LDS and no barrier in the loop, and a compute unit holds a few hundred KiB in flight.
//
//   a key row of D elements is shared by D/8 lanes (16 bytes each); a wave instruction takes up to four neighbouring
//   heads' rows of a key (512 bytes in one piece) and as many keys as are left of its 64 lanes: a memory access of 512
//   bytes streams a sixth faster than one of 128 or 256 (loads alone: 16 sequences of 8 heads of 128 over 2100 keys 29.8 ->
//   24.9 us, of 20 heads of 64 over 1500 keys 24.7 -> 21.1; of 1 KiB, 24.8 and 23.8)
//   score:   v_dot2_f32 over the lane's four pairs, summed over the row's lanes by DPP
//   softmax: every lane runs the online form over the keys of its own place in the wave, in the exponent's
//            units (scores scaled first, L365-370); probabilities stay f32 where the tile program rounds them
//            to the operands' type for its second matrix product (L432-444)
//   at the end the places of a wave, then the waves of the workgroup, merge their states (m, l, o) as key
//   splits do (L948-1014), and the workgroup writes the output rows, or with key splits its partial state for
//   combine_kernel (L899-921).
#include <hip/hip_runtime.h>
#include <sys/random.h>

#include <atomic>
#include <chrono>
#include <type_traits>

#include "kernels.h"
#include "launch.h"

namespace svodk {
namespace {

typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kNoKey = -1e30f;   // the running maximum before any key: finite, so that its differences are numbers
constexpr int kMaxWaves = 8;       // waves a workgroup
constexpr int kAhead = 2;          // passes a lane works on at a time, with as many more in flight
constexpr int kWordStride = kArrivalBytes / 8;  // of 64-bit words
constexpr int kCountBits = 7;      // of a word of arrivals: its low bits count, the others are the launch's tag
constexpr uint64_t kEnded = (1 << kCountBits) - 1;  // the count of a (batch, KV head) that is merged
static_assert(kMostMergedSplits < kEnded, "no launch under way counts that far");
constexpr int kMostSharingRows = 64;  // a lane a row

// Waves a workgroup: few workgroups take eight each, so that the launch still has its bytes in flight.
// `heads_splits`: (batch, KV head, split)s of the launch.
__host__ __device__ constexpr int decode_waves(uint32_t heads_splits) { return heads_splits >= 256 ? 4 : kMaxWaves; }
// What the kernel takes: AttnArgs without the fields a decoder step does not have.
struct DecodeArgs {
  const uint16_t *q, *k, *v;
  uint16_t *o;
  const void *key_lens, *key_mask;
  const void *row_map;
  const uint16_t *k_app, *v_app;
  const void *app_lens;
  float *o_part, *m_part, *l_part;
  int64_t q_row_elems, kv_row_elems;
  int32_t lens_i64, mask_bytes, row_map_i64, app_lens_i64;
  int32_t batch, t, tk, heads, kv_heads, group;
  int32_t splits, cached, kv_head_start, cache_rows, app_rows;
  float scale;
  uint64_t *arrivals, tag;  // of a launch that merges its splits itself: a word a (batch, KV head), of any content
};

template <bool F16>
__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
  f32x2 f = {lo, hi};
  if constexpr (F16)
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, f16x2));
  else
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2));
}
// The two 16-bit values of a word as f32.
template <bool F16>
__device__ __forceinline__ f32x2 unpack2(uint32_t x) {
  if constexpr (F16) {
    return __builtin_convertvector(__builtin_bit_cast(f16x2, x), f32x2);
  } else {
    return f32x2{__uint_as_float(x << 16), __uint_as_float(x & 0xffff0000u)};
  }
}
// c + a.lo * b.lo + a.hi * b.hi
template <bool F16>
__device__ __forceinline__ float dot2(uint32_t a, uint32_t b, float c) {
  if constexpr (F16)
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, a), __builtin_bit_cast(f16x2, b), c, false);
  else
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, a), __builtin_bit_cast(bf16x2, b), c, false);
}
// x of the lane a DPP control names.
template <int CTRL>
__device__ __forceinline__ float moved(float x) {
  return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(x), CTRL, 0xf, 0xf, true));
}
// x summed over the LANES (4, 8, 16 or 32) neighbouring lanes that share a key row; every one of them gets the sum.
template <int LANES>
__device__ __forceinline__ float sum_over(float x) {
  x += moved<0xB1>(x);                              // quad_perm [1,0,3,2]
  x += moved<0x4E>(x);                              // quad_perm [2,3,0,1]
  if constexpr (LANES >= 8) x += moved<0x141>(x);   // row_half_mirror
  if constexpr (LANES >= 16) x += moved<0x140>(x);  // row_mirror
  if constexpr (LANES >= 32) x += __shfl_xor(x, 16, 64);
  return x;
}

// The online-softmax state of one query row over some of the keys: the lane's eight output columns.
struct State {
  float m, l, acc[8];
};
// `op` of x and of the lane STEP away (lane l <-> l ^ STEP); op is commutative.
template <int STEP, typename Op>
__device__ __forceinline__ float folded(float x, Op op) {
  const uint32_t u = __float_as_uint(x);
  if constexpr (STEP == 32) {
    const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return op(__uint_as_float(r[0]), __uint_as_float(r[1]));
  } else if constexpr (STEP == 16) {
    const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    return op(__uint_as_float(r[0]), __uint_as_float(r[1]));
  } else if constexpr (STEP == 8) {
    return op(x, moved<0x128>(x));  // row_ror:8
  } else {
    return op(x, __shfl_xor(x, STEP, 64));
  }
}

// Partial states that another workgroup of the launch reads go past the L2s, each of which serves one XCD, and are read
// the same way: stores and loads that are coherent over the device (the instructions' sc1 bit), 16 bytes a lane.
struct Shared {
#if defined(__HIP_DEVICE_COMPILE__)
  __amdgpu_buffer_rsrc_t rsrc;
  static constexpr int kDevice = 16;
  __device__ __forceinline__ void name(float *p, uint32_t bytes) {
    rsrc = __builtin_amdgcn_make_buffer_rsrc(p, 0, (int)bytes, 0x00020000);
  }
  __device__ __forceinline__ void put4(uint32_t at, const f32x4 &x) const {
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, x), rsrc, (int)at, 0, kDevice);
  }
  __device__ __forceinline__ void put2(uint32_t at, const f32x2 &x) const {
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, x), rsrc, (int)at, 0, kDevice);
  }
  __device__ __forceinline__ f32x4 got4(uint32_t at) const {
    return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)at, 0, kDevice));
  }
  __device__ __forceinline__ f32x2 got2(uint32_t at) const {
    return __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(rsrc, (int)at, 0, kDevice));
  }
#endif
};

// Keys and values are read once a step, and by the next step the other layers' caches and the weights have been through
// the chip.  Without the mark a step of 34 sequences over 570 cached keys is faster on one layer called back to back (32.2
// -> 25.5 us with two layers' windows in turn), and slower over a model's (8 layers 30.5 -> 32.4, 16 layers 28.1 -> 30.3; 20 over
// 440 keys 15.8 -> 17.2, 8 over 2000 24.0 -> 24.9).
// The 16 bytes `off` past `base`, or zeros from `bytes` on.
__device__ __forceinline__ u32x4 load16(const uint8_t *base, uint32_t bytes, uint32_t off) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int kReadOnce = 2;  // the instruction's nt bit
  const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(base), 0, (int)bytes, 0x00020000);
  return __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)off, 0, kReadOnce);
#else
  return u32x4{};
#endif
}

// A value that every lane of a wave has, in a scalar register.
__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }

// The b-th of an array of 32- or 64-bit integers, as it comes from memory.
struct Integer {
  int lo, hi;
  bool wide;
};
__device__ __forceinline__ Integer ask(const void *p, int b, bool wide) {
  const int *at = (const int *)p + (wide ? 2 * (int64_t)b : (int64_t)b);
  return {at[0], at[wide ? 1 : 0], wide};
}
// The integer held in [0, most].
__device__ __forceinline__ int held(const Integer &x, int most) {
  int n = x.lo;
  if (x.wide) n = x.hi < 0 ? 0 : (x.hi > 0 || x.lo < 0 ? 0x7fffffff : x.lo);
  return n < 0 ? 0 : (n < most ? n : most);
}
// x summed over the lanes up to and with this one.
__device__ __forceinline__ int prefix_sum(int x) {
#if defined(__HIP_DEVICE_COMPILE__)
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);  // row_shr:1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true);
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true);
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1 and 3
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2 and 3
#endif
  return x;
}

// What a launch does with its splits: it has none; it leaves partial states for combine_kernel; the workgroup of a
// (batch, KV head) that ends last merges them; that too, of splits that the rows share out by their lengths.
enum { kWhole, kPartial, kMerged, kShared };

// The workgroup's program for `nw` waves (8 or 4) and 1 << hg_log2 heads, for the kernels below to inline.  ROOM: LDS for the
// states of one head of eight waves, or of two.
template <int D, int R, bool F16, int MODE, int ROOM>
__device__ __forceinline__ void decode_body(const DecodeArgs &p, const int nw, const int hg_log2) {
#if defined(__HIP_DEVICE_COMPILE__)
  // No contraction beyond the fused multiply-adds written out below: the library's kernel (its wave count a launch
  // argument) and a code object's (four waves, known to the compiler) are then the same arithmetic bit for bit.
#pragma clang fp contract(off)
  constexpr int kWide = D == 48 ? 64 : D;
  constexpr int LPK = kWide / 8;   // lanes a head's share of a key row
  constexpr int U = kAhead;  // the same for every R: a row's arithmetic does not depend on how many rows share the keys
  __shared__ __attribute__((aligned(16))) float merged[ROOM * kMaxWaves * R * LPK * 10];

  constexpr bool SPLIT = MODE != kWhole, MERGES = MODE == kMerged || MODE == kShared;
  const uint32_t wg = __builtin_amdgcn_workgroup_id_x();
  const int tid = (int)__builtin_amdgcn_workitem_id_x();
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // A workgroup's heads lie side by side in a key row; neighbouring workgroups take neighbouring heads, then the splits.
  const int hg = 1 << hg_log2, kpi = 64 / LPK >> hg_log2;  // heads, and key rows a wave instruction
  const int span = LPK << hg_log2;                         // lanes a key row
  const uint32_t groups = (uint32_t)p.kv_heads >> hg_log2;
  const uint32_t of_heads = wg / groups;
  const int group0 = (int)(wg - of_heads * groups);
  const int pos = lane % LPK;                       // which 16 bytes of a head
  const int kvh = (group0 << hg_log2) + (lane / LPK & (hg - 1));
  const int slot = lane / LPK >> hg_log2;           // which row of a wave instruction
  const bool pos_ok = 8 * pos < D;

  const int pass = nw * kpi, chunk = U * pass;  // key rows of a pass of the waves, and of a chunk of U passes
  static_assert(U == 2 && kMaxWaves == 8, "a chunk's rows are a power of two");
  const int chunk_log2 = __builtin_ctz(U * 64 / LPK) + (nw == kMaxWaves ? 3 : 2) - hg_log2;

  // The rows: row r is token r % t of the group's head r / t (a grouped tile's order).
  const int rows = p.group * p.t;
  // The batch row of this workgroup, which of the row's `turns` splits it is, and the row's integers: its length
  // (L533-536: len = min(key_lens[b], tk)), where it lies in a cache (L544-550) and how many appended rows it sees (the
  // last split scores them).  The integers are asked for together: one trip to memory for the three, so no load stands
  // under a branch and what a call does not have is read from q and dropped.
  const int tk = p.tk;
  const bool has_lens = p.key_lens != nullptr, has_map = p.cached && p.row_map != nullptr;
  const bool has_app = p.cached && p.k_app != nullptr;
  int b, split = 0, turns = 1, len, kv_row, app_seen;
  Integer len_b, row_b, seen_b;
  bool appends = has_app, has_seen = has_app && p.app_lens != nullptr;
  uint32_t place0 = 0;  // of a launch whose rows share its splits: the first of the row's places
  if constexpr (MODE == kShared) {
    // A row takes one of the launch's batch * splits places and, of the others, what its keys are of all rows' keys: with
    // the same count for each row the launch waits for its longest rows while most compute units have run out of keys.  16
    // sequences of 8 KV heads of 128 over 210 to 2100 cached keys 22.7 -> 18.9 us, over 525 to 2100 23.0 -> 21.0, over 1260 to
    // 2100 23.9 -> 24.2, over 2100 each 25.35 -> 25.55 (the lanes' sum); of 20 heads of 64 over 150 to 1500 20.0 -> 18.4, over
    // 900 to 1500 22.1 -> 21.75, over 1500 each 25.15 -> 25.45.  Every workgroup finds the rows' places for itself, a lane a
    // row, with a sum over the lanes and nothing else: a search for the shares that leave the longest split least cost
    // 0.8 us a launch, what it won.
    const bool there = lane < p.batch;
    const int row = there ? lane : 0;
    len_b = ask(p.key_lens, row, p.lens_i64 != 0);
    row_b = ask(has_map ? p.row_map : p.key_lens, row, has_map ? p.row_map_i64 != 0 : p.lens_i64 != 0);
    seen_b = ask(has_seen ? p.app_lens : p.key_lens, row, has_seen ? p.app_lens_i64 != 0 : p.lens_i64 != 0);
    const int row_len = there ? held(len_b, tk) : 0;
    const int weight = (row_len + chunk - 1) >> chunk_log2, up_to = prefix_sum(weight);
    const int others = p.batch * (p.splits - 1);
    const float each = (float)others * __builtin_amdgcn_rcpf((float)max(__builtin_amdgcn_readlane(up_to, 63), 1));
    // (Rows of one length share alike: what rounding, the reciprocal's too, takes off a sum is put back.)
    auto place = [&](int row, int keys) { return row + min((int)((float)keys * each + 0.01f), others); };
    const int from = place(lane, up_to - weight), to = place(lane + 1, up_to);
    const uint64_t mine = __builtin_amdgcn_ballot_w64(there && from <= (int)of_heads && (int)of_heads < to);
    if (mine == 0) return;  // the last places may be left to no one
    b = __builtin_ctzll(mine);
    place0 = (uint32_t)__builtin_amdgcn_readlane(from, b);
    turns = min(__builtin_amdgcn_readlane(to, b) - (int)place0, kMostMergedSplits);
    split = (int)(of_heads - place0);
    if (split >= turns) return;
    len = __builtin_amdgcn_readlane(row_len, b);
    kv_row = has_map ? __builtin_amdgcn_readlane(held(row_b, p.cache_rows - 1), b) : b;
    app_seen = !has_app || split != turns - 1 ? 0 : has_seen ? __builtin_amdgcn_readlane(held(seen_b, p.app_rows), b) : p.app_rows;
  } else {
    b = SPLIT ? (int)(of_heads / (uint32_t)p.splits) : (int)of_heads;
    if (SPLIT) split = (int)of_heads - b * p.splits, turns = p.splits;
    appends = has_app && (!SPLIT || split == turns - 1), has_seen = appends && p.app_lens != nullptr;
    len_b = ask(has_lens ? p.key_lens : p.q, has_lens ? b : 0, p.lens_i64 != 0 && has_lens);
    row_b = ask(has_map ? p.row_map : p.q, has_map ? b : 0, p.row_map_i64 != 0 && has_map);
    seen_b = ask(has_seen ? p.app_lens : p.q, has_seen ? b : 0, p.app_lens_i64 != 0 && has_seen);
  }
  uint32_t qf[R][4];
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int rr = min(r, rows - 1);
    const int in_group = (rr >= p.t) + (rr >= 2 * p.t) + (rr >= 3 * p.t);
    const int q_row = rr - in_group * p.t;
    const int q_head = kvh * p.group + in_group;
    const uint16_t *at = p.q + ((int64_t)b * p.t + q_row) * p.q_row_elems + (int64_t)q_head * D + 8 * pos;
    u32x4 x = {0, 0, 0, 0};
    if (pos_ok && r < rows) x = *reinterpret_cast<const u32x4 *>(at);
#pragma unroll
    for (int i = 0; i < 4; i++) qf[r][i] = x[i];
  }
  if constexpr (MODE != kShared) {
    asm volatile("" : "+s"(len_b.lo), "+s"(len_b.hi), "+s"(row_b.lo), "+s"(row_b.hi), "+s"(seen_b.lo), "+s"(seen_b.hi));
    len = has_lens ? uniform(held(len_b, tk)) : tk;
    kv_row = has_map ? uniform(held(row_b, p.cache_rows - 1)) : b;
    app_seen = !appends ? 0 : has_seen ? uniform(held(seen_b, p.app_rows)) : p.app_rows;
  }
  const int unit = b * (int)groups + group0;
  // The output row of this lane's head's row r.
  auto out_row = [&](int r, int kv_head) {
    const int in_group = (r >= p.t) + (r >= 2 * p.t) + (r >= 3 * p.t);  // r / t: at most four rows
    return ((int64_t)b * p.t + (r - in_group * p.t)) * p.heads + kv_head * p.group + in_group;
  };
  const float c_exp = p.scale * kLog2e;  // L619
  State st[R];
#pragma unroll
  for (int r = 0; r < R; r++) {
    st[r].m = kNoKey;
    st[r].l = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; j++) st[r].acc[j] = 0.0f;
  }

  // What the workgroup reads: the appended rows (L739-755, L827-846), which the last split scores, the first app_lens[b] of
  // them visible, from tensors of their own, and its chunks of the cached keys.  A pass is nw * kpi rows, a chunk U passes.
  // The splits of a row take its chunks in turn (chunk c is split c % splits's), so that workgroups that run together
  // read keys that lie together, and a workgroup starts some of its chunks in and wraps: the softmax does not care, and
  // the memory does.  Rows of a cache are very often a power of two apart, and so are the batch rows; workgroups that
  // all walk from key 0 then ask the same few memory channels for their rows at the same time.  Started by the cache row,
  // not by who asks: a batch lane mapped to another cache row reads it as that row's own lane would.
  const uint32_t of_row = ((uint32_t)len + (uint32_t)chunk - 1) >> chunk_log2;
  const int chunks = of_row > (uint32_t)split ? (int)((of_row - (uint32_t)split + (uint32_t)turns - 1) / (uint32_t)turns) : 0;
  const int first = (int)__umulhi((uint32_t)kv_row * 0x9e3779b1u, (uint32_t)chunks);  // a fraction that rows differ in
  const uint32_t in_row = (uint32_t)((lane / LPK & (hg - 1)) * (D * 2) + 16 * pos);
  const void *mask = nullptr;  // visibility bytes or words of the cached keys (rows share splits out by lengths, never with one)
  if (MODE != kShared && p.key_mask != nullptr) mask = (const uint8_t *)p.key_mask + (int64_t)b * tk * p.mask_bytes;

  struct Rows {
    u32x4 k[U], v[U];
    int there[U];  // rows of a pass's wave instruction that are there: lanes past them land zeros
    int seen[U];   // of a call with a key mask: this lane's element of it
  };
  // Rows of one tensor each, `row_bytes` apart, keys [0, to).
  struct Source {
    const uint8_t *k, *v;
    uint32_t row_bytes, off;  // off: of this lane's 16 bytes from a wave instruction's first row
    int to;
  };
  auto source = [&](const uint16_t *k, const uint16_t *v, int64_t at, uint32_t row_bytes, int to) {
    return Source{(const uint8_t *)(k + at), (const uint8_t *)(v + at), row_bytes,
                  pos_ok ? (uint32_t)slot * row_bytes + in_row : 0xfffffff0u, to};
  };
  // The rows of the chunk that starts at key `from`, asked for.  A wave instruction's rows are one descriptor, bounded at the
  // rows that are there: no load stands under a branch, so the compiler knows how many are out and waits for the ones it
  // needs alone.  (With a branch a load it waited for all of them, the chunk just asked for among them, before it
  // worked on the one before: with the heads together 16 sequences of 8 KV heads of 128 over 525 to 2100 keys 29.1 -> 24.6
  // us, over 2100 keys each 40.8 -> 28.9.)
  auto load = [&](auto masked, Rows &x, const Source &y, int from) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int key = from + u * pass + wave * kpi;
      int there = max(y.to - key, 0);
      asm("" : "+s"(there));  // on the scalar unit: the compiler makes a vector instruction of the two
      there = min(there, kpi);
      const uint64_t at = (uint64_t)(uint32_t)key * y.row_bytes;
      x.there[u] = there;
      x.k[u] = load16(y.k + at, (uint32_t)there * y.row_bytes, y.off);
      x.v[u] = load16(y.v + at, (uint32_t)there * y.row_bytes, y.off);
      if constexpr (decltype(masked)::value) {
        x.seen[u] = 0;
        if (slot < there)
          x.seen[u] = p.mask_bytes == 1 ? (int)((const uint8_t *)mask)[key + slot] : ((const int *)mask)[key + slot];
      }
    }
  };
  // The softmax and the second product of the U passes in `x`.
  auto work = [&](auto masked, Rows &x) {
    float e[U][R];
#pragma unroll
    for (int u = 0; u < U; u++) {
      bool seen = slot < x.there[u];
      if constexpr (decltype(masked)::value) {
        seen = x.seen[u] != 0;
        if (!seen) x.v[u] = u32x4{0, 0, 0, 0};  // a hidden row weighs nothing, whatever it holds
      }
#pragma unroll
      for (int r = 0; r < R; r++) {
        float s = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; i++) s = dot2<F16>(x.k[u][i], qf[r][i], s);
        s = sum_over<LPK>(s);
        e[u][r] = seen ? s * c_exp : -__builtin_inff();
      }
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
      float m = st[r].m;
#pragma unroll
      for (int u = 0; u < U; u++) m = __builtin_fmaxf(m, e[u][r]);
      const float corr = __builtin_amdgcn_exp2f(st[r].m - m);
      st[r].m = m;
      st[r].l *= corr;
#pragma unroll
      for (int j = 0; j < 8; j++) st[r].acc[j] *= corr;
      float pr[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
        pr[u] = __builtin_amdgcn_exp2f(e[u][r] - m);
        st[r].l += pr[u];
      }
#pragma unroll
      for (int u = 0; u < U; u += 2) {
        const float held[2] = {pr[u], pr[u + 1]};
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const f32x2 a = unpack2<F16>(x.v[u][i]), c = unpack2<F16>(x.v[u + 1][i]);
          st[r].acc[2 * i] = __builtin_fmaf(held[0], a[0], st[r].acc[2 * i]);
          st[r].acc[2 * i + 1] = __builtin_fmaf(held[0], a[1], st[r].acc[2 * i + 1]);
          st[r].acc[2 * i] = __builtin_fmaf(held[1], c[0], st[r].acc[2 * i]);
          st[r].acc[2 * i + 1] = __builtin_fmaf(held[1], c[1], st[r].acc[2 * i + 1]);
        }
      }
    }
  };
  // Two sets of rows take turns: one is worked on while the other is on its way.  A set past the last chunk has no rows.
  auto stream = [&](auto masked) {
    const int kv_col = (group0 << hg_log2) + (p.cached ? p.kv_head_start : 0);
    const Source cache = source(p.k, p.v, (int64_t)kv_row * tk * p.kv_row_elems + (int64_t)kv_col * D,
                                (uint32_t)p.kv_row_elems * 2, len);
    auto chunk_of = [&](int i) {
      int c = first + i;
      c = c >= chunks ? c - chunks : c;
      return i < chunks ? (split + c * turns) * chunk : len;
    };
    Rows one, two;
    const Source app = source(p.k_app, p.v_app, ((int64_t)b * p.app_rows * p.kv_heads + (group0 << hg_log2)) * D,
                              (uint32_t)p.kv_heads * (D * 2), app_seen);
    int app_from = 0;
    for (; app_from + chunk < app_seen; app_from += chunk) {
      load(std::false_type(), two, app, app_from);
      work(std::false_type(), two);
    }
    if (app_from < app_seen) {
      load(std::false_type(), two, app, app_from);
      load(masked, one, cache, chunk_of(0));  // under way with the last of them
      __builtin_amdgcn_sched_barrier(0);
      work(std::false_type(), two);
    } else {
      load(masked, one, cache, chunk_of(0));
    }
    for (int i = 0; i < chunks; i += 2) {
      load(masked, two, cache, chunk_of(i + 1));
      __builtin_amdgcn_sched_barrier(0);
      work(masked, one);
      if (i + 1 >= chunks) break;
      __builtin_amdgcn_sched_barrier(0);
      load(masked, one, cache, chunk_of(i + 2));
      __builtin_amdgcn_sched_barrier(0);
      work(masked, two);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // A word of arrivals is the workspace's and holds anything at first.  Every workgroup makes sure, before it counts
  // itself in, that the word carries this launch's tag: it becomes (tag, 0) by one compare-and-swap out of whatever was
  // there, and no other write of the launch leaves that tag again, so a late swap out of the old content fails.  Nothing
  // else ever carries the tag (57 bits, another one a launch) but the word as an earlier replay of the same captured
  // launch left it, and that one counts kEnded, which no word of a launch under way does: the workgroup that merges leaves
  // it behind (`splits` would not do, a row's share of them is another with other lengths).  The content is asked for ahead of the keys and the swap goes out behind them, so
  // that neither is waited for: with the swap ahead of the keys a launch takes 1.4 us more.
  uint64_t *arrivals = p.arrivals + (int64_t)unit * kWordStride;
  const bool counts = MERGES && tid == 0;
  uint64_t found = 0;
  if (counts) found = __hip_atomic_load(arrivals, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  // A wave that no row of the split's first chunk falls to has none at all, and its state stays as it is (8 KV heads of 64 over
  // 16 keys 4.0 -> 3.5 us, 64 sequences of 12 of 32 4.9 -> 4.3).
  const bool has_rows = app_seen > 0 || split * chunk + wave * kpi < len;
  if (has_rows) {
    if (mask != nullptr)
      stream(std::true_type());
    else
      stream(std::false_type());
  }
  if (counts && (found >> kCountBits != p.tag || (int)(found & ((1u << kCountBits) - 1)) >= turns))
    __hip_atomic_compare_exchange_strong(arrivals, &found, p.tag << kCountBits, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
  // The places of a wave that share output columns (lanes `span` apart) merge (L948-1014): the greatest maximum, what each
  // state weighs under it, the sums.  A step of it takes all values under one branch: their exchanges are then out together.
  // (A value's steps one after the other, each under a branch of its own, waited for every exchange by itself: 8 KV heads of 32
  // over 100 keys 4.76 -> 4.24 us, 16 sequences of 8 KV heads of 32 with two rows each 6.4 -> 5.3, of 64 5.5 -> 5.0, Whisper's
  // cross-attention 23.3 -> 23.0; the same bits.)
  auto over_places = [&](auto fold) {
    if (LPK <= 4 && 4 >= span) fold(std::integral_constant<int, 4>());
    if (LPK <= 8 && 8 >= span) fold(std::integral_constant<int, 8>());
    if (LPK <= 16 && 16 >= span) fold(std::integral_constant<int, 16>());
    if (32 >= span) fold(std::integral_constant<int, 32>());
  };
  float most[R];
#pragma unroll
  for (int r = 0; r < R; r++) most[r] = st[r].m;
  over_places([&](auto step) {
#pragma unroll
    for (int r = 0; r < R; r++)
      most[r] = folded<decltype(step)::value>(most[r], [](float x, float y) { return __builtin_fmaxf(x, y); });
  });
#pragma unroll
  for (int r = 0; r < R; r++) {
    const float w = __builtin_amdgcn_exp2f(st[r].m - most[r]);
    st[r].m = most[r];
    st[r].l *= w;
#pragma unroll
    for (int j = 0; j < 8; j++) st[r].acc[j] *= w;
  }
  over_places([&](auto step) {
    constexpr int kStep = decltype(step)::value;
    auto sum = [](float x, float y) { return x + y; };
#pragma unroll
    for (int r = 0; r < R; r++) {
      st[r].l = folded<kStep>(st[r].l, sum);
#pragma unroll
      for (int j = 0; j < 8; j++) st[r].acc[j] = folded<kStep>(st[r].acc[j], sum);
    }
  });
  // Then the waves do, through LDS, in the same way: the first wave's lanes take a (row, lane of a key row) each and ask for
  // all waves' states of it together.  (One state after the other, each read behind the sums of the one before: 0.17 us a
  // state, 1.9 us more for eight waves of two rows.)
  const int64_t states = (int64_t)p.batch * p.t * p.heads;  // of a split
  // A merging launch's states lie a unit together: [unit][split][row of the unit's heads][D], then their (m, l); the units
  // of a launch whose rows share its splits by heads, then by their places.
  const int unit_rows = rows << hg_log2;
  Shared shared_o, shared_ml;
  if (MERGES) {
    const uint32_t of_unit = (uint32_t)(turns * unit_rows);
    const int64_t before = MODE == kShared ? (int64_t)group0 * p.batch * p.splits + place0 : (int64_t)unit * turns;
    shared_o.name(p.o_part + before * unit_rows * D, of_unit * D * 4);
    shared_ml.name(p.m_part + before * unit_rows * 2, of_unit * 8);
  }
  auto merge_waves = [&](auto waves) {
    constexpr int W = decltype(waves)::value;
    constexpr int kRoom = ROOM * LPK * kMaxWaves / W;  // lanes of a key row that LDS holds the states of
    const int held_log2 = min(__builtin_ctz(kRoom), __builtin_ctz(LPK) + hg_log2), held = 1 << held_log2;
    for (int from = 0; from < span; from += held) {
      if (from > 0) __syncthreads();
      if (lane >= from && lane < from + held) {
#pragma unroll
        for (int r = 0; r < R; r++) {
          f32x2 *at = reinterpret_cast<f32x2 *>(merged + (((wave * R + r) << held_log2) + lane - from) * 10);
          at[0] = f32x2{st[r].m, st[r].l};
#pragma unroll
          for (int j = 0; j < 4; j++) at[1 + j] = f32x2{st[r].acc[2 * j], st[r].acc[2 * j + 1]};
        }
      }
      __syncthreads();
      if (wave != 0) continue;
      for (int item = lane; item < R << held_log2; item += 64) {
        const int r = item >> held_log2, of_row = from + (item & (held - 1));
        f32x2 x[W][5];
#pragma unroll
        for (int w = 0; w < W; w++) {
          const f32x2 *at = reinterpret_cast<const f32x2 *>(merged + ((w * R << held_log2) + item) * 10);
#pragma unroll
          for (int j = 0; j < 5; j++) x[w][j] = at[j];
        }
        float m = x[0][0][0];
#pragma unroll
        for (int w = 1; w < W; w++) m = __builtin_fmaxf(m, x[w][0][0]);
        float l = 0.0f, acc[8] = {};
#pragma unroll
        for (int w = 0; w < W; w++) {
          const float weight = __builtin_amdgcn_exp2f(x[w][0][0] - m);
          l += x[w][0][1] * weight;
#pragma unroll
          for (int j = 0; j < 8; j++) acc[j] += x[w][1 + j / 2][j & 1] * weight;
        }
        const int head = of_row / LPK, at_pos = of_row % LPK;
        if (r >= rows || 8 * at_pos >= D) continue;
        const int64_t orow = out_row(r, (group0 << hg_log2) + head);
        if (MERGES) {
          const uint32_t at = (uint32_t)(split * unit_rows + head * rows + r);
          if (at_pos == 0) shared_ml.put2(at * 8, f32x2{m, l});
          shared_o.put4((at * D + 8 * at_pos) * 4, f32x4{acc[0], acc[1], acc[2], acc[3]});
          shared_o.put4((at * D + 8 * at_pos + 4) * 4, f32x4{acc[4], acc[5], acc[6], acc[7]});
        } else if (SPLIT) {
          // L899-921: the accumulator as it stands, the maximum in the exponent's units, the sum.
          const int64_t at = split * states + orow;
          if (at_pos == 0) {
            p.m_part[at] = m;
            p.l_part[at] = l;
          }
          f32x4 *to = reinterpret_cast<f32x4 *>(p.o_part + at * D + 8 * at_pos);
          to[0] = f32x4{acc[0], acc[1], acc[2], acc[3]};
          to[1] = f32x4{acc[4], acc[5], acc[6], acc[7]};
        } else {
          // L892-898: out = o / (l == 0 ? 1 : l).
          const float inv = 1.0f / (l == 0.0f ? 1.0f : l);
          u32x4 out;
#pragma unroll
          for (int i = 0; i < 4; i++) out[i] = pack2<F16>(acc[2 * i] * inv, acc[2 * i + 1] * inv);
          *reinterpret_cast<u32x4 *>(p.o + orow * D + 8 * at_pos) = out;
        }
      }
    }
  };
  if (nw == kMaxWaves)
    merge_waves(std::integral_constant<int, kMaxWaves>());
  else
    merge_waves(std::integral_constant<int, kMaxWaves / 2>());
  if (!MERGES) return;
  // ---- the merge.  This wave's states are where every workgroup sees them before it counts itself in: they were stored
  // past the L2s, and vmcnt is at zero when the memory behind those has taken them all.  The workgroup that counts itself
  // in last reads them, from there as well.  No one waits for anyone.  The arithmetic is combine_kernel's, operation
  // for operation: a launch that leaves the merge to that kernel gives the same bits.  It is a chain of four
  // trips to memory, some 3 us, where a kernel of its own is a launch (2.6 us of host time) and 3.5 us: with a head a
  // workgroup one sequence over 8000 cached keys 36.1 -> 31.8 us, two over 4700 18.4 -> 16.1, sixteen over 1500 26.1 -> 25.8.
  // In a graph's replay, where a launch costs no host time: one over 8000 22.3 -> 16.7, two over 4700 20.8 -> 17.7, four over
  // 8100 36.1 -> 33.6, sixteen over 1500 26.3 -> 26.6.
  const int splits = turns;
  if (wave == 0) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    uint32_t before = 0;
    if (lane == 0) {
      before = (uint32_t)__hip_atomic_fetch_add(arrivals, (uint64_t)1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      merged[0] = __uint_as_float(before & ((1u << kCountBits) - 1));
    }
  }
  __syncthreads();
  if (uniform((int)__float_as_uint(merged[0])) != splits - 1) return;
  if (tid == 0) __hip_atomic_store(arrivals, p.tag << kCountBits | kEnded, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  asm volatile("" ::: "memory");  // the states are read from here on
  constexpr int kLanes = D / 4;
  // States are asked for `batch` together, the first ones with the maxima of all: two trips to memory for 32 splits.
  auto merge_splits = [&](auto batch) {
    constexpr int kBatch = decltype(batch)::value;
    for (int c = tid; c < hg * rows * kLanes; c += nw * 64) {
      const int of_group = c / kLanes, chunk = c - of_group * kLanes;  // a row of one of the heads, four of its columns
      const int in_heads = (int)((uint32_t)of_group / (uint32_t)rows);
      const int64_t orow = out_row(of_group - in_heads * rows, (group0 << hg_log2) + in_heads);
      f32x2 ml[kBatch];
      f32x4 part[kBatch];
      auto state = [&](int i) { return (uint32_t)(min(i, splits - 1) * unit_rows + of_group); };
      auto ask_states = [&](int from) {
#pragma unroll
        for (int i = 0; i < kBatch; i++) {
          ml[i] = shared_ml.got2(state(from + i) * 8);
          part[i] = shared_o.got4((state(from + i) * D + 4 * chunk) * 4);
        }
      };
      ask_states(0);
      float later = kNoKey;  // the greatest of the maxima past the first states
      for (int from = kBatch; from < splits; from += kBatch) {
        float y[kBatch];
#pragma unroll
        for (int i = 0; i < kBatch; i++) y[i] = shared_ml.got2(state(from + i) * 8)[0];
#pragma unroll
        for (int i = 0; i < kBatch; i++) later = __builtin_fmaxf(later, y[i]);
      }
      float m = later;
#pragma unroll
      for (int i = 0; i < kBatch; i++) m = __builtin_fmaxf(m, ml[i][0]);
      float l = 0.0f, acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
      for (int from = 0; from < splits; from += kBatch) {
        if (from > 0) ask_states(from);
#pragma unroll
        for (int i = 0; i < kBatch; i++) {
          // No branch: the loads would move into it, one trip after the other.
          const bool none = from + i == 0, there = from + i < splits;
          const float w = __builtin_amdgcn_exp2f(ml[i][0] - m);
          const float lw = ml[i][1] * w;
          l = none ? lw : (there ? l + lw : l);
#pragma unroll
          for (int j = 0; j < 4; j++) acc[j] = none ? part[i][j] * w : (there ? acc[j] + part[i][j] * w : acc[j]);
        }
      }
      const float ll = l == 0.0f ? 1.0f : l;
      const u32x2 out = {pack2<F16>(acc[0] / ll, acc[1] / ll), pack2<F16>(acc[2] / ll, acc[3] / ll)};
      *reinterpret_cast<u32x2 *>(p.o + orow * D + 4 * chunk) = out;
    }
  };
  if (splits <= 4)
    merge_splits(std::integral_constant<int, 4>());
  else if (splits <= 8)
    merge_splits(std::integral_constant<int, 8>());
  else
    merge_splits(std::integral_constant<int, 16>());
#endif  // __HIP_DEVICE_COMPILE__
}

#if !defined(SVODK_CODE_OBJECT)  // the library's kernel and its launch: not part of a code object build
// DecodeArgs as they travel: in 112 bytes (launch.h).  k and v are at the launch's first head, the states and the words of
// arrivals behind them are one piece, a row of keys is counted in heads.
struct Packed {
  const uint16_t *q, *k, *v;
  uint16_t *o;
  const void *keys;  // key_lens, key_mask or null
  const void *row_map;
  const uint16_t *k_app, *v_app;
  const void *app_lens;
  float *states;
  uint64_t tag : 64 - kCountBits, app_rows : 7;
  uint64_t splits : 26, kv_row_heads : 19, kv_heads : 16, mask : 1, wide_keys : 1, packed_rows : 1;
  uint32_t batch : 26, group_less_one : 2, t_less_one : 2, row_map_i64 : 1, app_lens_i64 : 1;
  uint32_t tk : 31, heads_lo : 1, cache_rows : 31, heads_hi : 1;  // heads: heads_together's two bits
  float scale;
};
static_assert(sizeof(Packed) <= 112 && kDecodeRows <= 4, "the record's size, the group's and the tokens' two bits");

template <int D, int R, bool F16, int MODE>
__global__ __launch_bounds__(kMaxWaves * 64) void decode_kernel(const Packed a) {
#if defined(__HIP_DEVICE_COMPILE__)
  DecodeArgs p;
  p.q = a.q, p.k = a.k, p.v = a.v, p.o = a.o;
  p.key_lens = a.mask ? nullptr : a.keys, p.key_mask = a.mask ? a.keys : nullptr;
  p.lens_i64 = a.wide_keys, p.mask_bytes = a.wide_keys ? 4 : 1;
  p.row_map = a.row_map, p.row_map_i64 = a.row_map_i64, p.cache_rows = a.cache_rows;
  p.k_app = a.k_app, p.v_app = a.v_app, p.app_lens = a.app_lens, p.app_lens_i64 = a.app_lens_i64, p.app_rows = a.app_rows;
  p.batch = a.batch, p.tk = a.tk, p.t = a.t_less_one + 1, p.group = a.group_less_one + 1;
  p.kv_heads = a.kv_heads, p.heads = p.kv_heads * p.group;
  p.splits = MODE == kWhole ? 1 : (int32_t)a.splits;
  p.kv_row_elems = (int64_t)a.kv_row_heads * D, p.q_row_elems = a.packed_rows ? p.kv_row_elems : (int64_t)p.heads * D;
  p.cached = 1, p.kv_head_start = 0, p.scale = a.scale;
  const int64_t states = (int64_t)p.splits * p.batch * p.t * p.heads;
  p.o_part = a.states, p.m_part = a.states + states * D, p.l_part = p.m_part + states;
  p.arrivals = reinterpret_cast<uint64_t *>(p.l_part + states), p.tag = a.tag;
  const uint32_t heads_splits = (uint32_t)p.batch * (uint32_t)p.kv_heads * (uint32_t)p.splits;  // below 2^31
  decode_body<D, R, F16, MODE, D == 48 || D <= 64 ? 2 : 1>(p, decode_waves(heads_splits), a.heads_lo | a.heads_hi << 1);
#endif
}

template <int D, int R, bool F16>
hipError_t launch_r(const Packed &p, int mode, hipStream_t stream) {
  const int64_t heads_splits = (int64_t)p.batch * p.kv_heads * p.splits;
  if (heads_splits == 0) return hipSuccess;
  const uint32_t threads = (uint32_t)decode_waves((uint32_t)heads_splits) * 64;
  const int64_t grid = heads_splits >> (p.heads_lo | p.heads_hi << 1);
  auto run = [&](auto mode) {
    return Launch<decode_kernel<D, R, F16, decltype(mode)::value>>::run(grid, threads, 0, 0, stream, p);
  };
  switch (mode) {
    case kWhole: return run(std::integral_constant<int, kWhole>());
    case kPartial: return run(std::integral_constant<int, kPartial>());
    case kMerged: return run(std::integral_constant<int, kMerged>());
    default: return run(std::integral_constant<int, kShared>());
  }
}

template <int D>
hipError_t launch_d(const Packed &p, int rows, int mode, bool f16, hipStream_t stream) {
  if (rows <= 1) return f16 ? launch_r<D, 1, true>(p, mode, stream) : launch_r<D, 1, false>(p, mode, stream);
  if (rows <= 2) return f16 ? launch_r<D, 2, true>(p, mode, stream) : launch_r<D, 2, false>(p, mode, stream);
  return f16 ? launch_r<D, 4, true>(p, mode, stream) : launch_r<D, 4, false>(p, mode, stream);
}

// A launch's tag: no two of a process have the same, and where they start differs from process to process.
uint64_t next_tag() {
  static std::atomic<uint64_t> next{[] {
    uint64_t seed = 0;
    if (getrandom(&seed, sizeof seed, GRND_NONBLOCK) != (ssize_t)sizeof seed)
      seed = (uint64_t)std::chrono::steady_clock::now().time_since_epoch().count() * 0x9e3779b97f4a7c15u;
    return seed;
  }()};
  return next.fetch_add(1, std::memory_order_relaxed) & ((uint64_t)-1 >> kCountBits);
}

std::atomic<int> g_decode_rows{kDecodeRowsDefault};

}  // namespace

void attention_decode_rows(int32_t rows) {
  g_decode_rows.store(rows < 0 ? 0 : (rows > kDecodeRows ? kDecodeRows : rows), std::memory_order_relaxed);
}

int32_t attention_decode_limit() { return g_decode_rows.load(std::memory_order_relaxed); }

bool attention_decodes(const AttnArgs &a, int32_t limit) {
  const bool ranged = a.win_left >= 0 || a.chunk_size > 0 || a.seg_start != nullptr;
  if (a.causal || ranged || a.bias != nullptr || a.kv_heads <= 0 || a.heads % a.kv_heads != 0) return false;
  const int64_t rows = (int64_t)(a.heads / a.kv_heads) * a.t;
  return rows >= 1 && rows <= limit;
}

hipError_t launch_decode(const AttnArgs &a, hipStream_t stream) {
  const int splits = a.splits > 1 ? a.splits : 1;
  if (splits > 1 && (a.o_part == nullptr || a.m_part == nullptr || a.l_part == nullptr)) return hipErrorInvalidValue;
  const int64_t q_row = a.q_row_elems > 0 ? a.q_row_elems : (int64_t)a.heads * a.d;
  const int64_t kv_row = a.kv_row_elems > 0 ? a.kv_row_elems : (int64_t)a.kv_heads * a.d;
  const bool packed_rows = q_row != (int64_t)a.heads * a.d;
  // The fields' widths; the op layer's own limits (64 rows of keys in 2^31 bytes, 64 tiles a row and head in 31 bits, 64
  // appended rows) are within them.
  if (kv_row % a.d != 0 || kv_row / a.d >= 1 << 19 || (packed_rows && q_row != kv_row) || a.kv_heads > 0xffff ||
      a.app_rows > 127 || a.batch >= 1 << 26 || splits >= 1 << 26)
    return hipErrorInvalidValue;
  Packed p{};
  p.q = (const uint16_t *)a.q;
  p.k = (const uint16_t *)a.k + (a.cached ? (int64_t)a.kv_head_start * a.d : 0);
  p.v = (const uint16_t *)a.v + (a.cached ? (int64_t)a.kv_head_start * a.d : 0);
  p.o = (uint16_t *)a.o;
  p.keys = a.key_mask != nullptr ? a.key_mask : a.key_lens;
  p.mask = a.key_mask != nullptr;
  p.wide_keys = a.key_mask != nullptr ? a.mask_bytes == 4 : a.lens_i64 != 0;
  if (a.cached) {
    p.row_map = a.row_map;
    p.row_map_i64 = a.row_map_i64 != 0;
    p.cache_rows = (uint32_t)a.cache_rows;
    p.k_app = (const uint16_t *)a.k_app;
    p.v_app = (const uint16_t *)a.v_app;
    p.app_rows = (uint64_t)a.app_rows;
    p.app_lens = a.app_lens;
    p.app_lens_i64 = a.app_lens_i64 != 0;
  }
  p.states = a.o_part;
  p.tk = (uint32_t)a.tk;
  p.batch = (uint32_t)a.batch;
  p.kv_row_heads = (uint64_t)(kv_row / a.d);
  p.scale = a.scale;
  p.splits = (uint64_t)splits;
  p.kv_heads = (uint64_t)a.kv_heads;
  p.group_less_one = (uint32_t)(a.heads / a.kv_heads - 1);
  p.t_less_one = (uint32_t)(a.t - 1);
  p.packed_rows = packed_rows;
  const int64_t heads_splits = (int64_t)a.batch * a.kv_heads * splits;
  if (heads_splits > 0x7fffffffLL) return hipErrorInvalidConfiguration;
  const int together = heads_together(a.d, (uint32_t)heads_splits, (uint32_t)a.kv_heads);
  p.heads_lo = (uint32_t)together & 1;
  p.heads_hi = (uint32_t)together >> 1;
  const int rows = a.heads / a.kv_heads * a.t;
  const bool merged = splits > 1 && a.merges;
  if (merged && splits > kMostMergedSplits) return hipErrorInvalidValue;
  // Rows share the splits out by their lengths; a count that the caller named is every row's.  From four splits a row on: at
  // two, a row that rounding leaves one short reads twice as long (32 sequences over 600 to 1000 keys 23 -> 29 us).  And from
  // 96 MiB of a cache on (8 KV heads of 128, equal splits -> shared): over less the sum over the lanes and the rounding give back
  // what the rows whose lengths differ by less win.  At 80 MiB 4 sequences over 1280 to 5120 keys 17.5 -> 17.3 us, over 3072 to
  // 5120 17.8 -> 18.3, 16 over 768 to 1280 17.2 -> 17.1; at 64 MiB 4 over 2457 to 4096 15.6 -> 16.4; at 112 MiB 4 over 1792 to
  // 7168 22.1 -> 20.8, over 4300 to 7168 22.1 -> 22.3, 8 over 896 to 3584 21.0 -> 18.6, over 2150 to 3584 21.3 -> 20.8.  One
  // length costs 0.1 to 0.2 us.  The line goes by what the cache holds at most, which is what the host knows: of 8192 keys a
  // row, 200 each there take 8.0 us either way, 500 each 8.7 -> 8.8, 100 to 300 8.5 -> 8.0.  The sum holds 2^31 keys.
  const bool shared = merged && a.shares && a.key_lens != nullptr && a.key_mask == nullptr && splits >= 4 &&
                      a.batch >= 4 && a.batch <= kMostSharingRows && (int64_t)a.batch * a.tk < 0x7fffffffLL &&
                      (int64_t)a.batch * a.tk * a.kv_heads * a.d * 4 >= 96 << 20;
  if (merged) p.tag = next_tag();
  const int mode = splits == 1 ? kWhole : !merged ? kPartial : shared ? kShared : kMerged;
  switch (a.d) {
    case 32: return launch_d<32>(p, rows, mode, a.f16 != 0, stream);
    case 48: return launch_d<48>(p, rows, mode, a.f16 != 0, stream);
    case 64: return launch_d<64>(p, rows, mode, a.f16 != 0, stream);
    case 128: return launch_d<128>(p, rows, mode, a.f16 != 0, stream);
    case 256: return launch_d<256>(p, rows, mode, a.f16 != 0, stream);
  }
  return hipErrorInvalidValue;
}

}  // namespace svodk

#else  // SVODK_CODE_OBJECT
}  // namespace
}  // namespace svodk
// ---------------------------------------------------------------------------------------------
// The same program as kernels a loader outside the HIP runtime can run (a flat argument record, static LDS, no
// dispatch packet: the workgroup is 256 threads, which the kernel cannot ask and therefore fixes).  One kernel an
// instantiation, svodk_decode_d<D>_r<rows>_<type>_s<split>, all with one record.  Buffers, an address of 0 for what
// a call does not have: q, k, v, o, key_lens, key_mask, row_map, k_app, v_app, app_lens, then the partial states of
// a split call o_part, m_part, l_part.  Scalars: batch, t, tk, heads, kv_heads, scale_bits, lens_i64, mask_bytes (1 or
// 4), q_row_elems, kv_row_elems (0: heads * D and kv_heads * D), splits, cached, kv_head_start, row_map_i64,
// cache_rows, app_rows, app_lens_i64.  Launch: batch * kv_heads * (s ? splits : 1) workgroups of 256 threads; r is
// the least of 1, 2, 4 that holds heads / kv_heads * t.
// ---------------------------------------------------------------------------------------------
#define SVODK_DECODE_ENTRY(D, R, T, F16, S)                                                                           \
  extern "C" __global__ __launch_bounds__(256) void svodk_decode_d##D##_r##R##_##T##_s##S(                            \
      const uint16_t *__restrict__ q, const uint16_t *__restrict__ k, const uint16_t *__restrict__ v,                 \
      uint16_t *__restrict__ o, const void *__restrict__ key_lens, const void *__restrict__ key_mask,                 \
      const void *__restrict__ row_map, const uint16_t *__restrict__ k_app, const uint16_t *__restrict__ v_app,       \
      const void *__restrict__ app_lens, float *__restrict__ o_part, float *__restrict__ m_part,                      \
      float *__restrict__ l_part, int32_t batch, int32_t t, int32_t tk, int32_t heads, int32_t kv_heads,              \
      int32_t scale_bits, int32_t lens_i64, int32_t mask_bytes, int32_t q_row_elems, int32_t kv_row_elems,            \
      int32_t splits, int32_t cached, int32_t kv_head_start, int32_t row_map_i64, int32_t cache_rows,                 \
      int32_t app_rows, int32_t app_lens_i64) {                                                                       \
    if (batch <= 0 || t <= 0 || tk < 0 || kv_heads <= 0 || heads < kv_heads) return;                                  \
    svodk::DecodeArgs p;                                                                                              \
    p.q = q, p.k = k, p.v = v, p.o = o, p.key_lens = key_lens, p.key_mask = key_mask, p.row_map = row_map;            \
    p.k_app = k_app, p.v_app = v_app, p.app_lens = app_lens, p.o_part = o_part, p.m_part = m_part, p.l_part = l_part; \
    p.q_row_elems = q_row_elems > 0 ? q_row_elems : heads * D;                                                        \
    p.kv_row_elems = kv_row_elems > 0 ? kv_row_elems : kv_heads * D;                                                  \
    p.lens_i64 = lens_i64, p.mask_bytes = mask_bytes, p.row_map_i64 = row_map_i64, p.app_lens_i64 = app_lens_i64;     \
    p.batch = batch, p.t = t, p.tk = tk, p.heads = heads, p.kv_heads = kv_heads, p.group = heads / kv_heads;          \
    p.splits = (S) && splits > 1 ? splits : 1, p.cached = cached, p.kv_head_start = kv_head_start;                    \
    p.cache_rows = cache_rows, p.app_rows = app_rows, p.scale = __builtin_bit_cast(float, scale_bits);                \
    p.arrivals = nullptr, p.tag = 0;                                                                                  \
    const uint32_t heads_splits = (uint32_t)batch * (uint32_t)kv_heads * (uint32_t)p.splits;                          \
    const int hg_log2 = svodk::heads_together(D, heads_splits, kv_heads);                                            \
    if (__builtin_amdgcn_workgroup_id_x() >= heads_splits >> hg_log2) return; /* launch: a (batch, KV head, split) */ \
    svodk::decode_body<D, R, F16, (S) != 0 ? svodk::kPartial : svodk::kWhole, 1>(                                        \
        p, 4, hg_log2);                                                                                               \
  }
#define SVODK_DECODE_ROWS_OF(D, T, F16, S) \
  SVODK_DECODE_ENTRY(D, 1, T, F16, S) SVODK_DECODE_ENTRY(D, 2, T, F16, S) SVODK_DECODE_ENTRY(D, 4, T, F16, S)
#define SVODK_DECODE_FAMILY(D)                                              \
  SVODK_DECODE_ROWS_OF(D, bf16, false, 0) SVODK_DECODE_ROWS_OF(D, bf16, false, 1) \
  SVODK_DECODE_ROWS_OF(D, f16, true, 0) SVODK_DECODE_ROWS_OF(D, f16, true, 1)
SVODK_DECODE_FAMILY(32) SVODK_DECODE_FAMILY(48) SVODK_DECODE_FAMILY(64) SVODK_DECODE_FAMILY(128) SVODK_DECODE_FAMILY(256)
#endif  // SVODK_CODE_OBJECT
