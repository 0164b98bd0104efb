// qf_spec_attn.hip — split-KV, GQA-packed verification attention for MI355X (gfx950).
//
// Causal attention for a uniform speculative-decode batch (every request has q_len query tokens)
// over a paged bf16 KV cache; the C ABI is declared in include/qf_spec_attn.h.  Same decomposition
// as the reference (plugin/qwen_fastpath/spec_attn.py:1-10): the cached prefix, which every query of a
// request sees in full, is split across workgroups that stream each kv head once for all the
// q_len * G query rows sharing it; a second kernel attends this step's q_len positions causally and
// merges everything by log-sum-exp.  The kernels themselves are designed for CDNA4:
//
//   prefix kernel, one workgroup of 4 or 8 wavefronts per (split, kv head, request); the last active split also takes
//   this step's q_len in-flight positions, masked causally per query row:
//   * A stage is one 16-position key tile a wavefront.  Each wavefront copies its tile's K and V rows global -> LDS with
//     16-byte direct-to-LDS loads (no VGPR staging), 16-byte pieces XOR-swizzled per row so that the MFMA fragment reads
//     below are free of bank conflicts, into two slots of its own per tensor: the K of the stage after next and the V of
//     the next stage are in flight while a stage is computed (64 KiB a workgroup at D = 256).
//   * S^T = K . Q^T on v_mfma_f32_16x16x32_bf16 with K as the A operand (16 positions x 32 d) and the packed query rows
//     as B (16 rows), each wavefront its own key tile and every row: no score is computed twice.  A lane's accumulator
//     holds 4 positions of ONE row.
//   * The softmax weights (rounded to bf16) meet in LDS, and each wavefront multiplies its own share of the head
//     dimension for the whole stage: O^T = V^T . P^T on v_mfma_f32_16x16x32_bf16 over two key tiles at once, each V^T
//     fragment two transposing LDS reads (ds_read_b64_tr_b16) of the row-major V rows.  So the accumulators are an
//     eighth or a quarter of the output a wavefront, nothing is merged at the end but the rows' sums, and a stage costs
//     one barrier.
//   * The exponent reference of a row is shared by the wavefronts and moves only when a score exceeds it by 2^8; a stage
//     in which one does is seen by all of them after its barrier and weighed again against the new references.
//   What bounds it: memory at long contexts (38000 positions, D = 256, 4 kv heads: 30.2 us, 5.2 TB/s of K and V), the
//   chain of dependent latencies at short ones (1000 positions: 7.7 us, of which the launch 1.7, sequence length ->
//   block ids -> K and V about 3.5).  Against the form before it (4 wavefronts in two halves of the head dimension, each
//   half computing every score, 32-position stages, a register state of the whole output merged through LDS), with its
//   combine launch, us a layer: 38000 positions 40.1 -> 35.0; 1000 12.0 -> 10.8; D = 128, 30000 positions, 64 packed
//   rows 55.0 -> 33.8; D = 64, four requests of 5000 18.3 -> 14.3.  Per-wavefront accumulators of the whole head
//   dimension without a barrier in the loop measured 37.1 and 12.9 on the first two: their merge alone took 2.4 us.
//   combine kernel, one 256-thread workgroup per (token, head, 64 d values): the row's split partials
//   are merged by log-sum-exp in thread groups, then the groups through LDS.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <mutex>
#include <unordered_set>

#include "qf_spec_attn.h"

namespace qfa {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef const void __attribute__((address_space(1)))* gptr_t;
typedef void __attribute__((address_space(3)))* lptr_t;

constexpr int kWave = 64;
constexpr int kThreads = 256;                      // combine kernel
constexpr int kKeyBlock = QF_SPEC_ATTN_KEY_BLOCK;  // splits are whole multiples of this many positions
constexpr int kMaxBalanced = kWave;                // requests of a balanced call: one lane of a wavefront each
constexpr size_t kMaxLds = 160 * 1024;             // gfx950 LDS per workgroup
static_assert(kMaxBalanced * sizeof(int2) <= QF_SPEC_ATTN_PLAN_BYTES, "a slot range a request");
constexpr int kMaxRows = QF_SPEC_ATTN_MAX_ROWS;
constexpr int kMaxChunk = 0x7fffffff / kKeyBlock * kKeyBlock;  // the longest split: any larger min_chunk means one split
constexpr int kNonTemporal = 2;  // cache-policy operand of a direct-to-LDS load: read once
constexpr float kLog2e = 1.4426950408889634f;
constexpr size_t kMaxDynLds = 160 * 1024 - 8 * 1024;  // gfx950 LDS per workgroup, less the static arrays
constexpr size_t kDefaultLds = 64 * 1024;

// Division of 0 <= n < 2^31 by an invariant d >= 1 (Granlund and Montgomery, PLDI 1994): with l = ceil(log2 d) and
// m = ceil(2^(31 + l) / d), which has 32 bits, floor(n / d) = (n * m) >> (31 + l).
struct Divisor {
  uint32_t m;
  int shift;  // of the upper half of the product; l = 0 (d = 1) is handled as m = 2^31, shift -1
};
inline Divisor divisor(int d) {
  int l = 0;
  while (((int64_t)1 << l) < d) ++l;
  return Divisor{(uint32_t)((((uint64_t)1 << (31 + l)) + d - 1) / d), l - 1};
}
__device__ __forceinline__ int divide(int n, Divisor d) {
  return (int)((((uint64_t)(uint32_t)n * d.m) >> 31) >> (d.shift + 1));
}

struct AttnArgs {
  const uint16_t* q;
  int64_t sq_t, sq_h;
  const uint16_t* kc;
  int64_t sk_b, sk_t, sk_h;
  const uint16_t* vc;
  int64_t sv_b, sv_t, sv_h;
  const int32_t* bt;
  int64_t sbt;
  const int32_t* seq_lens;
  uint16_t* out;
  int64_t so_t, so_h;
  float* o_part;    // [B][HKV][S][R][D]; balanced: [HKV][S][R][D], request b's splits at its slots
  float* lse_part;  // [B][HKV][S][R]; balanced: [HKV][S][R]
  int B, Q, H, HKV, G, R, page, splits, min_chunk;
  // Not null: balanced.  The splits of a kv head are shared out over the requests by length; the prefix kernel leaves
  // request b's first slot and slot count here for the combine kernel.
  int2* plan;
  Divisor by_g, by_splits, by_page;
  float qk_scale;  // softmax scale * log2(e): scores are kept in base 2
};

// Positions per prefix split (the reference's split arithmetic, spec_attn.py:38-40, with this
// kernel's key block): both kernels derive it from the sequence length alone.  Lengths are below
// kMaxChunk and run bounds min_chunk by it, so the rounding up stays in range.
__device__ __forceinline__ int split_chunk(int prefix, const AttnArgs& a) {
  int c = prefix > 0 ? divide(prefix - 1, a.by_splits) + 1 : 0;
  c = c > a.min_chunk ? c : a.min_chunk;
  return (c + kKeyBlock - 1) / kKeyBlock * kKeyBlock;
}

// Inclusive scan over the wavefront's 64 lanes by DPP adds (every lane active).
__device__ __forceinline__ int wave_scan(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr 1, 2, 4, 8: within 16 lanes
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast 15: row 0 into 1, row 2 into 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast 31: rows 0, 1 into 2, 3
  return v;
}

// The balanced split (every lane of the wavefront active; at most kMaxBalanced requests, splits >= requests): one
// chunk length for all requests, the shortest of a rising sequence of multiples of kKeyBlock whose splits fit the
// a.splits slots of a kv head (each candidate an eighth above the last), so the longest split of a ragged batch is
// near the batch's mean and not the longest request's share (six requests of 9000 to 2335 positions: 640 positions,
// 55 of 64 slots used, the mean 531).  A request without a prefix takes one split (its in-flight positions).  Slots
// go to the requests in order.  Lane i returns request i's length, splits (n) and first slot; `total` slots are used.
// In unsigned arithmetic and in units of kKeyBlock, so that min_chunk may be any int and the batch hold up to 2^36
// positions.
__device__ __forceinline__ void balance(const AttnArgs& a, int lane, int& seq, int& chunk, int& n, int& first, int& total) {
  seq = lane < a.B ? a.seq_lens[lane] : 0;
  const uint32_t prefix = (uint32_t)max(seq - a.Q, 0);
  const uint32_t units =
      (uint32_t)__builtin_amdgcn_readlane(wave_scan((int)((prefix + kKeyBlock - 1) / kKeyBlock)), kWave - 1);
  const uint32_t lo = max((units + a.splits - 1) / (uint32_t)a.splits, ((uint32_t)a.min_chunk + kKeyBlock - 1) / kKeyBlock);
  uint32_t len = lo * kKeyBlock;
  for (;;) {  // ends: once len covers the longest prefix, every request takes one split and a.B <= a.splits
    n = lane < a.B ? (prefix > 0 ? (int)((prefix - 1) / len) + 1 : 1) : 0;
    const int upto = wave_scan(n);
    first = upto - n;
    total = __builtin_amdgcn_readlane(upto, kWave - 1);
    if (total <= a.splits) break;
    len += (len / 8 + kKeyBlock - 1) / kKeyBlock * kKeyBlock;
  }
  chunk = (int)min(len, (uint32_t)kMaxChunk);
}

// s_waitcnt with vmcnt = n (0..63) and the other counters unconstrained.
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0F70);
}

// 32-bit LDS address of a pointer into the workgroup's LDS
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}

// Transposing LDS read (gfx950 ds_read_b64_tr_b16).  Within each group of 16 lanes, lane i receives
// word i % 4 of the 8 bytes addressed by lane 4 j + i / 4, for j = 0..3.  Issued as inline assembly
// because the compiler treats the builtin's read as depending on every direct-to-LDS copy still in
// flight and waits for all of them (vmcnt(0)) before it; here the copies a read depends on have
// been waited for explicitly before the stage barrier.  The result is valid only after
// wait_lds_all.
__device__ __forceinline__ u32x2_t ds_read_tr16_b64(uint32_t addr) {
  u32x2_t v;
  asm volatile("ds_read_b64_tr_b16 %0, %1" : "=v"(v) : "v"(addr));
  return v;
}

// A 16-byte LDS read issued the same way, for the K fragments.
__device__ __forceinline__ u32x4_t ds_read_b128(uint32_t addr) {
  u32x4_t v;
  asm volatile("ds_read_b128 %0, %1" : "=v"(v) : "v"(addr));
  return v;
}

__device__ __forceinline__ u32x2_t ds_read_b64(uint32_t addr) {
  u32x2_t v;
  asm volatile("ds_read_b64 %0, %1" : "=v"(v) : "v"(addr));
  return v;
}

// LDS writes issued the same way; done (for this wavefront) at the wait of stage_barrier.
__device__ __forceinline__ void ds_write_b64(uint32_t addr, u32x2_t v) {
  asm volatile("ds_write_b64 %0, %1" : : "v"(addr), "v"(v) : "memory");
}
__device__ __forceinline__ void ds_write_b32(uint32_t addr, uint32_t v) {
  asm volatile("ds_write_b32 %0, %1" : : "v"(addr), "v"(v) : "memory");
}

// Waits for every outstanding LDS access of the wavefront; the fragments read are tied to the wait, so no use of them
// is scheduled before it.
template <int N, typename V>
__device__ __forceinline__ void tie(V (&v)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" : "+v"(v[i]));
}
template <int N, typename V>
__device__ __forceinline__ void wait_lds_all(V (&v)[N]) {
  asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
  tie(v);
}
template <int N, int M, typename V>
__device__ __forceinline__ void wait_lds_all(V (&v)[N], V (&w)[M]) {
  asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
  tie(v);
  tie(w);
}

// Workgroup barrier after this wavefront's LDS accesses.  The direct-to-LDS copies it makes visible are those the
// wavefronts have waited for (wait_vmcnt); later ones stay in flight across it.
__device__ __forceinline__ void stage_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" : : : "memory");
}

// Two 4-value fragments as one of 8.
__device__ __forceinline__ bf16x8_t pair(u32x2_t a, u32x2_t b) {
  return __builtin_bit_cast(bf16x8_t, u32x4_t{a.x, a.y, b.x, b.y});
}

// A pointer that is the same in every lane, in scalar registers.
__device__ __forceinline__ const char* scalar_ptr(const char* p) {
  const uint64_t v = (uint64_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((int)(uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
  return (const char*)(((uint64_t)hi << 32) | lo);
}

__device__ __forceinline__ float wave_max_q(float v) {  // over the 4 lanes l, l^16, l^32, l^48
  v = fmaxf(v, __shfl_xor(v, 16));
  return fmaxf(v, __shfl_xor(v, 32));
}
__device__ __forceinline__ float wave_sum_q(float v) {
  v += __shfl_xor(v, 16);
  return v + __shfl_xor(v, 32);
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// bf16 <-> fp32 on 32-bit words (element order: low half first)
__device__ __forceinline__ float bf16_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
__device__ __forceinline__ f32x4_t bf16x4_to_f32(u32x2_t w) {
  return f32x4_t{bf16_lo(w.x), bf16_hi(w.x), bf16_lo(w.y), bf16_hi(w.y)};
}
// two fp32 -> two bf16 (round to nearest even), `a` in the low half
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t{a, b}), bf16x2_t));
}

// Geometry of the prefix kernel for head size D and RT row tiles.
template <int D, int RT>
struct Geo {
  // A stage is one 16-position key tile a wavefront.  4 wavefronts at D = 256, where two stages of 64 positions fill
  // 128 KiB of LDS, and at D = 128, where LDS then holds two workgroups a CU, for grids of more workgroups than CUs (8
  // wavefronts up to 48 rows, 105 to 25000 positions, 1 to 64 requests: 1.08 times the time up to 500 positions, 1.03 to
  // 2000, 1.00 above).  8 at D = 64: 4 have too few bytes in flight for long contexts (above 2000 positions up to 1.37
  // times the time, 1.10 by geometric mean), though they take 0.92 of it up to 500.
  static constexpr int kWaves = D == 64 ? 8 : 4;
  static constexpr int kThreads = kWaves * kWave;
  static constexpr int kTile = 16;                          // positions of a key tile
  static constexpr int kStage = kTile * kWaves;             // positions of a stage
  static constexpr int kRowBytes = 2 * D;                   // one cache row (bf16)
  static constexpr int kChunks = D / 8;                     // 16-byte pieces per row
  static constexpr int kTileBytes = kTile * kRowBytes;      // one tensor, one tile
  static constexpr int kCopies = kTileBytes / 1024;         // 1 KiB copies of a tile
  static constexpr int kRowsPerCopy = 1024 / kRowBytes;
  static constexpr int kDChunks = D / 32;                   // 32-d MFMA steps of a score
  // The output's 16-wide d tiles over the wavefronts: kOwn for each of kDGroups; wavefronts beyond those (D = 64) take
  // every other row tile.
  static constexpr int kDTiles = D / 16;
  static constexpr int kDGroups = kDTiles < kWaves ? kDTiles : kWaves;
  static constexpr int kOwn = kDTiles / kDGroups;
  static constexpr int kRowGroups = kWaves / kDGroups;
  static constexpr int kOwnRows = (RT + kRowGroups - 1) / kRowGroups;
  // LDS: K and V tiles [2][wavefront], then the softmax weights [2][wavefront][RT][64 lanes x 8 bytes].
  static constexpr int kWeights = 2 * kWaves * 2 * kTileBytes;
  static constexpr int kLds = kWeights + 2 * kWaves * RT * 512;
  static_assert(kLds + RT * kWaves * 128 + 256 <= (int)kMaxLds, "LDS budget");
  // Wavefronts a SIMD: of one workgroup, or of two where LDS holds two.
  static constexpr int kMinOnSimd = kWaves / 4;
  static constexpr int kMaxOnSimd = kWaves == 4 && 2 * (kLds + RT * kWaves * 64 + 64) <= (int)kMaxLds ? 2 : kWaves / 4;
  // The 16-byte piece of row n that lands at LDS position p is piece p ^ swz(n): 16 consecutive rows
  // read at one piece index then hit 16 distinct bank groups.
  __device__ static __forceinline__ int swz(int n) { return kChunks >= 16 ? (n & 15) : ((n >> 1) & 7); }
};

// ALIGNED: the page size is a multiple of 16, so a key tile lies in one page (splits start on multiples of 32) and a copy
// takes one scalar base.  Otherwise each lane finds its row's page among the two a tile can touch.  Both forms are free
// of branches, so that the compiler can count the vector-memory instructions outstanding.
template <int D, int RT, bool ALIGNED>
__global__ __launch_bounds__((Geo<D, RT>::kThreads))
__attribute__((amdgpu_waves_per_eu((Geo<D, RT>::kMinOnSimd), (Geo<D, RT>::kMaxOnSimd)))) void
spec_prefix_kernel(AttnArgs a) {
  using Gm = Geo<D, RT>;
  constexpr int kWaves = Gm::kWaves;
  constexpr int NK = Gm::kCopies;
  extern __shared__ __align__(16) uint8_t lds[];
  __shared__ float row_exchange[RT][kWaves][16];      // a value a row and wavefront: the maxima, at the end the sums
  __shared__ __align__(16) uint32_t moved[2][8];      // a wavefront found a score above the reference, stage parity

  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int hkv = blockIdx.y;
  int b = blockIdx.z, split = blockIdx.x, seq, chunk, n = 0, first = 0;
  if (a.plan != nullptr) {
    int total;
    balance(a, lane, seq, chunk, n, first, total);
    if ((int)blockIdx.x >= total) return;  // a slot of no request: the combine kernel reads the used ones only
    b = 63 - __builtin_clzll(__ballot(lane < a.B && first <= (int)blockIdx.x));
    split = blockIdx.x - __builtin_amdgcn_readlane(first, b);
    seq = __builtin_amdgcn_readlane(seq, b);
    chunk = __builtin_amdgcn_readfirstlane(chunk);
  }

  // Packed query rows: B fragments of the score product (rows >= R repeat row R - 1), requested first, so that they
  // arrive while the sequence length and the block ids do.
  const int l16 = lane & 15;
  const int qg = lane >> 4;
  bf16x8_t qf[RT][Gm::kDChunks];
  int q_index[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const int r = min(rt * 16 + l16, a.R - 1);
    q_index[rt] = divide(r, a.by_g);
    const int h = hkv * a.G + (r - q_index[rt] * a.G);
    const uint16_t* qrow = a.q + (int64_t)(b * a.Q + q_index[rt]) * a.sq_t + (int64_t)h * a.sq_h + qg * 8;
#pragma unroll
    for (int c = 0; c < Gm::kDChunks; ++c) qf[rt][c] = *reinterpret_cast<const bf16x8_t*>(qrow + c * 32);
  }

  if (a.plan == nullptr) seq = a.seq_lens[b];
  const int prefix = seq - a.Q > 0 ? seq - a.Q : 0;
  if (a.plan == nullptr) chunk = split_chunk(prefix, a);
  const int64_t part = (((int64_t)b * (a.plan != nullptr ? 0 : a.HKV) + hkv) * a.splits + blockIdx.x) * a.R;
  // Split s takes positions [s * chunk, min((s + 1) * chunk, prefix)); the last active split (split 0
  // when the prefix is empty) also takes this step's in-flight positions [prefix, seq).  Query qi sees
  // the positions up to seq - q_len + qi, which include the whole prefix, so one causal bound per
  // row covers both kinds of position.
  const int64_t first_pos = (int64_t)split * chunk;  // past 2^31 for the unused splits of a large min_chunk
  const bool active = split == 0 || first_pos < prefix;
  const int start = active ? (int)first_pos : 0;
  const int end = chunk >= prefix - start ? seq : start + chunk;
  if (a.plan != nullptr && blockIdx.x == 0 && blockIdx.y == 0 && wave == 0 && lane < a.B) a.plan[lane] = make_int2(first, n);
  if (!active || start >= end) {
    // no position here: the split's rows get log-sum-exp -inf, so the combine kernel can read every
    // split without knowing the sequence length (uniform: the whole workgroup leaves)
    for (int r = threadIdx.x; r < a.R; r += Gm::kThreads) a.lse_part[part + r] = -__builtin_inff();
    return;
  }
  int last[RT];  // last visible position of the lane's score row in each row tile
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) last[rt] = seq - a.Q + q_index[rt];

  // ---- this wavefront's key tiles: tile `wave` of every stage (past the end: the split's last tile again) ----
  const int n_tiles = (end - start + Gm::kTile - 1) / Gm::kTile;
  const int n_stages = (n_tiles + kWaves - 1) / kWaves;
  const int32_t* bt_row = a.bt + (int64_t)b * a.sbt;
  const char* kbytes = reinterpret_cast<const char*>(a.kc + (int64_t)hkv * a.sk_h);
  const char* vbytes = reinterpret_cast<const char*>(a.vc + (int64_t)hkv * a.sv_h);
  const int last_page = divide(end - 1, a.by_page);

  // Block ids of 64 of the wavefront's tiles, one a lane: the page of the tile's first row (and the page after it: a
  // tile of 16 rows touches at most two pages of 16 or more), and the first row's place in its page.
  int blk0, blk1 = 0, in_page;
  auto load_blocks = [&](int base) {
    const int pos = start + min(wave + (base + lane) * kWaves, n_tiles - 1) * Gm::kTile;
    const int pg = divide(pos, a.by_page);
    in_page = pos - pg * a.page;
    blk0 = bt_row[pg];
    if constexpr (!ALIGNED) blk1 = bt_row[min(pg + 1, last_page)];
  };
  load_blocks(0);
  wait_vmcnt<0>();  // the queries too: none may be outstanding when the copies are counted below

  // ---- copies: lane l of copy j moves the 16-byte piece p of row n = j * kRowsPerCopy + l / kChunks of the tile to
  // piece l % kChunks = p ^ swz(n) ----
  const int t_lane = lane / Gm::kChunks;
  auto piece = [&](int j) {
    return (uint32_t)(((lane % Gm::kChunks) ^ Gm::swz(j * Gm::kRowsPerCopy + t_lane)) * 16);
  };
  struct Where {
    int blk0, blk1, in_page;
  };
  auto where = [&](int stage) {
    const int i = stage & (kWave - 1);
    return Where{__builtin_amdgcn_readlane(blk0, i), ALIGNED ? 0 : __builtin_amdgcn_readlane(blk1, i),
                 __builtin_amdgcn_readlane(in_page, i)};
  };
  auto copy = [&](const char* bytes, int64_t sb, int64_t st, Where at, int stage, uint8_t* dst) {
    const char* base = bytes + (at.blk0 * sb + at.in_page * st) * 2;
#pragma unroll
    for (int j = 0; j < NK; ++j) {
      const char* p;
      if constexpr (ALIGNED) {  // a scalar base and a 32-bit lane offset; rows past the end are the page's own
        p = scalar_ptr(base + (int64_t)j * Gm::kRowsPerCopy * 2 * st) + ((uint32_t)(t_lane * (int)st * 2) + piece(j));
      } else {  // rows past the end re-read the tile's first row; rows past the page count back from the next one
        const char* base1 = bytes + (at.blk1 * sb + (at.in_page - a.page) * st) * 2;
        const int pos = start + min(wave + stage * kWaves, n_tiles - 1) * Gm::kTile;
        int row = j * Gm::kRowsPerCopy + t_lane;
        row = row < end - pos ? row : 0;
        p = (row < a.page - at.in_page ? base : base1) + row * st * 2 + piece(j);
      }
      __builtin_amdgcn_global_load_lds((gptr_t)p, (lptr_t)(dst + j * 1024), 16, 0, kNonTemporal);
    }
  };
  // slot (stage & 1) of a tensor: [2][kWaves] tiles of K, then of V
  auto k_slot = [&](int stage, int w) { return lds + ((stage & 1) * kWaves + w) * Gm::kTileBytes; };
  auto v_slot = [&](int stage, int w) { return lds + ((2 + (stage & 1)) * kWaves + w) * Gm::kTileBytes; };
  auto copy_k = [&](Where at, int stage) { copy(kbytes, a.sk_b, a.sk_t, at, stage, k_slot(stage, wave)); };
  auto copy_v = [&](Where at, int stage) { copy(vbytes, a.sv_b, a.sv_t, at, stage, v_slot(stage, wave)); };

  if (wave < n_tiles) {  // a split of less than a stage: the other wavefronts have no tile (and no later copy to count)
    copy_k(where(0), 0);
    copy_v(where(0), 0);
  }
  Where next = where(1);  // the next stage's tile (its V is requested a stage after its K)
  if (n_stages > 1) copy_k(next, 1);

  // byte offsets of this lane's LDS reads in a tile: the K fragment of d step c at k_off ^ 64 c, the transposing V
  // read of d tile dt at v_off ^ 32 dt (the swizzle's bits and the step's do not overlap)
  const uint32_t k_off = (uint32_t)(l16 * Gm::kRowBytes + ((qg ^ Gm::swz(l16)) << 4));
  uint32_t v_off;
  {
    const int n = 4 * (lane >> 4) + ((lane >> 2) & 3);
    const int d = 4 * (lane & 3);
    v_off = (uint32_t)(n * Gm::kRowBytes + (((d >> 3) ^ Gm::swz(n)) << 4) + (d & 7) * 2);
  }
  // the output tiles of this wavefront: d tiles dg * kOwn .. + kOwn - 1 of the row tiles rg, rg + kRowGroups, ...
  const int dg = wave % Gm::kDGroups;
  const int rg = wave / Gm::kDGroups;
  v_off ^= 32 * (dg * Gm::kOwn);

  // Online softmax state.  m_ref is the row's exponent reference, the same in every wavefront, moved only when a
  // score exceeds it by more than kRescale (log2 units), so the weights stay below 2^kRescale and the accumulators are
  // rarely rescaled; the result equals the running-maximum form up to rounding.  l_run sums this wavefront's weights
  // (its key tiles, its lanes' positions).
  constexpr float kRescale = 8.f;
  float m_ref[RT], l_run[RT];
  f32x4_t o_acc[Gm::kOwnRows][Gm::kOwn];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    m_ref[rt] = -__builtin_inff();
    l_run[rt] = 0.f;
  }
#pragma unroll
  for (int q = 0; q < Gm::kOwnRows; ++q)
#pragma unroll
    for (int u = 0; u < Gm::kOwn; ++u) o_acc[q][u] = f32x4_t{0.f, 0.f, 0.f, 0.f};

#pragma unroll 1
  for (int st = 0; st < n_stages; ++st) {
    // The copies are requested in the order K0 V0 K1 | K2 V1 | K3 V2 | ...  K of stage 0 has landed once V0 and K1
    // alone are outstanding, K of stage 1 with K2 and V1; a later stage's did before the last barrier (it is ahead of
    // that stage's V, which every wavefront waited for).
    if (st < 2) {
      if (n_stages > 1 + st) {
        wait_vmcnt<2 * NK>();
      } else {
        wait_vmcnt<NK>();
      }
    }

    Where after_next;

    // S^T of the wavefront's key tile: positions 4 qg + i, row 16 rt + l16
    f32x4_t sc[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) sc[rt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    {
      const uint32_t ks = lds_addr(k_slot(st, wave));
      u32x4_t kf[Gm::kDChunks];
#pragma unroll
      for (int c = 0; c < Gm::kDChunks; ++c) kf[c] = ds_read_b128(ks + (k_off ^ (64 * c)));
      wait_lds_all<Gm::kDChunks>(kf);
      after_next = next;
      if (st + 2 < n_stages) {  // the K reads have returned: their slot is free
        if (((st + 2) & (kWave - 1)) == 0) {
          load_blocks(st + 2);
          wait_vmcnt<0>();  // here, once in 64 stages, and not at every use of the block ids
        }
        after_next = where(st + 2);
        copy_k(after_next, st + 2);
      }
#pragma unroll
      for (int c = 0; c < Gm::kDChunks; ++c)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
          sc[rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, kf[c]), qf[rt][c], sc[rt], 0, 0, 0);
    }

    // scores in base 2; a tile wholly inside every row's visible range needs no mask
    const int pos = start + (wave + st * kWaves) * Gm::kTile;
    const int pos0 = pos + qg * 4;
    float mx[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) sc[rt] *= a.qk_scale;
    if (pos + Gm::kTile > end || pos + Gm::kTile - 1 > seq - a.Q) {
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int i = 0; i < 4; ++i) sc[rt][i] = pos0 + i < end && pos0 + i <= last[rt] ? sc[rt][i] : -__builtin_inff();
    }
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) mx[rt] = fmaxf(fmaxf(sc[rt][0], sc[rt][1]), fmaxf(sc[rt][2], sc[rt][3]));

    // The weights against the present references, rounded to bf16, to the other wavefronts through LDS: lane (qg, l16)
    // holds those of 4 positions of one row, its part of the B fragment of O^T = V^T P^T.
    float sum[RT];
    const uint32_t w_slot = lds_addr(lds) + Gm::kWeights + (uint32_t)((st & 1) * kWaves * RT * 512) + lane * 8;
    auto weigh = [&]() {
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        const float m_base = m_ref[rt] == -__builtin_inff() ? 0.f : m_ref[rt];  // -inf: a row that has seen nothing yet
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = fast_exp2(sc[rt][i] - m_base);
        sum[rt] = (v[0] + v[1]) + (v[2] + v[3]);
        ds_write_b64(w_slot + (wave * RT + rt) * 512, u32x2_t{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])});
      }
    };
    bool move = st == 0;
    if (!move) {
      bool above = false;
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) above |= mx[rt] > m_ref[rt] + kRescale;
      weigh();
      ds_write_b32(lds_addr(&moved[st & 1][wave]), __any(above) ? 1u : 0u);  // every lane the same word
    }
    // V of this stage has landed once only the K copies requested after it are outstanding
    if (st + 2 >= n_stages) {
      if (st == 0 && n_stages > 1) {
        wait_vmcnt<NK>();
      } else {
        wait_vmcnt<0>();
      }
    } else if (st == 0) {
      wait_vmcnt<2 * NK>();
    } else {
      wait_vmcnt<NK>();
    }
    if (!move) {
      stage_barrier();
      u32x4_t f[kWaves / 4];
#pragma unroll
      for (int i = 0; i < kWaves / 4; ++i) f[i] = ds_read_b128(lds_addr(&moved[st & 1][4 * i]));
      wait_lds_all<kWaves / 4>(f);
      uint32_t any = 0;
#pragma unroll
      for (int i = 0; i < kWaves / 4; ++i) any |= (f[i].x | f[i].y) | (f[i].z | f[i].w);
      move = __builtin_amdgcn_readfirstlane(any) != 0;
    }
    if (move) {  // the same in every wavefront: the rows' new references, and the weights again
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        mx[rt] = wave_max_q(mx[rt]);
        ds_write_b32(lds_addr(&row_exchange[rt][wave][l16]), __float_as_uint(mx[rt]));  // four lanes the same word
      }
      stage_barrier();
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        float m_new = m_ref[rt];
#pragma unroll
        for (int w = 0; w < kWaves; ++w) m_new = fmaxf(m_new, row_exchange[rt][w][l16]);
        const float alpha = fast_exp2(m_ref[rt] - (m_new == -__builtin_inff() ? 0.f : m_new));
        m_ref[rt] = m_new;
        l_run[rt] *= alpha;
        if (st > 0 && rt % Gm::kRowGroups == rg) {
#pragma unroll
          for (int u = 0; u < Gm::kOwn; ++u) o_acc[rt / Gm::kRowGroups][u] *= alpha;
        }
      }
      weigh();
      stage_barrier();
    }
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) l_run[rt] += sum[rt];
    // every wavefront is past the previous stage's V
    if (st + 1 < n_stages) copy_v(next, st + 1);
    next = after_next;

    // O^T += V^T P^T over the stage, two key tiles an instruction: k slot (qg, j) is position 4 qg + j of the first
    // tile for j < 4 and 4 qg + j - 4 of the second for j >= 4.  The V^T fragment of a d tile comes from one
    // transposing LDS read a key tile: lane 16 g + 4 j + q points at the 8 bytes of row 4 g + j holding d values
    // d0 + 4 q .. d0 + 4 q + 3, and the read hands lane 16 g + i the values V[4 g + j][d0 + i], j = 0..3.
    u32x2_t vf[Gm::kOwn * kWaves], pf[Gm::kOwnRows * kWaves];
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const uint32_t vs = lds_addr(v_slot(st, w));
#pragma unroll
      for (int u = 0; u < Gm::kOwn; ++u) vf[w * Gm::kOwn + u] = ds_read_tr16_b64(vs + (v_off ^ (32 * u)));
#pragma unroll
      for (int q = 0; q < Gm::kOwnRows; ++q)
        pf[w * Gm::kOwnRows + q] = ds_read_b64(w_slot + (w * RT + min(q * Gm::kRowGroups + rg, RT - 1)) * 512);
    }
    wait_lds_all(vf, pf);
    if (st + 1 == n_stages && start + n_stages * Gm::kStage > end) {
      // Rows past the end hold whatever the page, or the slot, does (perhaps NaN): their weight is 0, their V made 0.
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        const int p0 = start + (w + st * kWaves) * Gm::kTile + qg * 4;
        const uint32_t w0 = (p0 < end ? 0xffffu : 0u) | (p0 + 1 < end ? 0xffff0000u : 0u);
        const uint32_t w1 = (p0 + 2 < end ? 0xffffu : 0u) | (p0 + 3 < end ? 0xffff0000u : 0u);
#pragma unroll
        for (int u = 0; u < Gm::kOwn; ++u) vf[w * Gm::kOwn + u] &= u32x2_t{w0, w1};
      }
    }
#pragma unroll
    for (int w = 0; w < kWaves; w += 2)
#pragma unroll
      for (int u = 0; u < Gm::kOwn; ++u)
#pragma unroll
        for (int q = 0; q < Gm::kOwnRows; ++q)
          o_acc[q][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              pair(vf[w * Gm::kOwn + u], vf[(w + 1) * Gm::kOwn + u]),
              pair(pf[w * Gm::kOwnRows + q], pf[(w + 1) * Gm::kOwnRows + q]), o_acc[q][u], 0, 0, 0);
  }

  // ---- the rows' sums over the wavefronts, then the partial output (normalised) and base-2 log-sum-exp of each packed
  // row; a row that saw no position (possible only in the split holding the in-flight positions) is written as 0 with
  // log-sum-exp -inf ----
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) l_run[rt] = wave_sum_q(l_run[rt]);
  stage_barrier();  // the last maxima have been read
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) ds_write_b32(lds_addr(&row_exchange[rt][wave][l16]), __float_as_uint(l_run[rt]));
  stage_barrier();
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const int r = rt * 16 + l16;
    if (rt % Gm::kRowGroups != rg || r >= a.R) continue;
    float lt = 0.f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) lt += row_exchange[rt][w][l16];
    const float inv = lt > 0.f ? 1.f / lt : 0.f;
    float* orow = a.o_part + (part + r) * D + dg * Gm::kOwn * 16 + qg * 4;
#pragma unroll
    for (int u = 0; u < Gm::kOwn; ++u) *reinterpret_cast<f32x4_t*>(orow + u * 16) = o_acc[rt / Gm::kRowGroups][u] * inv;
    if (dg == 0 && qg == 0) a.lse_part[part + r] = lt > 0.f ? m_ref[rt] + __log2f(lt) : -__builtin_inff();
  }
}

// One workgroup per (token, head, 64-wide slice of d): the row's split partials merged by log-sum-exp (the merge of
// the reference's _suffix_combine_kernel, spec_attn.py:119-131).  Every split has written its rows' log-sum-exp (-inf
// where it saw nothing), so all loads issue at once, with no dependence on the sequence length (balanced calls read
// the request's place among the slots first); 16 groups of 16 threads merge every 16th split, then LDS merges the
// groups.
constexpr int kCombSlice = 64;  // d values per combine workgroup

template <int D>
__global__ __launch_bounds__(kThreads) void spec_combine_kernel(AttnArgs a) {
  constexpr int NQ = kCombSlice / 4;  // threads per group, 4 d values each
  constexpr int NGRP = kThreads / NQ;
  constexpr int kBatch = 4;           // parts a thread loads before merging them
  __shared__ float sm_m[NGRP], sm_l[NGRP];
  __shared__ __align__(16) float sm_acc[NGRP][kCombSlice];

  const int row = blockIdx.x;
  const int d0 = blockIdx.y * kCombSlice;
  const int tok = row / a.H;
  const int h = row - tok * a.H;
  const int b = __builtin_amdgcn_readfirstlane(tok / a.Q);
  const int qi = tok - b * a.Q;
  const int hkv = h / a.G;
  const int r = qi * a.G + (h - hkv * a.G);
  const int grp = threadIdx.x / NQ;
  const int dq = threadIdx.x - grp * NQ;

  float m = -__builtin_inff(), l = 0.f;
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  int parts = a.splits;
  int64_t part0 = ((int64_t)(b * a.HKV + hkv) * a.splits) * a.R + r;
  if (a.plan != nullptr) {
    const int2 place = a.plan[b];
    parts = place.y;
    part0 = ((int64_t)hkv * a.splits + place.x) * a.R + r;
  }
  // group grp merges the parts grp, grp + NGRP, ...
  for (int base = grp; base < parts; base += NGRP * kBatch) {
    float e[kBatch];
    f32x4_t o[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const int i = base + u * NGRP;
      e[u] = -__builtin_inff();
      if (i < parts) {
        const int64_t idx = part0 + (int64_t)i * a.R;
        e[u] = a.lse_part[idx];
        o[u] = *reinterpret_cast<const f32x4_t*>(a.o_part + idx * D + d0 + dq * 4);
      }
    }
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      if (e[u] == -__builtin_inff()) continue;  // a split with no position, or a row that saw none
      const float mn = fmaxf(m, e[u]);
      const float c_old = fast_exp2(m - mn);
      const float w = fast_exp2(e[u] - mn);
      acc = acc * c_old + o[u] * w;
      l = l * c_old + w;
      m = mn;
    }
  }

  if (dq == 0) {
    sm_m[grp] = m;
    sm_l[grp] = l;
  }
  *reinterpret_cast<f32x4_t*>(&sm_acc[grp][dq * 4]) = acc;
  __syncthreads();
  if (grp != 0) return;
  float mt = -__builtin_inff();
#pragma unroll
  for (int g = 0; g < NGRP; ++g) mt = fmaxf(mt, sm_m[g]);
  f32x4_t at = {0.f, 0.f, 0.f, 0.f};
  float lt = 0.f;
  if (mt != -__builtin_inff()) {
#pragma unroll
    for (int g = 0; g < NGRP; ++g) {
      const float w = fast_exp2(sm_m[g] - mt);  // 0 for an empty group
      at += *reinterpret_cast<const f32x4_t*>(&sm_acc[g][dq * 4]) * w;
      lt += sm_l[g] * w;
    }
  }
  const float inv = lt > 0.f ? 1.f / lt : 0.f;  // a row that sees no position is written as zeros
  *reinterpret_cast<u32x2_t*>(a.out + (int64_t)tok * a.so_t + (int64_t)h * a.so_h + d0 + dq * 4) =
      u32x2_t{pack_bf16(at[0] * inv, at[1] * inv), pack_bf16(at[2] * inv, at[3] * inv)};
}

typedef void (*KernelFn)(AttnArgs);

struct Prefix {
  KernelFn fn;
  int threads;
  size_t lds;
};

template <int D, int RT>
Prefix prefix_of(bool aligned) {
  using Gm = Geo<D, RT>;
  return Prefix{aligned ? &spec_prefix_kernel<D, RT, true> : &spec_prefix_kernel<D, RT, false>, Gm::kThreads,
                (size_t)Gm::kLds};
}

template <int D>
Prefix prefix_for(int rt, bool aligned) {
  switch (rt) {
    case 1: return prefix_of<D, 1>(aligned);
    case 2: return prefix_of<D, 2>(aligned);
    case 3: return prefix_of<D, 3>(aligned);
    case 4: return prefix_of<D, 4>(aligned);
    default: return Prefix{nullptr, 0, 0};
  }
}

std::mutex g_lds_mutex;
std::unordered_set<const void*> g_lds_raised;

int launch(KernelFn fn, dim3 grid, int threads, size_t smem, hipStream_t stream, const AttnArgs& a) {
  void* args[] = {const_cast<AttnArgs*>(&a)};
  if (smem > kDefaultLds) {
    std::lock_guard<std::mutex> lock(g_lds_mutex);
    const void* key = reinterpret_cast<const void*>(fn);
    if (g_lds_raised.find(key) == g_lds_raised.end()) {
      if (hipFuncSetAttribute(key, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMaxDynLds) != hipSuccess)
        return QF_ERR_HIP;
      g_lds_raised.insert(key);
    }
  }
  if (hipLaunchKernel(reinterpret_cast<const void*>(fn), grid, dim3(threads), args, smem, stream) != hipSuccess)
    return QF_ERR_HIP;
  return QF_OK;
}

inline bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

size_t workspace_for(int B, int Q, int H, int HKV, int D, int S) {
  if (B < 1 || Q < 1 || H < 1 || HKV < 1 || H % HKV || D < 1 || S < 1) return 0;
  const size_t R = (size_t)Q * (H / HKV);
  const size_t n = (size_t)B * HKV * S * R * (D + 1) * sizeof(float);
  return (n + 255) / 256 * 256;
}

int run(const uint16_t* query, int64_t q_stride_tok, int64_t q_stride_head, const uint16_t* key_cache,
        int64_t k_stride_block, int64_t k_stride_tok, int64_t k_stride_head, const uint16_t* value_cache,
        int64_t v_stride_block, int64_t v_stride_tok, int64_t v_stride_head, const int32_t* block_table,
        int64_t bt_stride, const int32_t* seq_lens, uint16_t* out, int64_t o_stride_tok, int64_t o_stride_head,
        int num_reqs, int q_len, int num_heads, int num_kv_heads, int head_size, int page_size, float scale,
        int num_splits, int min_chunk, int balanced, void* workspace, size_t workspace_bytes, void* stream) {
  if (!query || !key_cache || !value_cache || !block_table || !seq_lens || !out) return QF_ERR_INVALID_ARG;
  if (num_reqs < 1 || q_len < 1 || num_heads < 1 || num_kv_heads < 1 || page_size < 1 || num_splits < 1 ||
      num_splits > 65535 || min_chunk < 1 || bt_stride < 0)
    return QF_ERR_INVALID_ARG;
  if (!(scale == scale)) return QF_ERR_INVALID_ARG;
  if (num_heads % num_kv_heads) return QF_ERR_UNSUPPORTED;
  const int G = num_heads / num_kv_heads;
  const int R = q_len * G;
  if (R > kMaxRows || page_size < QF_SPEC_ATTN_MIN_PAGE) return QF_ERR_UNSUPPORTED;
  if (head_size != 64 && head_size != 128 && head_size != 256) return QF_ERR_UNSUPPORTED;
  if ((int64_t)num_reqs * num_kv_heads > 65535 || (int64_t)num_reqs * q_len * num_heads > 0x7fffffff)
    return QF_ERR_UNSUPPORTED;
  const int64_t strides[] = {q_stride_tok, q_stride_head, k_stride_block, k_stride_tok, k_stride_head,
                             v_stride_block, v_stride_tok, v_stride_head, o_stride_tok, o_stride_head};
  for (int64_t s : strides)
    if (s < 0 || s % 8) return QF_ERR_UNSUPPORTED;
  // the prefix kernel keeps per-lane byte offsets of up to one stage of rows in 32 bits
  if ((k_stride_tok > v_stride_tok ? k_stride_tok : v_stride_tok) * 2 * kKeyBlock >= ((int64_t)1 << 31))
    return QF_ERR_UNSUPPORTED;
  if (!aligned16(query) || !aligned16(key_cache) || !aligned16(value_cache) || !aligned16(out))
    return QF_ERR_UNSUPPORTED;
  if (balanced && (num_reqs > kMaxBalanced || num_splits < num_reqs)) return QF_ERR_UNSUPPORTED;
  // split slots per kv head: one set a request, or one set shared by all
  const int sets = balanced ? 1 : num_reqs;
  const size_t part_bytes = workspace_for(sets, q_len, num_heads, num_kv_heads, head_size, num_splits);
  const size_t need = part_bytes + (balanced ? QF_SPEC_ATTN_PLAN_BYTES : 0);
  if (workspace == nullptr || workspace_bytes < need || !aligned16(workspace)) return QF_ERR_WORKSPACE;

  AttnArgs a;
  a.q = query;
  a.sq_t = q_stride_tok;
  a.sq_h = q_stride_head;
  a.kc = key_cache;
  a.sk_b = k_stride_block;
  a.sk_t = k_stride_tok;
  a.sk_h = k_stride_head;
  a.vc = value_cache;
  a.sv_b = v_stride_block;
  a.sv_t = v_stride_tok;
  a.sv_h = v_stride_head;
  a.bt = block_table;
  a.sbt = bt_stride;
  a.seq_lens = seq_lens;
  a.out = out;
  a.so_t = o_stride_tok;
  a.so_h = o_stride_head;
  const size_t n_o = (size_t)sets * num_kv_heads * num_splits * R * head_size;
  a.o_part = static_cast<float*>(workspace);
  a.lse_part = a.o_part + n_o;
  a.B = num_reqs;
  a.Q = q_len;
  a.H = num_heads;
  a.HKV = num_kv_heads;
  a.G = G;
  a.R = R;
  a.page = page_size;
  a.splits = num_splits;
  a.min_chunk = min_chunk < kMaxChunk ? min_chunk : kMaxChunk;
  a.qk_scale = scale * kLog2e;
  a.by_g = divisor(G);
  a.by_splits = divisor(num_splits);
  a.by_page = divisor(page_size);
  a.plan = balanced ? reinterpret_cast<int2*>(static_cast<uint8_t*>(workspace) + part_bytes) : nullptr;

  hipStream_t s = static_cast<hipStream_t>(stream);
  const int rt = (R + 15) / 16;
  Prefix pre;
  KernelFn comb;
  switch (head_size) {
    case 64: pre = prefix_for<64>(rt, page_size % 16 == 0); comb = &spec_combine_kernel<64>; break;
    case 128: pre = prefix_for<128>(rt, page_size % 16 == 0); comb = &spec_combine_kernel<128>; break;
    default: pre = prefix_for<256>(rt, page_size % 16 == 0); comb = &spec_combine_kernel<256>; break;
  }
  if (pre.fn == nullptr) return QF_ERR_UNSUPPORTED;
  int st = launch(pre.fn, dim3(num_splits, num_kv_heads, sets), pre.threads, pre.lds, s, a);
  if (st != QF_OK) return st;
  return launch(comb, dim3(num_reqs * q_len * num_heads, head_size / kCombSlice), kThreads, 0, s, a);
}

}  // namespace qfa

using namespace qfa;

extern "C" {

int qf_spec_attn_abi_version(void) { return QF_SPEC_ATTN_ABI_VERSION; }

size_t qf_spec_attn_workspace_bytes(int num_reqs, int q_len, int num_heads, int num_kv_heads, int head_size,
                                    int num_splits) {
  return workspace_for(num_reqs, q_len, num_heads, num_kv_heads, head_size, num_splits);
}

int qf_spec_attention(const uint16_t* query, int64_t q_stride_tok, int64_t q_stride_head,
                      const uint16_t* key_cache, int64_t k_stride_block, int64_t k_stride_tok,
                      int64_t k_stride_head,
                      const uint16_t* value_cache, int64_t v_stride_block, int64_t v_stride_tok,
                      int64_t v_stride_head,
                      const int32_t* block_table, int64_t bt_stride,
                      const int32_t* seq_lens,
                      uint16_t* out, int64_t o_stride_tok, int64_t o_stride_head,
                      int num_reqs, int q_len, int num_heads, int num_kv_heads, int head_size,
                      int page_size, float scale, int num_splits, int min_chunk,
                      void* workspace, size_t workspace_bytes, void* stream) {
  return run(query, q_stride_tok, q_stride_head, key_cache, k_stride_block, k_stride_tok, k_stride_head, value_cache,
             v_stride_block, v_stride_tok, v_stride_head, block_table, bt_stride, seq_lens, out, o_stride_tok,
             o_stride_head, num_reqs, q_len, num_heads, num_kv_heads, head_size, page_size, scale, num_splits,
             min_chunk, 0, workspace, workspace_bytes, stream);
}

int qf_spec_attention_balanced(const uint16_t* query, int64_t q_stride_tok, int64_t q_stride_head,
                               const uint16_t* key_cache, int64_t k_stride_block, int64_t k_stride_tok,
                               int64_t k_stride_head,
                               const uint16_t* value_cache, int64_t v_stride_block, int64_t v_stride_tok,
                               int64_t v_stride_head,
                               const int32_t* block_table, int64_t bt_stride,
                               const int32_t* seq_lens,
                               uint16_t* out, int64_t o_stride_tok, int64_t o_stride_head,
                               int num_reqs, int q_len, int num_heads, int num_kv_heads, int head_size,
                               int page_size, float scale, int total_splits, int min_chunk,
                               void* workspace, size_t workspace_bytes, void* stream) {
  return run(query, q_stride_tok, q_stride_head, key_cache, k_stride_block, k_stride_tok, k_stride_head, value_cache,
             v_stride_block, v_stride_tok, v_stride_head, block_table, bt_stride, seq_lens, out, o_stride_tok,
             o_stride_head, num_reqs, q_len, num_heads, num_kv_heads, head_size, page_size, scale, total_splits,
             min_chunk, 1, workspace, workspace_bytes, stream);
}

}  // extern "C"
