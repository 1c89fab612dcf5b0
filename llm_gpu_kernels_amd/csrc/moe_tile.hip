// LDS-tiled grouped GEMMs of the MoE forward on gfx950 for large row counts.
//
// When experts receive many rows (prefill chunks, skewed routing), streaming
// each weight byte once per 16/32-row task would re-read the hot experts'
// weights dozens of times.  Here a work unit is (expert, block of up to 160 of
// its grouped rows, tile of 256 weight rows).  An expert's rows are cut into
// the fewest such blocks, of equal height (a multiple of 32), taken from
// counts[] and offsets[]: the planner's 64-row task list is not used, only its
// length (zero when the plan stalled).  Units are numbered expert-major and
// weight-tile-major within an expert, and that sequence is cut into one
// contiguous chunk per XCD, so the row blocks that share a weight tile, and
// the weight tiles that share a block's token rows, meet in one XCD's L2.
//
// Per unit: a K loop over 64-wide stages.  Each stage's weight tile [256][64]
// and token tile [32 nb][64] go global -> LDS with buffer loads that write LDS
// directly (16-byte chunks XOR-swizzled by row on the global side, so that the
// MFMA operand reads are bank-conflict free).  The descriptors are bounded at
// the expert's matrix: weight rows past I or H, and the chunks of the last
// stage past K, read as zero, so any H and I that are multiples of 32 run
// here.  (W4G128 gate/up: load_role_w4 below; the down weights are bf16 in both
// formats.)
//
// Epilogues match the streaming kernels: gate/up round to bf16, SwiGLU in
// fp32, bf16 act rows; down rounds to bf16 and scatters rows to route order.
#include <type_traits>

#include "common.h"
#include "moe_internal.h"

#define MOE_CONST __attribute__((address_space(4)))
#define MOE_LDS __attribute__((address_space(3)))

namespace moe {

namespace {

template <typename T>
__device__ __forceinline__ const MOE_CONST T *as_const(const T *p) {
  return (const MOE_CONST T *)p;
}

__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

__device__ __forceinline__ f32x16 mfma32(u32x4 a, u32x4 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(a), as_bf16x8(b), c, 0, 0, 0);
}

// ---- shape of the kernel -------------------------------------------------------
// One 512-thread workgroup per CU: four MFMA waves, one per SIMD, and four
// loader waves, so each may use 256 VGPRs.  MFMA wave w owns 64 weight rows
// (gate/up: 32 gate and the 32 up rows of the same features) against all of
// the block's token rows: 2 x nb tiles of 32 x 32, at most 160 accumulator
// registers.  Per 16-K step it reads 2 + nb operand fragments for 2 nb MFMAs
// and reads each step's fragments before the MFMAs of the step before, across
// stage boundaries too.  The loader waves issue every global load and carry
// every vector-memory wait; one workgroup barrier per stage publishes that
// stage (the loaders waited for it) and frees the oldest slot of the ring.
//
// Measured at E = 128, H = 2048, I = 768, K = 8 against 64-row tasks with 64 x
// 32 wave tiles and every fragment of a stage read before its MFMAs: T = 4096
// gate/up 350 -> 237 us, down 215 -> 146 us; T = 1024 Zipf 153 -> 137 and 92 ->
// 80 us (with a SwiGLU of hardware exponentials; swiglu below: + 15 us at T =
// 4096).  At T = 4096 the loads alone take 188 us (2.5 GB through L2, 966 MB of
// HBM reads, 5.1 TB/s), the MFMAs and LDS reads alone 111 us, the epilogues 27.
constexpr int kBN = 256;                // weight rows per tile
constexpr int kBK = 64;                 // K per stage: one 128-byte piece per row
constexpr int kMaxNB = 5;               // 32-row token blocks per unit
constexpr int kABytes = kBN * kBK * 2;
constexpr int kRingBytes = (int)kMaxLds;
// Ring slots for units of up to NBM token blocks: three of 52 KiB, or four of
// 40 KiB (three stages in flight) where no unit is higher than 64 rows.
constexpr int slot_bytes(int NBM) { return kABytes + NBM * 32 * kBK * 2; }
constexpr int ring_slots(int NBM) { return kRingBytes / slot_bytes(NBM); }
constexpr int kMfmaWaves = 4;
constexpr int kLoaders = 4;
constexpr int kThreads = (kMfmaWaves + kLoaders) * kWave;
constexpr int kAPer = kBN / kLoaders / 8;  // weight loads per loader wave and stage
// Where stage buffers sit in the LDS.  bf16: each slot holds a weight tile and a
// token tile.  W4: two weight tiles (written by the loaders during the stage
// before they are read) and, in what is left, as many token tiles as fit up
// to eight, so that their loads are three stages ahead or more.
template <int NBM, bool W4>
struct Ring {
  static constexpr int kBBytes = NBM * 32 * kBK * 2;
  static constexpr int kASlots = W4 ? 2 : ring_slots(NBM);
  static constexpr int kBFit = (kRingBytes - 2 * kABytes) / kBBytes;
  static constexpr int kBSlots = W4 ? (kBFit < 8 ? kBFit : 8) : ring_slots(NBM);
  static constexpr int kAStride = W4 ? kABytes : slot_bytes(NBM);
  static constexpr int kB0 = W4 ? 2 * kABytes : kABytes;
  static constexpr int kBStride = W4 ? kBBytes : slot_bytes(NBM);
  static constexpr int kBytes = W4 ? kB0 + kBSlots * kBBytes : kASlots * kAStride;
};
static_assert(ring_slots(2) == 4 && ring_slots(kMaxNB) == 3, "the loaders' wait counts cover three and four slots");

// s_waitcnt with only the vector-memory counter bounded (gfx9 encoding).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}
// At most n vector-memory operations outstanding (n wave-uniform: the loads of
// one or two stages, or 0).
__device__ __forceinline__ void wait_vmcnt_upto(int n) {
  switch (n) {
#define MOE_W(N) case N: wait_vmcnt<N>(); break;
    MOE_W(9) MOE_W(10) MOE_W(11) MOE_W(12) MOE_W(13)   // one stage
    MOE_W(18) MOE_W(19) MOE_W(20)                       // two stages of one or two token blocks
#undef MOE_W
    default: wait_vmcnt<0>(); break;
  }
}

// 16 bytes per lane from a buffer straight into LDS (lane l's bytes at
// dst + 16 l); lanes whose voff is past the descriptor's size write zeros
// (soff is not part of that check).  Device pass only, as in the attention.
__device__ __forceinline__ void buffer_load_lds16(__amdgpu_buffer_rsrc_t rs, uint8_t *dst, uint32_t voff,
                                                  uint32_t soff) {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (MOE_LDS void *)dst, 16, voff, soff, 0, 0);
#endif
}

// Ends a group of loads.  A counted wait is right only while the groups are
// issued in program order; loads with an LDS destination and loads into
// registers do not alias, so without this the scheduler may swap them.
__device__ __forceinline__ void order_loads() { asm volatile("" ::: "memory"); }

__device__ __forceinline__ int sgpr(int v) { return __builtin_amdgcn_readfirstlane(v); }

// The unit sequence, held by every wave: lane l has the row counts and first
// grouped rows of experts 4 l .. 4 l + 3 and the number of units before them.
struct UnitMap {
  int cnt[4], off[4];
  int before;
  int total;
  int ntiles;
  uint32_t max_rows;  // rows per unit at most (a multiple of 32)

  __device__ __forceinline__ int blocks(int n) const { return (int)(((uint32_t)n + max_rows - 1) / max_rows); }

  __device__ __forceinline__ void init(const int32_t *counts, const int32_t *offsets, int E, int nt, int rows,
                                       int lane) {
    ntiles = nt;
    max_rows = (uint32_t)rows;
    int mine = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int e = min(4 * lane + j, E - 1);
      cnt[j] = counts[e];
      off[j] = offsets[e];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      cnt[j] = 4 * lane + j < E ? cnt[j] : 0;
      mine += blocks(cnt[j]) * nt;
    }
    int incl = mine;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const int up = __shfl_up(incl, o, kWave);
      if (lane >= o) incl += up;
    }
    before = incl - mine;
    total = __builtin_amdgcn_readlane(incl, kWave - 1);
  }

  struct Unit {
    int e, row0, rows, nt;  // expert, first grouped row, rows, weight tile
  };
  __device__ __forceinline__ Unit at(int u) const {
    // The last lane whose experts start at or before u.
    const int src = __builtin_popcountll(__builtin_amdgcn_ballot_w64(before <= u)) - 1;
    int local = u - __builtin_amdgcn_readlane(before, src);
    Unit un;
    un.e = 4 * src;
    int n = __builtin_amdgcn_readlane(cnt[0], src), o = __builtin_amdgcn_readlane(off[0], src);
#pragma unroll
    for (int j = 1; j < 4; ++j) {
      const int sz = blocks(n) * ntiles;
      const bool past = un.e == 4 * src + j - 1 && local >= sz;
      const int nn = __builtin_amdgcn_readlane(cnt[j], src), on = __builtin_amdgcn_readlane(off[j], src);
      local -= past ? sz : 0;
      un.e += past ? 1 : 0;
      n = past ? nn : n;
      o = past ? on : o;
    }
    const int m = blocks(n);
    un.nt = local / m;
    const int b = local - un.nt * m;
    const int per = ((n + m - 1) / m + 31) & ~31;  // equal heights, whole 32-row blocks
    un.row0 = o + b * per;
    un.rows = min(per, n - b * per);
    return un;
  }
};

// SiLU(g) * u in fp32, bit for bit what the streaming kernels compute.  The
// hardware's base-2 exponential and reciprocal instead of expf and the division
// would take 419 us for 434 (T = 4096 layer, E = 128, H = 2048, I = 768, K = 8),
// but are up to 57 units of 2^-24 off for large |g| and flush g < -87 to 0.
__device__ __forceinline__ float swiglu(float g, float u) { return g / (1.0f + expf(-g)) * u; }

// Streaming stores: act and routed rows are read by the next launch only, and
// lines left dirty in L2 (up to 32 MiB over the XCDs) are written back at the
// end of the kernel, when nothing else runs (down at T = 1024: 87 -> 79 us).
__device__ __forceinline__ void store_row(uint16_t *p, u32x4 v) { __builtin_nontemporal_store(v, (u32x4 *)p); }

// 16-byte chunk c of row m of a stage's 32-row fragment sits at chunk c ^
// swz(m).  A 128-byte row covers half of the 64 banks, so sixteen lanes served
// together must hold each of the eight chunks twice, in an even and an odd row.
// Those are lanes 0-3, 12-15, 20-23 and 24-27 of a 16-byte operand read (and the
// other sixteen of 32), not consecutive ones: with (m >> 1) ^ (m >> 3 & 2), which
// is conflict-free for consecutive lanes only, half of the LDS cycles were
// conflicts (SQ_LDS_BANK_CONFLICT / SQ_LDS_IDX_ACTIVE 0.50).  The Gray code of m / 4
// serves both groupings (consecutive rows, one chunk): 0.02 in gate/up, 0.08 with
// the down epilogue; the W4 kernel, whose loaders write rows 8 q + 4 hb + i of one
// chunk, keeps 0.30.  Times moved by less than 1 %: the LDS does not bound these
// kernels.
__device__ __forceinline__ int swz(int m) { return (((m >> 2) ^ (m >> 3)) & 3) << 1 | ((m >> 1) & 1); }
// swz(8 j + lr) for lr < 8 is (lr >> 1) ^ swz8(j).
__device__ __forceinline__ uint32_t swz8(int j) { return (uint32_t)(4 * ((j ^ (j >> 1)) & 1) | 2 * (j & 1)); }

// Weight row within a 32-row fragment that LDS row m of it holds: the MFMA
// leaves output rows 8 q + 4 h + i (q, i = 0..3) in lane half h, so with this
// order a lane's sixteen outputs are sixteen consecutive columns.
__device__ __forceinline__ int frag_row(int m) { return 16 * ((m >> 2) & 1) + 4 * (m >> 3) + (m & 3); }

// Token of this lane's row 32 b + 8 lw + lr of each token block of a unit, rows
// past the unit's end repeating its first row.  Scalar loads, every one of
// them issued before the first is used and none behind a branch: the
// vector-memory counter holds only LDS loads, so nothing here waits on those,
// and the loaders stand still for one memory round trip per unit (with the
// loads behind per-row conditions, up to forty in a row, T = 4096 gate/up took
// 237 us instead of 232).  Blocks past the unit's rows read block 0's tokens.
template <int NBM>
__device__ __forceinline__ void token_rows(const ExpertArgs &a, const UnitMap::Unit &un, int lw, int lr,
                                           uint32_t (&rows)[NBM]) {
  const MOE_CONST int32_t *rt = as_const(a.row_token) + un.row0;
  const int nb = (un.rows + 31) >> 5;
  const int t0 = rt[0];
  int tk[NBM][8];
#pragma unroll
  for (int b = 0; b < NBM; ++b) {
    const MOE_CONST int32_t *p = rt + (b < nb ? b : 0) * 32 + lw * 8;  // at most 31 rows past the unit's end
#pragma unroll
    for (int k = 0; k < 8; ++k) tk[b][k] = p[k];
  }
#pragma unroll
  for (int b = 0; b < NBM; ++b) {
    int tok = tk[b][0];
#pragma unroll
    for (int k = 1; k < 8; ++k) tok = lr == k ? tk[b][k] : tok;
    rows[b] = (uint32_t)(b * 32 + lw * 8 + lr < un.rows ? tok : t0);
  }
}

template <int KIND, int NBM>
__device__ __forceinline__ void load_role(const ExpertArgs &a, const UnitMap &map, int first, int stride, int nu,
                                          int lw, int lane, uint8_t *smem) {
  constexpr int kSlots = ring_slots(NBM), kSlotBytes = slot_bytes(NBM);
  const int H = a.H, I = a.I;
  const int Kdim = KIND == 0 ? H : I;
  const int KT = (Kdim + kBK - 1) / kBK;
  const int nstages = nu * KT;
  const uint32_t pitch = (uint32_t)Kdim * 2u;
  const uint32_t tail = (uint32_t)(Kdim % kBK) / 8u;  // 16-byte chunks in a partial last stage
  const int lr = lane >> 3;

  // Loader wave lw moves LDS rows [64 lw, +64) of the weight tile and rows
  // 32 b + 8 lw .. + 8 of each token block, eight rows (1 KiB) per load.  LDS
  // chunk lane % 8 of row r holds logical chunk (lane % 8) ^ swz(r).
  const uint8_t *xbase = KIND == 0 ? (const uint8_t *)a.x : (const uint8_t *)a.act;
  const uint32_t xbytes = KIND == 0 ? (uint32_t)a.T * pitch : (uint32_t)a.R * pitch;
  const auto brs = __builtin_amdgcn_make_buffer_rsrc((void *)xbase, (short)0, (int)xbytes, 0x00020000);
  __amdgpu_buffer_rsrc_t ars;
  uint32_t aoff[kAPer], boff[NBM];
  const uint32_t c0 = (uint32_t)((lane & 7) ^ (lr >> 1));
  int cur = -1, nb = 0;
  auto setup = [&](int i) {
    const UnitMap::Unit un = map.at(first + i * stride);
    nb = (un.rows + 31) >> 5;
    const size_t mat = (size_t)(KIND == 0 ? I : H) * pitch;  // one expert's gate, up or down matrix
    const uint8_t *wb = KIND == 0 ? (const uint8_t *)a.gate_up + ((size_t)un.e * 2 + (lw >> 1)) * mat
                                  : (const uint8_t *)a.down + (size_t)un.e * mat;
    ars = __builtin_amdgcn_make_buffer_rsrc((void *)wb, (short)0, (int)(uint32_t)mat, 0x00020000);
    // gate/up: LDS rows 0..127 are gate rows, 128..255 the up rows (the base above).
    const int wrow0 = KIND == 0 ? un.nt * (kBN / 2) + (lw & 1) * 64 : un.nt * kBN + lw * 64;
#pragma unroll
    for (int j = 0; j < kAPer; ++j) {
      const int row = wrow0 + (j / 4) * 32 + frag_row((j & 3) * 8 + lr);
      aoff[j] = (uint32_t)row * pitch + ((c0 ^ swz8(j & 3)) << 4);
    }
    uint32_t rows[NBM];
    if (KIND == 0) token_rows<NBM>(a, un, lw, lr, rows);
#pragma unroll
    for (int b = 0; b < NBM; ++b) {
      const int r0 = b * 32 + lw * 8 + lr;
      if (KIND == 1) rows[b] = (uint32_t)(un.row0 + (r0 < un.rows ? r0 : 0));
      boff[b] = rows[b] * pitch + ((c0 ^ swz8(lw)) << 4);
    }
  };
  int slot = 0, kt_next = 0, unit_next = 0;
  // Issue stage (unit_next, kt_next); returns the loads issued.
  auto issue = [&]() {
    if (unit_next != cur) {
      setup(unit_next);
      cur = unit_next;
    }
    uint8_t *buf = smem + slot * kSlotBytes;
    const uint32_t koff = (uint32_t)kt_next * (kBK * 2);
    const bool part = tail != 0 && kt_next == KT - 1;
    // Chunks past K are out of range; tail is 4, so bit 2 of the chunk decides.
    const uint32_t past[2] = {part && c0 >= tail ? 0xffffffffu : 0u, part && (c0 ^ 4u) >= tail ? 0xffffffffu : 0u};
#pragma unroll
    for (int j = 0; j < kAPer; ++j)
      buffer_load_lds16(ars, buf + (lw * 64 + j * 8) * 128, aoff[j] | past[swz8(j & 3) >> 2], koff);
    const uint32_t ob = past[swz8(lw) >> 2];
#pragma unroll
    for (int b = 0; b < NBM; ++b) {
      if (b >= nb) break;
      buffer_load_lds16(brs, buf + kABytes + (b * 32 + lw * 8) * 128, boff[b] | ob, koff);
    }
    order_loads();
    slot = slot == kSlots - 1 ? 0 : slot + 1;
    if (++kt_next == KT) {
      kt_next = 0;
      ++unit_next;
    }
    return kAPer + nb;
  };
  // Loads of the stages in flight behind stage st: st + 1 (and, with four
  // slots, st + 2).
  int n1 = 0, n2 = 0;
  if (nstages > 0) issue();
  if (nstages > 1) n1 = issue();
  if (kSlots == 4 && nstages > 2) n2 = issue();
  for (int st = 0; st < nstages; ++st) {
    wait_vmcnt_upto(n1 + n2);  // stage st has landed
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    // The slot of stage st - 1 was last read before this barrier.
    const int n = st + kSlots - 1 < nstages ? issue() : 0;
    n1 = kSlots == 4 ? n2 : n;
    n2 = kSlots == 4 ? n : 0;
  }
}

// 16 bytes of LDS per lane, written from inline assembly: the compiler would
// make an LDS store of its own wait for every LDS-destination load in flight,
// here the token tiles of the next stages.  Completed by an explicit
// lgkmcnt(0) before the stage's barrier.
template <int OFF>
__device__ __forceinline__ void lds_write_b128(uint32_t addr, u32x4 v) {
  asm volatile("ds_write_b128 %0, %1 offset:%2" ::"v"(addr), "v"(v), "i"(OFF) : "memory");
}

// W4G128 gate/up: the loader waves stream the int4 words into registers (one
// 1 KiB load per 16 rows x 128 K, i.e. per two stages, three pairs of stages ahead),
// decode them bit-exactly and write the bf16 weight tile of stage st + 1 while
// the MFMA waves multiply stage st, so each weight is decoded once per unit of
// up to 160 rows and the MFMA waves issue no decode.  Token tiles come as in
// the bf16 kernel, always NBM loads per stage (blocks past the unit's rows are
// out of range), so every wait is a constant count.  T = 4096, E = 128, H =
// 2048, I = 768, K = 8: 233 us (885 TFLOP/s) against 311 us with the pair
// kernel, as fast as the bf16 weights; without the word loads and the decode
// 203 us.  The MFMAs are busy 30 % of its cycles (T = 3001, Zipf), so they do not
// bound it; real operands cost clock (zero ones: 271 -> 214 us back to back).
template <int NBM>
__device__ __forceinline__ void load_role_w4(const ExpertArgs &a, const UnitMap &map, int first, int stride, int nu,
                                             int lw, int lane, uint8_t *smem) {
  using R = Ring<NBM, true>;
  constexpr int kLead = R::kBSlots - 1;  // token tiles in flight, in stages
  constexpr int kWLoads = 8;  // words and scales of the wave's four row blocks, per pair
  const int H = a.H, I = a.I;
  const int KP = H / 128, KT = 2 * KP;  // pairs and stages per unit
  const int nstages = nu * KT;
  if (nstages == 0) return;
  const uint32_t pitch = (uint32_t)H * 2u;
  const int r = lane & 15, g = lane >> 4;

  // ---- token tiles ----
  const auto brs = __builtin_amdgcn_make_buffer_rsrc((void *)a.x, (short)0, (int)((uint32_t)a.T * pitch), 0x00020000);
  const int lr = lane >> 3;
  const uint32_t bchunk = (uint32_t)((lane & 7) ^ swz(8 * lw + lr)) << 4;
  uint32_t boff[NBM];
  int b_unit = 0, b_kt = 0, b_slot = 0;
  auto issue_b = [&]() __attribute__((always_inline)) {
    if (b_kt == 0) {
      const bool in = b_unit < nu;  // past the last unit: loads that read nothing
      const UnitMap::Unit un = map.at(first + (in ? b_unit : nu - 1) * stride);
      uint32_t rows[NBM];
      token_rows<NBM>(a, un, lw, lr, rows);
#pragma unroll
      for (int b = 0; b < NBM; ++b) boff[b] = in && b * 32 < un.rows ? rows[b] * pitch + bchunk : 0xffffffffu;
    }
    uint8_t *dst = smem + R::kB0 + b_slot * R::kBStride + lw * 8 * 128;
#pragma unroll
    for (int b = 0; b < NBM; ++b) buffer_load_lds16(brs, dst + b * 32 * 128, boff[b], (uint32_t)b_kt * (kBK * 2));
    order_loads();
    b_slot = b_slot == R::kBSlots - 1 ? 0 : b_slot + 1;
    if (++b_kt == KT) {
      b_kt = 0;
      ++b_unit;
    }
  };

  // ---- weight words: blocks f, hb = rows 32 f + 16 hb .. + 16 of the wave's 64 ----
  u32x4 wq[3][4];
  uint32_t sc[3][4];
  const uint32_t half_words = (uint32_t)I * (uint32_t)H / 2u, half_scales = (uint32_t)(I / 16) * KP * 32u;
  __amdgpu_buffer_rsrc_t wrs, srs;
  uint32_t woff = 0, soff = 0;
  int w_unit = 0, w_kp = 0;
  auto issue_w = [&](int buf) __attribute__((always_inline)) {
    if (w_kp == 0) {
      const UnitMap::Unit un = map.at(first + min(w_unit, nu - 1) * stride);
      const size_t half = (size_t)un.e * 2 + (lw >> 1);  // gate rows, then up rows
      wrs = __builtin_amdgcn_make_buffer_rsrc((void *)((const uint8_t *)a.w4_words + half * half_words), (short)0,
                                              (int)half_words, 0x00020000);
      srs = __builtin_amdgcn_make_buffer_rsrc((void *)((const uint8_t *)a.w4_scales + half * half_scales), (short)0,
                                              (int)half_scales, 0x00020000);
      const uint32_t n16 = (uint32_t)(un.nt * (kBN / 2) + (lw & 1) * 64) / 16u;
      woff = n16 * (uint32_t)KP * 1024u + (uint32_t)lane * 16u;
      soff = n16 * (uint32_t)KP * 32u + (uint32_t)r * 2u;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      wq[buf][j] = __builtin_bit_cast(
          u32x4, __builtin_amdgcn_raw_buffer_load_b128(wrs, woff + (uint32_t)(j * KP) * 1024u, w_kp * 1024, 0));
      sc[buf][j] = __builtin_amdgcn_raw_buffer_load_b16(srs, soff + (uint32_t)(j * KP) * 32u, w_kp * 32, 0);
    }
    order_loads();
    if (++w_kp == KP) {
      w_kp = 0;
      ++w_unit;
    }
  };
  // Weight row 16 hb + r of a fragment sits in LDS row m = 8 (r / 4) + 4 hb +
  // r % 4 (frag_row's inverse); word 2 s + jj of a lane is chunk 4 jj + g of
  // stage half s.
  uint32_t wdst[2][2];
#pragma unroll
  for (int hb = 0; hb < 2; ++hb)
#pragma unroll
    for (int jj = 0; jj < 2; ++jj) {
      const int m = 8 * (r >> 2) + 4 * hb + (r & 3);
      wdst[hb][jj] = (uint32_t)(lw * 64 + m) * 128u + (((4 * jj + g) ^ swz(m)) << 4) +
                     (uint32_t)(uintptr_t)(const MOE_LDS uint8_t *)smem;
    }
  int d_slot = 0;
  auto decode = [&](int buf, int s) __attribute__((always_inline)) {
    const uint32_t base = (uint32_t)(d_slot * R::kAStride);
#pragma unroll
    for (int hb = 0; hb < 2; ++hb)
#pragma unroll
      for (int f = 0; f < 2; ++f) {
        const W4Scale k = w4_scale(bf16_bits_to_f32(sc[buf][2 * f + hb]));
#pragma unroll
        for (int jj = 0; jj < 2; ++jj) {
          const u32x4 v = w4_decode8(wq[buf][2 * f + hb][2 * s + jj], k);
          if (f == 0) lds_write_b128<0>(base + wdst[hb][jj], v);
          else lds_write_b128<4096>(base + wdst[hb][jj], v);
        }
      }
    d_slot ^= 1;
  };

#pragma unroll
  for (int i = 0; i < kLead; ++i) issue_b();
  issue_w(0);
  issue_w(1);
  issue_w(2);
  decode(0, 0);
  int st = 0;
  // Stage st is published, stage st + 1 decoded (half 1 of a pair in even
  // stages) and the token tile of stage st + kLead requested.  The token tile
  // of stage st was followed by kLead - 1 later ones and by the words issued
  // in the even ones of stages st - kLead .. st - 1.
  auto stage = [&](auto even, int buf) __attribute__((always_inline)) {
    constexpr int kWords = decltype(even)::value ? kLead / 2 : (kLead + 1) / 2;
    constexpr int kLater = (kLead - 1) * NBM + kWords * kWLoads;
    constexpr int kWait = kLater < 63 ? kLater : 63;
    __builtin_amdgcn_s_waitcnt((kWait & 15) | ((kWait >> 4) << 14) | (7 << 4));
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    issue_b();
    if (st + 1 < nstages) decode(buf, decltype(even)::value ? 1 : 0);
    if (decltype(even)::value) issue_w(buf);  // the pair three after the one just decoded
    ++st;
  };
  const std::true_type even;
  const std::false_type odd;
  while (true) {  // nstages is even; word buffers 0, 1, 2 in turn
    stage(even, 0);
    stage(odd, 1);
    if (st >= nstages) break;
    stage(even, 1);
    stage(odd, 2);
    if (st >= nstages) break;
    stage(even, 2);
    stage(odd, 0);
    if (st >= nstages) break;
  }
  wait_vmcnt<0>();  // nothing may reach the LDS after the workgroup has ended
}

// One unit on MFMA wave w with NB token blocks; a_slot and b_slot are the ring
// slots of the unit's first stage, advanced past its last.
template <int KIND, int NB, int NBM, bool W4>
__device__ __forceinline__ void mfma_unit(const ExpertArgs &a, const UnitMap::Unit &un, int KT, int &a_slot,
                                          int &b_slot, int w, int lane, const uint8_t *smem) {
  using R = Ring<NBM, W4>;
  const int r = lane & 31, h = lane >> 5;
  f32x16 acc[2][NB];
#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[q][b][i] = 0.f;
  // Down: route of each of this lane's rows, requested before the K loop (a
  // load between the epilogue's stores would wait for them).
  int route[NB];
  if (KIND == 1) {
#pragma unroll
    for (int b = 0; b < NB; ++b) route[b] = 32 * b + r < un.rows ? a.row_route[un.row0 + 32 * b + r] : -1;
  }
  // Byte offset of this lane's chunk of K-step ks within a 32-row fragment.
  uint32_t lo[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) lo[ks] = (uint32_t)(r * 128 + (((2 * ks + h) ^ swz(r)) << 4));
  const uint32_t a0 = KIND == 0 ? w * 4096 : w * 8192, a1 = KIND == 0 ? 16384 + w * 4096 : w * 8192 + 4096;

  // One K-step: the MFMAs of the fragments read a step ago, with the next
  // step's fragment reads issued between them.
  u32x4 af[2][2], bf[2][NB];
  const uint8_t *abuf = smem, *bbuf = smem;
  auto read_one = [&](int set, int ks, int i) __attribute__((always_inline)) {
    if (i == 0) af[set][0] = *(const u32x4 *)(abuf + a0 + lo[ks]);
    else if (i == 1) bf[set][0] = *(const u32x4 *)(bbuf + lo[ks]);
    else if (i == 2) af[set][1] = *(const u32x4 *)(abuf + a1 + lo[ks]);
    else if (i < NB + 2) bf[set][i - 2] = *(const u32x4 *)(bbuf + (i - 2) * 4096 + lo[ks]);
  };
  auto step = [&](int set, int ks) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2 * NB; ++i) {
      acc[i & 1][i >> 1] = mfma32(af[set][i & 1], bf[set][i >> 1], acc[i & 1][i >> 1]);
      if (i < NB + 2) {
        __builtin_amdgcn_sched_barrier(0);
        read_one(set ^ 1, ks, i);
        if (i == 2 * NB - 1)
          for (int j = 2 * NB; j < NB + 2; ++j) read_one(set ^ 1, ks, j);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  for (int kt = 0; kt < KT; ++kt) {
    lds_barrier();  // the stage is published; every read of the stage before it is done
    abuf = smem + a_slot * R::kAStride;
    bbuf = smem + R::kB0 + b_slot * R::kBStride;
    a_slot = a_slot == R::kASlots - 1 ? 0 : a_slot + 1;
    b_slot = b_slot == R::kBSlots - 1 ? 0 : b_slot + 1;
    if (kt == 0) {
#pragma unroll
      for (int i = 0; i < NB + 2; ++i) read_one(0, 0, i);
    } else {
      step(1, 0);
    }
    step(0, 1);
    step(1, 2);
    step(0, 3);
  }
#pragma unroll
  for (int i = 0; i < 2 * NB; ++i) acc[i & 1][i >> 1] = mfma32(af[1][i & 1], bf[1][i >> 1], acc[i & 1][i >> 1]);

  // Epilogue.  Lane (r, h) holds token row 32 b + r, columns 16 h .. + 16 of
  // each fragment.  The rows go out through this wave's own weight rows of the
  // last stage (8 KiB that only this wave reads, and that the loaders refill
  // only after the next barrier), so that every store instruction writes whole
  // 64-byte (act) or 128-byte (routed) pieces of its rows: straight from the
  // accumulators (16-byte pieces of 32 rows) the stores took 45 of the down
  // projection's 150 us at T = 4096.
  uint8_t *const scratch = const_cast<uint8_t *>(abuf);
  if (KIND == 0) {
    if (un.nt * (kBN / 2) + w * 32 >= a.I) return;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      uint8_t *const sc = scratch + (b & 1 ? a1 : a0);  // 32 rows of 64 bytes
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        u32x4 o;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int i = 8 * c + 2 * j;
          const uint32_t g = pack_bf16x2(acc[0][b][i], acc[0][b][i + 1]);
          const uint32_t u = pack_bf16x2(acc[1][b][i], acc[1][b][i + 1]);
          o[j] = pack_bf16x2(swiglu(bf16_bits_to_f32(g & 0xffffu), bf16_bits_to_f32(u & 0xffffu)),
                             swiglu(bf16_bits_to_f32(g >> 16), bf16_bits_to_f32(u >> 16)));
        }
        *(u32x4 *)(sc + r * 64 + (((2 * h + c) ^ ((r >> 2) & 3)) << 4)) = o;
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int row = 16 * i + (lane >> 2), c = lane & 3;
        const u32x4 o = *(const u32x4 *)(sc + row * 64 + ((c ^ ((row >> 2) & 3)) << 4));
        if (32 * b + row < un.rows)
          store_row(a.act + (size_t)(un.row0 + 32 * b + row) * a.I + un.nt * (kBN / 2) + w * 32 + c * 8, o);
      }
    }
  } else {
    const int col = un.nt * kBN + w * 64 + (lane & 7) * 8;
    const bool live = un.nt * kBN + w * 64 + (lane & 4) * 8 < a.H;  // 32-column fragments
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      uint8_t *const sc = scratch + (b & 1 ? a1 : a0);  // 32 rows of 128 bytes
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          u32x4 o;
#pragma unroll
          for (int j = 0; j < 4; ++j) o[j] = pack_bf16x2(acc[q][b][8 * c + 2 * j], acc[q][b][8 * c + 2 * j + 1]);
          *(u32x4 *)(sc + r * 128 + (((4 * q + 2 * h + c) ^ ((r >> 1) & 7)) << 4)) = o;
        }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = 8 * i + (lane >> 3);
        const u32x4 o = *(const u32x4 *)(sc + row * 128 + (((lane & 7) ^ ((row >> 1) & 7)) << 4));
        const int q0 = __shfl(route[b], row, kWave);
        if (q0 >= 0 && live) store_row(a.routed + (size_t)q0 * a.H + col, o);
      }
    }
  }
}

template <int KIND, int NBM, bool W4>
__global__ __launch_bounds__(kThreads) void tile_kernel(ExpertArgs a, int max_rows) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int wave = sgpr(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int tasks = *as_const(a.num_tasks);
  UnitMap map;
  map.init(a.counts, a.offsets, a.E, KIND == 0 ? (a.I + kBN / 2 - 1) / (kBN / 2) : (a.H + kBN - 1) / kBN, max_rows,
           lane);
  if (tasks == 0) return;  // no route, or a plan that stalled
  // One contiguous chunk of the unit sequence per XCD (consecutive workgroup
  // IDs go round-robin over the XCDs), walked by the XCD's workgroups together.
  const int G = gridDim.x;
  const bool xcd_mode = G % 8 == 0;
  const int P = xcd_mode ? G / 8 : G;  // workgroups per chunk
  const int xcd = xcd_mode ? (int)blockIdx.x % 8 : 0;
  const int p = xcd_mode ? (int)blockIdx.x / 8 : (int)blockIdx.x;
  const int CH = xcd_mode ? (map.total + 7) / 8 : map.total;  // units per chunk
  const int c_end = min(CH, map.total - xcd * CH);
  const int nu = p < c_end ? (c_end - p + P - 1) / P : 0;
  const int first = xcd * CH + p;
  if (wave >= kMfmaWaves) {
    if constexpr (W4) load_role_w4<NBM>(a, map, first, P, nu, wave - kMfmaWaves, lane, smem);
    else load_role<KIND, NBM>(a, map, first, P, nu, wave - kMfmaWaves, lane, smem);
    return;
  }
  const int KT = ((KIND == 0 ? a.H : a.I) + kBK - 1) / kBK;
  int sa = 0, sb = 0;
  for (int i = 0; i < nu; ++i) {
    const UnitMap::Unit un = map.at(first + i * P);
    sa = sgpr(sa);
    sb = sgpr(sb);
    const int nb = sgpr((un.rows + 31) >> 5);
    if (nb == 1) {
      mfma_unit<KIND, 1, NBM, W4>(a, un, KT, sa, sb, wave, lane, smem);
    } else if (NBM == 2 || nb == 2) {
      mfma_unit<KIND, 2, NBM, W4>(a, un, KT, sa, sb, wave, lane, smem);
    } else if constexpr (NBM > 2) {
      if (NBM == 3 || nb == 3) {
        mfma_unit<KIND, 3, NBM, W4>(a, un, KT, sa, sb, wave, lane, smem);
      } else if constexpr (NBM > 3) {
        if (nb == 4) mfma_unit<KIND, 4, NBM, W4>(a, un, KT, sa, sb, wave, lane, smem);
        else mfma_unit<KIND, 5, NBM, W4>(a, un, KT, sa, sb, wave, lane, smem);
      }
    }
  }
}

template <int KIND, int NBM, bool W4>
hipError_t launch_nbm(const ExpertArgs &a, int max_rows, int num_cus, hipStream_t s) {
  auto k = tile_kernel<KIND, NBM, W4>;
  const size_t lds = (size_t)Ring<NBM, W4>::kBytes;
  static bool attr = [&] {
    return hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)lds) == hipSuccess;
  }();
  if (!attr) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k, dim3(num_cus), dim3(kThreads), lds, s, a, max_rows);
  return hipGetLastError();
}

// Token blocks per unit at most, from the shape alone (a captured launch stays
// valid for any routes).  High units load each weight tile least often and win
// where experts have many rows: 160-row units against 96-row ones took 307 vs
// 334 us per layer at E = 128, H = 2048, I = 768, K = 8, T = 2048 (mean 128)
// and 425 vs 448 at E = 32, H = I = 2880, K = 4, T = 1024 (Zipf routing).
// Below a mean of 128 rows 96-row units waste less of the last round: T = 1024
// Zipf 242 vs 255 us, uniform 266 vs 267 (64-row units: 262 and 293).  While
// the units leave half the CUs idle, lower ones that make more of them: the
// four-slot ring of 64 rows (16 experts, H = 2048, I = 768, 64 rows each: 66.3 vs
// 67.9 us), 96 rows where one 128- or 160-row block holds the mean expert (128
// rows each, gate/up: 81.4 -> 74.3 us, Zipf 78.7 -> 74.9), then 32-row units where
// an expert's rows still make more of them (E = 8, H = 512, I = 256, 256 rows
// each: 26.5 vs 28.3 us).  Where they would then fill all the CUs, the experts
// above the mean of a skewed routing make a second round (16 experts of 88 rows,
// down with 64 rows: uniform 67.8 -> 65.8 us, Zipf 68.6 -> 75.3), so exactly half
// is lowered only where three quarters result (E = 16, H = 1024, I = 512, 175 rows
// each: 46.2 -> 37.7 us, Zipf 46.8 -> 37.8).  Two 64-row blocks instead of two in 96-row units under the
// same condition: with a quarter of the round to spare up to 112 rows, with
// half above (gate/up of 16 experts of 97 / 119 rows 74.3 -> 69.8 / 74.0 -> 75.0, Zipf
// 73.6 -> 70.9 / 74.1 -> 72.2, of 127 rows Zipf 80.9 -> 95.4; H = 1024, I = 512, 128
// rows 39.7 -> 36.7).
int unit_blocks(long long R, int E, int ntiles, int num_cus) {
  const long long mean = (R + E - 1) / E;
  auto units = [&](int nb) { return (long long)E * ntiles * ((mean + 32 * nb - 1) / (32 * nb)); };
  int nb = mean >= 128 ? kMaxNB : mean > 40 ? 3 : 2;
  if (nb == 3 && mean <= 64 && 2 * units(2) <= num_cus) nb = 2;
  while (2 * units(nb) <= num_cus) {
    int n = nb - 1;
    while (n > 1 && units(n) == units(nb)) --n;  // the next height that makes more units
    if (n < 1 || (n == 1 && mean <= 64)) break;
    if (2 * units(nb) == num_cus && 4 * units(n) > 3LL * num_cus) break;
    nb = n;
  }
  if (nb == 3 && mean > 96 && mean <= 128 && 4 * units(2) <= (mean <= 112 ? 3LL : 2LL) * num_cus) nb = 2;
  return nb;
}

int unit_blocks(const ExpertArgs &a, bool down, int num_cus) {
  return unit_blocks(a.R, a.E, down ? (a.H + kBN - 1) / kBN : (a.I + kBN / 2 - 1) / (kBN / 2), num_cus);
}

template <int KIND, bool W4>
hipError_t launch_tile(const ExpertArgs &a, int num_cus, hipStream_t s) {
  const int nb = unit_blocks(a, KIND == 1, num_cus);
  if (nb <= 2) return launch_nbm<KIND, 2, W4>(a, 32 * nb, num_cus, s);
  // W4 loads (and zero-fills) NBM token blocks per stage.
  if (W4 && nb == 3) return launch_nbm<KIND, W4 ? 3 : kMaxNB, W4>(a, 32 * nb, num_cus, s);
  return launch_nbm<KIND, kMaxNB, W4>(a, 32 * nb, num_cus, s);
}

}  // namespace

bool tile_gemm_ok(int H, int I) {
  // Whole 32-row fragments and 16-byte chunks; byte offsets within one
  // expert's gate, up or down matrix, the last tile's rows past its end
  // included (they must not wrap back into it), fit 32 bits.  (Descriptors of a
  // wave's own 64 rows instead of the matrix would take larger ones, but
  // lengthen the loaders' set-up per unit: T = 4096 442 -> 453 us, W4 T = 3001 391
  // -> 419, E = 128, H = 2048, I = 768, K = 8.)
  const long long limit = 1LL << 32;
  return H % 32 == 0 && I % 32 == 0 && 2LL * H * (I + kBN / 2) < limit && 2LL * I * (H + kBN) < limit;
}

bool tile_shape_ok(int H, int I) { return I % 128 == 0 && H % 256 == 0 && tile_gemm_ok(H, I); }

int tile_unit_rows(const ExpertArgs &a, bool down, int num_cus) { return 32 * unit_blocks(a, down, num_cus); }

hipError_t launch_tile_gate_up(const ExpertArgs &a, bool w4, int num_cus, hipStream_t s) {
  return w4 ? launch_tile<0, true>(a, num_cus, s) : launch_tile<0, false>(a, num_cus, s);
}

hipError_t launch_tile_down(const ExpertArgs &a, int num_cus, hipStream_t s) {
  return launch_tile<1, false>(a, num_cus, s);
}

}  // namespace moe
