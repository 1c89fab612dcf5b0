// Segmented-KV GQA prefill attention for long chunks on gfx950 (semantics as in
// gqa_attention.hip; reference: compact_gqa_forward,
// cuda_gqa_attention_compact.cu:77-209).
//
// The kernel of gqa_attention.hip lets every wave stream its own share of the
// keys for 32 query rows: each K/V byte goes into LDS once per 32 rows, and the
// LDS traffic and the short dependent steps bound it.  With many query rows
// there is work for sharing instead: here a workgroup owns 256 query rows of
// one KV head (all its query heads x 256 / group tokens), 32 per MFMA wave,
// and all eight MFMA waves read the same 64-key stages.  Four loader waves
// move the stages global -> LDS (buffer loads with an LDS destination, whole
// 256-byte rows, three stages ahead in a ring of four) and carry every
// vector-memory wait; one workgroup barrier per stage publishes it and frees
// the oldest.
//
// Per 32 keys a wave computes S^T = K Q^T with 32x32x16 MFMAs (Q fragments in
// registers for the whole kernel), so a lane holds sixteen scores of its own
// query, the online softmax is lane-local (the partner lane l ^ 32 holds the
// other sixteen; their maxima meet only when a rescale is due), and P is
// already the B operand of O^T = V^T P^T: the keys of each 16-key step are
// taken in the order the scores lie in, and V is read transposed in that order
// with ds_read_b64_tr_b16.  O^T keeps a query per lane, so rescaling is
// lane-local too.
#include <type_traits>

#include "common.h"
#include "gqa_internal.h"

namespace moe {

namespace {

constexpr int kD = 128;
constexpr int kStageKeys = 64;
constexpr int kMfmaWaves = 8;
constexpr int kLoaders = 4;
constexpr int kThreads = (kMfmaWaves + kLoaders) * 64;
// A stage's tile in LDS: sixteen blocks of 1 KiB, block b holding the rows of
// keys b, b + 16, b + 32, b + 48 (one load instruction), padded so that the
// blocks start 16 bytes (K) or 64 bytes (V) further through the banks: the
// sixteen lanes of a K operand read take one chunk of sixteen consecutive
// keys, the lanes of a transposed V read 64 bytes of four, and both then
// cover all banks with one address register and immediate offsets.
constexpr int kKBlock = 1024 + 16;
constexpr int kVBlock = 1024 + 64;
constexpr int kVTile = 16 * kKBlock;  // V after K
constexpr int kStageBytes = 16 * (kKBlock + kVBlock);
constexpr int kSlots = 4;
constexpr int kKRing = 5;  // K fragments in registers
constexpr int kPerStage = 8;  // loads of a loader wave per stage
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kRescaleSlack = 8.f;  // as in gqa_attention.hip
static_assert(kSlots * kStageBytes <= 160 * 1024, "stage ring fits the LDS");

#define GQA_LDS __attribute__((address_space(3)))
typedef short i16x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ int sgpr(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ uint64_t sgpr64(uint64_t v) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return ((uint64_t)hi << 32) | lo;
}
__device__ __forceinline__ f32x16 mfma32(u32x4 a, u32x4 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(a), as_bf16x8(b), c, 0, 0, 0);
}
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}
__device__ __forceinline__ void buffer_load_lds16(__amdgpu_buffer_rsrc_t rs, uint8_t *dst, uint32_t off) {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (GQA_LDS void *)dst, 16, off, 0, 0, 0);
#endif
}
// Within each group of 16 lanes, lane 4a + b receives element b of the 8-byte
// rows addressed by lanes a, a + 4, a + 8, a + 12.
__device__ __forceinline__ u32x2 lds_read_tr16(const uint8_t *p) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((GQA_LDS i16x4 *)p));
#else
  return u32x2{0u, 0u};
#endif
}
// The value of this lane and of lane l ^ 32, in the same order on both.
__device__ __forceinline__ f32x2_t halves(float x) {
  const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return f32x2_t{__uint_as_float(h[0]), __uint_as_float(h[1])};
}

constexpr int kXcds = 8;
__device__ __forceinline__ int xcd_logical_block(int id, int n) {
  const int x = id % kXcds, slot = id / kXcds, per = n / kXcds, extra = n % kXcds;
  return x * per + min(x, extra) + slot;
}

// The stage sequence of a workgroup: 64-key tiles that never straddle a
// segment (a segment's last tile may be short; empty segments have none).
struct Tiles {
  int len[kGqaMaxSegments];  // visible keys per segment
  int nseg;
  __device__ __forceinline__ int count() const {
    int t = 0;
#pragma unroll
    for (int s = 0; s < kGqaMaxSegments; ++s) t += (len[s] + kStageKeys - 1) / kStageKeys;
    return t;
  }
  __device__ __forceinline__ int length(int seg) const {
    return seg == 0 ? len[0] : seg == 1 ? len[1] : seg == 2 ? len[2] : len[3];
  }
  struct Tile {
    int seg, local0, n;
  };
  __device__ __forceinline__ Tile at(int t) const {
    Tile r{0, 0, 0};
#pragma unroll
    for (int s = 0; s < kGqaMaxSegments; ++s) {
      const int nt = (len[s] + kStageKeys - 1) / kStageKeys;
      const bool here = t >= 0 && t < nt;
      r.seg = here ? s : r.seg;
      r.local0 = here ? t * kStageKeys : r.local0;
      r.n = here ? min(kStageKeys, len[s] - t * kStageKeys) : r.n;
      t -= nt;
    }
    return r;
  }
};

// G query heads per KV head; wave w owns head w % G, tokens 32 (w / G) .. + 32
// of the workgroup's 256 / G.
template <int G>
__global__ __launch_bounds__(kThreads) void gqa_prefill_kernel(GqaArgs a, int nqb, int nsplit) {
  constexpr int QT = 32 * (kMfmaWaves / G);
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int lane = threadIdx.x & 63;
  const int wave = sgpr(threadIdx.x >> 6);
  const int lb = xcd_logical_block(blockIdx.x, gridDim.x);
  // The last query blocks first: they see the most keys.
  const int qb = nqb - 1 - lb % nqb, split = (lb / nqb) % nsplit, kvh = lb / (nqb * nsplit);
  const int q0 = qb * QT, T = a.T;

  Tiles tiles;
  tiles.nseg = a.num_segments;
#pragma unroll
  for (int s = 0; s < kGqaMaxSegments; ++s)
    tiles.len[s] = s >= a.num_segments ? 0 : s == a.num_segments - 1 ? min(T, q0 + QT) : a.len[s];
  const int total = tiles.count();
  const int t_beg = (int)((long long)total * split / nsplit), t_end = (int)((long long)total * (split + 1) / nsplit);
  const int nst = t_end - t_beg;

  if (wave >= kMfmaWaves) {
    // ---- loaders: wave lw moves blocks 4 lw .. + 4 of a stage's K and V tiles;
    // keys past a short tile's end are out of the descriptor's range: zeros.
    const int lw = wave - kMfmaWaves;
    const int kr = lane >> 4;
    int slot = 0;
    auto issue = [&](int st) {
      const Tiles::Tile t = tiles.at(t_beg + st);
      const uint32_t ksb = (uint32_t)(2 * a.k_stride[t.seg]), vsb = (uint32_t)(2 * a.v_stride[t.seg]);
      const uint64_t kb = (uint64_t)(a.k[t.seg] + (int64_t)t.local0 * a.k_stride[t.seg] + (int64_t)kvh * kD);
      const uint64_t vb = (uint64_t)(a.v[t.seg] + (int64_t)t.local0 * a.v_stride[t.seg] + (int64_t)kvh * kD);
      const auto krs = __builtin_amdgcn_make_buffer_rsrc((void *)sgpr64(kb), (short)0,
                                                         sgpr((int)((uint32_t)(t.n - 1) * ksb + 256u)), 0x00020000);
      const auto vrs = __builtin_amdgcn_make_buffer_rsrc((void *)sgpr64(vb), (short)0,
                                                         sgpr((int)((uint32_t)(t.n - 1) * vsb + 256u)), 0x00020000);
      uint8_t *const buf = smem + slot * kStageBytes;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t b = (uint32_t)(lw * 4 + j);
        buffer_load_lds16(krs, buf + b * kKBlock, (b + 16u * kr) * ksb + (uint32_t)((lane & 15) << 4));
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t b = (uint32_t)(lw * 4 + j);
        buffer_load_lds16(vrs, buf + kVTile + b * kVBlock, (b + 16u * kr) * vsb + (uint32_t)((lane & 15) << 4));
      }
      asm volatile("" ::: "memory");  // the counted waits below rely on the stages' order
      slot = slot == kSlots - 1 ? 0 : slot + 1;
    };
    for (int st = 0; st < kSlots - 1 && st < nst; ++st) issue(st);
    for (int st = 0; st < nst; ++st) {
      const int later = min(kSlots - 2, nst - 1 - st);  // stages in flight behind stage st
      if (later >= 2) wait_vmcnt<2 * kPerStage>();
      else if (later == 1) wait_vmcnt<kPerStage>();
      else wait_vmcnt<0>();
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if (st + kSlots - 1 < nst) issue(st + kSlots - 1);  // into the slot read before this barrier
    }
    return;
  }

  // ---- MFMA waves ----
  const int r = lane & 31, h = lane >> 5;
  const int head = kvh * G + wave % G;
  const int tok0 = q0 + 32 * (wave / G), tok = tok0 + r;
  u32x4 qf[8];
  {
    const uint16_t *qp = a.q + ((int64_t)min(tok, T - 1) * a.Hq + head) * kD + 8 * h;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) qf[ks] = *(const u32x4 *)(qp + 16 * ks);
  }
  float m_run = -INFINITY, l_run = 0.f;  // base-2 domain; l of this lane's keys only
  f32x16 o[4];
#pragma unroll
  for (int db = 0; db < 4; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[db][i] = 0.f;
  const float sl2 = a.scale * kLog2e;

  // K fragment ks of keys 32 hh + r: chunk 2 ks + h.  V, dims 32 db .. + 32: lane
  // 16 gi + 4 c + x reads dims 16 (gi % 2) + 4 x .. + 4 of key 4 (gi / 2) + c.
  const uint32_t kbase = (uint32_t)((r & 15) * kKBlock + (r >> 4) * 256 + h * 16);
  const uint32_t vbase = (uint32_t)(kVTile + (4 * (lane >> 5) + ((lane >> 2) & 3)) * kVBlock + ((lane >> 4) & 1) * 32 +
                                    (lane & 3) * 8);

  // The wave's half stages of 32 keys: all up to the diagonal of the causal
  // segment, where its 32 tokens meet their own keys (with the keys split that
  // half may lie in another workgroup).  The halves behind it hold nothing its
  // tokens see; they are left out, not only masked, because a probability of 0
  // times a V that is not finite is NaN.
  const int diag = tok0 < T ? 2 * (total - (min(T, q0 + QT) + kStageKeys - 1) / kStageKeys - t_beg) + tok0 / 32 : -1;
  const int nhalf = max(0, min(diag + 1, 2 * nst));

  // One half stage straight from global memory, each key's V only to the tokens
  // that see it.
  auto take_half = [&](const Tiles::Tile &t, int first, bool causal) __attribute__((always_inline)) {
    const int sg = sgpr(t.seg), row0 = t.local0 + first, n = min(32, t.n - first);
    if (n <= 0) return;
    const uint16_t *kp = a.k[sg] + (int64_t)(row0 + min(r, n - 1)) * a.k_stride[sg] + (int64_t)kvh * kD + 8 * h;
    f32x16 s;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.f;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) s = mfma32(*(const u32x4 *)(kp + 16 * ks), qf[ks], s);
    const int lim = causal ? min(n - 1, r) : n - 1;  // the last key that the lane's token sees
    float lmax = -INFINITY;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      s[i] = 8 * (i >> 2) + (i & 3) + 4 * h <= lim ? s[i] : -INFINITY;
      lmax = fmaxf(lmax, s[i] * sl2);
    }
    const f32x2_t top = halves(lmax);
    const float m_new = fmaxf(m_run, fmaxf(top[0], top[1]));
    const float alpha = __builtin_amdgcn_exp2f(m_run - (m_new == -INFINITY ? 0.f : m_new));
    l_run *= alpha;
    m_run = m_new;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[db][i] *= alpha;
    const float neg_m = m_run == -INFINITY ? 0.f : -m_run;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      s[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i], sl2, neg_m));
      l_run += s[i];
    }
#pragma clang loop unroll(disable)
    for (int key = 0; key < n; ++key) {
      // Lane half key / 4 % 2 holds the probability in s[4 (key / 8) + key % 4].
      const int at = 4 * (key >> 3) + (key & 3);
      float mine = s[0];
#pragma unroll
      for (int i = 1; i < 16; ++i) mine = at == i ? s[i] : mine;
      const f32x2_t both = halves(bf16_round(mine));
      const float p = key & 4 ? both[1] : both[0];
      const uint16_t *vp = a.v[sg] + (int64_t)(row0 + key) * a.v_stride[sg] + (int64_t)kvh * kD + 4 * h;
#pragma unroll
      for (int m = 0; m < 16; ++m) {
        const u32x2 v = *(const u32x2 *)(vp + 8 * m);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const float x = bf16_bits_to_f32(c & 1 ? v[c / 2] >> 16 : v[c / 2] & 0xffffu);
          const float acc = o[m / 4][4 * (m % 4) + c];
          o[m / 4][4 * (m % 4) + c] = key <= lim ? __builtin_fmaf(p, x, acc) : acc;
        }
      }
    }
  };

  // Keys of the current segment from the next stage on, and of the half stage
  // at hand and the rest of its stage.
  const Tiles::Tile t0 = tiles.at(t_beg);
  int seg = t0.seg, rem = nst > 0 ? tiles.length(seg) - t0.local0 : 0, left = 0, slot = 0;
  const uint8_t *buf = smem;
  auto enter = [&](int hf) __attribute__((always_inline)) {
    if (hf & 1) {
      left -= 32;
      buf += 512;
      return;
    }
    while (rem <= 0 && seg < kGqaMaxSegments - 1) rem = tiles.length(++seg);
    left = min(rem, kStageKeys);
    rem -= kStageKeys;
    lds_barrier();
    buf = smem + sgpr(slot) * kStageBytes;
    slot = slot == kSlots - 1 ? 0 : slot + 1;
  };
  for (int hf = 0; hf < nhalf; ++hf) {
    enter(hf);
    // The operand reads are issued in batches ahead of their MFMAs (left to
    // itself the compiler, short of registers, waits for each one).
    u32x4 kf[kKRing];
    auto read_k = [&](int ks) __attribute__((always_inline)) {
      kf[ks % kKRing] = *(const u32x4 *)(buf + kbase + ks * 32);
    };
#pragma unroll
    for (int ks = 0; ks < kKRing; ++ks) read_k(ks);
    __builtin_amdgcn_sched_barrier(0);
    f32x16 s;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.f;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
      s = mfma32(kf[ks % kKRing], qf[ks], s);
      if (ks + kKRing < 8) {
        __builtin_amdgcn_sched_barrier(0);
        read_k(ks + kKRing);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    // V of the first 16 keys: its reads return behind the softmax.
    u32x4 vf[2][4];
    auto read_v = [&](int j) __attribute__((always_inline)) {
#pragma unroll
      for (int db = 0; db < 4; ++db) {
        const uint8_t *vp = buf + vbase + j * 256 + db * 64;
        const u32x2 lo = lds_read_tr16(vp), hi = lds_read_tr16(vp + 8 * kVBlock);
        vf[j][db] = u32x4{lo[0], lo[1], hi[0], hi[1]};
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    read_v(0);
    if (hf == diag || left < 32) {
      const int lim = (hf == diag ? min(left - 1, r) : left - 1) - 4 * h;
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] = 8 * (i >> 2) + (i & 3) <= lim ? s[i] : -INFINITY;
    }
    float mx[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) mx[q] = fmaxf(fmaxf(s[4 * q], s[4 * q + 1]), fmaxf(s[4 * q + 2], s[4 * q + 3]));
    const float lmax = fmaxf(fmaxf(mx[0], mx[1]), fmaxf(mx[2], mx[3])) * sl2;
    if (__builtin_amdgcn_ballot_w64(lmax > m_run + kRescaleSlack)) {
      const f32x2_t both = halves(lmax);
      const float m_new = fmaxf(m_run, fmaxf(both[0], both[1]));
      const float alpha = __builtin_amdgcn_exp2f(m_run - (m_new == -INFINITY ? 0.f : m_new));
      l_run *= alpha;
      m_run = m_new;
#pragma unroll
      for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[db][i] *= alpha;
    }
    const float neg_m = m_run == -INFINITY ? 0.f : -m_run;
    u32x4 pb[2];
    float sum[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 16; i += 2) {
      const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i], sl2, neg_m));
      const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i + 1], sl2, neg_m));
      sum[i / 4] += p0 + p1;
      pb[i / 8][(i / 2) % 4] = pack_bf16x2(p0, p1);
    }
    l_run += (sum[0] + sum[1]) + (sum[2] + sum[3]);
    __builtin_amdgcn_sched_barrier(0);
    read_v(1);
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int db = 0; db < 4; ++db) o[db] = mfma32(vf[j][db], pb[j], o[db]);
    __builtin_amdgcn_sched_barrier(0);
  }
  for (int st = (nhalf + 1) / 2; st < nst; ++st) lds_barrier();

  // A V of the diagonal itself that is not finite has reached tokens that do not
  // see it.  Then (looked for only where O is not finite) the wave takes its
  // halves again, slowly.  A test inside the loop, or of V before it, costs
  // every launch 2 to 5 %; this one nothing that shows (T = 2048 against 10816
  // keys 390 -> 392 us, without history 64 -> 64).
  float zero = 0.f;
#pragma unroll
  for (int db = 0; db < 4; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) zero = __builtin_fmaf(o[db][i], 0.f, zero);
  if (__builtin_expect(__builtin_amdgcn_ballot_w64(zero != 0.f) != 0 && nhalf == diag + 1, 0)) {
    const int cur = sgpr(tiles.nseg - 1);
    bool bad = false;
#pragma clang loop unroll(disable)
    for (int i = 0; i < 8; ++i) {
      const int row = min(tok0 + 4 * i + (lane >> 4), T - 1);
      const u32x4 v = *(const u32x4 *)(a.v[cur] + (int64_t)row * a.v_stride[cur] + (int64_t)kvh * kD + (lane & 15) * 8);
#pragma unroll
      for (int c = 0; c < 4; ++c) bad |= (v[c] & 0x7f80u) == 0x7f80u || (v[c] & 0x7f800000u) == 0x7f800000u;
    }
    if (__builtin_amdgcn_ballot_w64(bad)) {
      m_run = -INFINITY;
      l_run = 0.f;
#pragma unroll
      for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[db][i] = 0.f;
#pragma clang loop unroll(disable)
      for (int hf = 0; hf < nhalf; ++hf)
        take_half(tiles.at(t_beg + hf / 2), 32 * (hf & 1), hf == diag);
    }
  }

  const f32x2_t lb2 = halves(l_run);
  const float L = lb2[0] + lb2[1];
  if (tok >= T) return;
  // Lane (r, h): dims 32 db + 8 q + 4 h + i of its token.
  if (nsplit == 1) {
    const float inv = L > 0.f ? 1.0f / L : 0.f;
    uint16_t *op = a.out + ((int64_t)tok * a.Hq + head) * kD + 4 * h;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        u32x2 v;
        v[0] = pack_bf16x2(o[db][4 * q] * inv, o[db][4 * q + 1] * inv);
        v[1] = pack_bf16x2(o[db][4 * q + 2] * inv, o[db][4 * q + 3] * inv);
        *(u32x2 *)(op + 32 * db + 8 * q) = v;
      }
  } else {
    // Partial state: [split][token][head] {m, l, O[128]} fp32.
    float *pp = a.partial + (((int64_t)split * T + tok) * a.Hq + head) * (kD + 2);
    if (h == 0) {
      pp[0] = m_run;
      pp[1] = L;
    }
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float *d = pp + 2 + 32 * db + 8 * q + 4 * h;  // 8-byte aligned rows
        *(f32x2_t *)d = f32x2_t{o[db][4 * q], o[db][4 * q + 1]};
        *(f32x2_t *)(d + 2) = f32x2_t{o[db][4 * q + 2], o[db][4 * q + 3]};
      }
  }
}

template <int G>
hipError_t launch_g(const GqaArgs &a, int nsplit, hipStream_t s) {
  auto k = gqa_prefill_kernel<G>;
  constexpr int lds = kSlots * kStageBytes;
  static const bool attr = hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, lds) ==
                           hipSuccess;
  if (!attr) return hipErrorInvalidValue;
  const int qt = 32 * (kMfmaWaves / G), nqb = (a.T + qt - 1) / qt;
  hipLaunchKernelGGL(k, dim3(nqb * a.Hkv * nsplit), dim3(kThreads), lds, s, a, nqb, nsplit);
  return hipGetLastError();
}

}  // namespace

int gqa_prefill_workgroups(int T, int Hq, int Hkv) {
  const int qt = 32 * (kMfmaWaves / (Hq / Hkv));
  return ((T + qt - 1) / qt) * Hkv;
}

hipError_t launch_gqa_prefill(const GqaArgs &a, int nsplit, hipStream_t s) {
  switch (a.Hq / a.Hkv) {
    case 1: return launch_g<1>(a, nsplit, s);
    case 2: return launch_g<2>(a, nsplit, s);
    case 4: return launch_g<4>(a, nsplit, s);
    case 8: return launch_g<8>(a, nsplit, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace moe
