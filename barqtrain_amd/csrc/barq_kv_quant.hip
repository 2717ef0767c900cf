// fp8 cold store of a page pool for MI355X (gfx950), behind the C ABI of include/barq_kv.h:
// blocks behind a row's residual window are quantised (barq_kv_compress) to OCP FP8 E4M3 codes
// with power-of-two (E8M0) scales -- keys per channel over the page's tokens, values per token
// over head_dim, KIVI's grouping -- and dequantised on the way out (barq_kv_gather_cold).
//
// Power-of-two scales make scaling exact, so a code depends only on its element and its group's
// largest finite magnitude, and a dequantised value is exactly code * 2^e before the final
// rounding to the pool's element type: the same numbers on every run and every device.
//
// The reference plans this path (IMPLEMENTATION_PLAN.md:106-129: quantized KV storage, a
// full-precision residual window, dequant-on-read) and has no implementation.

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <climits>
#include <type_traits>

#include "barq_kv.h"
#include <atomic>

#include "barq_kv_commit.h"
#include "barq_kv_fp8.h"
#include "barq_kv_internal.h"
#include "fastdiv.h"

namespace {

// s_waitcnt vmcnt(K), the other counters left alone (vmcnt bits 3:0, expcnt 6:4, lgkmcnt 11:8).
template <int K>
__device__ __forceinline__ void wait_vm() {
  static_assert(K >= 0 && K < 16, "vmcnt field");
  __builtin_amdgcn_s_waitcnt(K | (0x7 << 4) | (0xF << 8));
}

constexpr int kThreads = 256;
constexpr int kWave = 64;
constexpr int kWaves = kThreads / kWave;
constexpr int kMaxTokenHeads = 4096;  // page_size * kv_heads: a compress workgroup's value maxima
constexpr int kMaxChannels = 16384;   // kv_heads * head_dim: a compress workgroup's key exponents
constexpr int kUnroll = 4;            // vectors in flight per gather thread
constexpr int kGatherThreads = 256;   // a gather workgroup: 4 waves
constexpr int64_t kI32Max = 0x7fffffffLL;

__device__ __forceinline__ int checked_id(int id, int64_t n) { return (id >= 0 && (int64_t)id < n) ? id : -1; }

__device__ __forceinline__ int ceil_div_fd(int n, const FastDiv& d) {
  return n <= 0 ? 0 : (int)d.div((uint32_t)(n + (int)d.d - 1));
}

__device__ __forceinline__ int wave_incl_scan(int v) {
  const int lane = threadIdx.x & (kWave - 1);
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const int up = __shfl_up(v, o, kWave);
    if (lane >= o) v += up;
  }
  return v;
}

// Exclusive prefix sum over the workgroup; *total gets the sum.  Every thread must call it.
__device__ __forceinline__ int block_exclusive_scan(int v, int* lds, int* total) {
  const int wave = threadIdx.x / kWave;
  const int incl = wave_incl_scan(v);
  if ((threadIdx.x & (kWave - 1)) == kWave - 1) lds[wave] = incl;
  __syncthreads();
  int before = 0, all = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    const int t = lds[w];
    if (w < wave) before += t;
    all += t;
  }
  __syncthreads();
  *total = all;
  return before + incl - v;
}

using barq_fp8::codes_normal;
using barq_fp8::e4m3_decode;
using barq_fp8::e4m3_encode;
using barq_fp8::e4m3_encode4;
using barq_fp8::Elem;
using barq_fp8::fast_pair;
using barq_fp8::finite_abs;
using barq_fp8::group_exponent;
using barq_fp8::scale_fast;
using barq_fp8::spread_hi;
using barq_fp8::spread_lo;

struct ColdPtrs {
  uint8_t* codes[2];   // key, value
  uint8_t* key_scales;
  uint8_t* value_scales;
  int32_t* free_cold;
  int32_t* shares;     // references beyond the first, or null
  int64_t num_cold;
  int32_t window;
};

// ---------------------------------------------------------------------------------------------
// Compress: workgroup per row, any geometry (quant_blocks_kernel below takes the common ones).
// ---------------------------------------------------------------------------------------------

struct CompressArgs {
  barq_kv_pool p;
  ColdPtrs c;
  int32_t batch;
  int32_t ahead;       // tokens the rows are about to receive: quantise for lengths + ahead
  FastDiv div_page;
  FastDiv div_dim;     // head_dim
  FastDiv div_groups;  // kv_heads * head_dim / VE vectors per token
};

template <int BYTES>
struct RawC;
template <>
struct RawC<16> { using T = uint32_t __attribute__((ext_vector_type(4))); };
template <>
struct RawC<8> { using T = uint32_t __attribute__((ext_vector_type(2))); };
template <>
struct RawC<4> { using T = uint32_t; };
template <>
struct RawC<2> { using T = uint16_t; };
template <>
struct RawC<1> { using T = uint8_t; };

// VE elements of one token, as floats, from a page.
template <int KIND, int VE>
struct Lanes {
  using Bits = typename Elem<KIND>::Bits;
  using Raw = typename RawC<VE * (int)sizeof(Bits)>::T;
  union U {
    Raw v;
    Bits e[VE];
  };
  __device__ static void load(const Bits* src, float* out) {
    U u;
    u.v = *(const Raw*)src;
#pragma unroll
    for (int e = 0; e < VE; ++e) out[e] = Elem<KIND>::to_float(u.e[e]);
  }
};

template <int VE>
struct CodeVec {
  using Raw = typename RawC<VE>::T;
  union U {
    Raw v;
    uint8_t b[VE];
  };
};

// Quantise hot page hp into cold page cp (keys per channel, values per (token, head)), in vectors
// of VE elements along head_dim: maxima first (keys: a thread's channels over the page's tokens;
// values: a thread's (token, head) groups over head_dim), exponents to LDS, then codes.
template <int KIND, int VE>
__device__ void quantise_page(const CompressArgs& a, int hp, int cp, int8_t* s_kexp, int8_t* s_vexp) {
  using Bits = typename Elem<KIND>::Bits;
  const barq_kv_pool& p = a.p;
  const int P = (int)p.page_size, H = (int)p.kv_heads, D = (int)p.head_dim, C = H * D;
  const Bits* __restrict__ kp = (const Bits*)p.key_pages + (int64_t)hp * P * C;
  const Bits* __restrict__ vp = (const Bits*)p.value_pages + (int64_t)hp * P * C;
  const int groups = C / VE;
  for (int g = threadIdx.x; g < groups; g += kThreads) {
    float m[VE];
#pragma unroll
    for (int e = 0; e < VE; ++e) m[e] = 0.0f;
#pragma unroll 4
    for (int t = 0; t < P; ++t) {
      float x[VE];
      Lanes<KIND, VE>::load(kp + (int64_t)t * C + g * VE, x);
#pragma unroll
      for (int e = 0; e < VE; ++e) m[e] = fmaxf(m[e], finite_abs(x[e]));
    }
    typename CodeVec<VE>::U sc;
#pragma unroll
    for (int e = 0; e < VE; ++e) {
      const int ex = group_exponent(m[e]);
      s_kexp[g * VE + e] = (int8_t)ex;
      sc.b[e] = (uint8_t)(ex + 127);
    }
    *(typename CodeVec<VE>::Raw*)(a.c.key_scales + (int64_t)cp * C + g * VE) = sc.v;
  }
  const int dv = D / VE;
  for (int th = threadIdx.x; th < P * H; th += kThreads) {
    const Bits* src = vp + (int64_t)th * D;  // token t = th / H, head h = th % H: contiguous
    float m = 0.0f;
#pragma unroll 4
    for (int k = 0; k < dv; ++k) {
      float x[VE];
      Lanes<KIND, VE>::load(src + k * VE, x);
#pragma unroll
      for (int e = 0; e < VE; ++e) m = fmaxf(m, finite_abs(x[e]));
    }
    const int ex = group_exponent(m);
    s_vexp[th] = (int8_t)ex;
    a.c.value_scales[(int64_t)cp * P * H + th] = (uint8_t)(ex + 127);
  }
  __syncthreads();
  uint8_t* __restrict__ kc = a.c.codes[0] + (int64_t)cp * P * C;
  uint8_t* __restrict__ vc = a.c.codes[1] + (int64_t)cp * P * C;
#pragma unroll 2
  for (int v = threadIdx.x; v < P * groups; v += kThreads) {
    const int t = (int)a.div_groups.div((uint32_t)v);
    const int g = v - t * groups;
    const int ch = g * VE;
    const int th = t * H + (int)a.div_dim.div((uint32_t)ch);
    const int64_t at = (int64_t)t * C + ch;
    float xk[VE], xv[VE];
    Lanes<KIND, VE>::load(kp + at, xk);
    Lanes<KIND, VE>::load(vp + at, xv);
    const int ve = s_vexp[th];
    typename CodeVec<VE>::U ck, cv;
    if constexpr (VE % 4 == 0) {
      uint32_t wk[VE / 4], wv[VE / 4];
#pragma unroll
      for (int q = 0; q < VE / 4; ++q) {
        const int e = 4 * q;
        wk[q] = e4m3_encode4(ldexpf(xk[e], -(int)s_kexp[ch + e]), ldexpf(xk[e + 1], -(int)s_kexp[ch + e + 1]),
                             ldexpf(xk[e + 2], -(int)s_kexp[ch + e + 2]), ldexpf(xk[e + 3], -(int)s_kexp[ch + e + 3]));
        wv[q] = e4m3_encode4(ldexpf(xv[e], -ve), ldexpf(xv[e + 1], -ve), ldexpf(xv[e + 2], -ve), ldexpf(xv[e + 3], -ve));
      }
      __builtin_memcpy(ck.b, wk, VE);
      __builtin_memcpy(cv.b, wv, VE);
    } else {
#pragma unroll
      for (int e = 0; e < VE; ++e) {
        ck.b[e] = (uint8_t)e4m3_encode(ldexpf(xk[e], -(int)s_kexp[ch + e]));
        cv.b[e] = (uint8_t)e4m3_encode(ldexpf(xv[e], -ve));
      }
    }
    *(typename CodeVec<VE>::Raw*)(kc + at) = ck.v;
    *(typename CodeVec<VE>::Raw*)(vc + at) = cv.v;
  }
}

template <int KIND, int VE>
__global__ void __launch_bounds__(kThreads) compress_kernel(const CompressArgs a) {
  __shared__ int lds_scan[kWaves];
  __shared__ int s_blocks[kThreads];
  __shared__ int s_cold;
  __shared__ int8_t s_vexp[kMaxTokenHeads];
  __shared__ int8_t s_kexp[kMaxChannels];
  const barq_kv_pool& p = a.p;
  const int r = blockIdx.x;
  const int mb = (int)p.max_blocks;
  const int len = p.seq_lens[r] + a.ahead;
  const int old_len = len - a.c.window;
  const int jmax = min(old_len > 0 ? (int)a.div_page.div((uint32_t)old_len) : 0,
                       min(ceil_div_fd(max(p.high_water[r], len), a.div_page), mb));
  int32_t* row = p.block_table + (int64_t)r * mb;
  int err = 0;
  for (int j0 = 0; j0 < jmax; j0 += kThreads) {
    const int j = j0 + (int)threadIdx.x;
    int hot = 0;
    if (j < jmax) {
      const int page = checked_id(row[j], p.num_pages);
      hot = page >= 0 && (!p.page_shares || p.page_shares[page] == 0);
    }
    int count = 0;
    const int k = block_exclusive_scan(hot, lds_scan, &count);
    if (hot) s_blocks[k] = j;
    __syncthreads();
    for (int q = 0; q < count; ++q) {
      const int jb = s_blocks[q];
      if (threadIdx.x == 0) {
        int cp = -1;
        const int before = atomicSub(&p.ctrl[BARQ_KV_CTRL_COLD_TOP], 1);
        if (before <= 0 || (int64_t)before > a.c.num_cold) {
          atomicAdd(&p.ctrl[BARQ_KV_CTRL_COLD_TOP], 1);
          err |= before <= 0 ? BARQ_KV_ERRBIT_POOL_EXHAUSTED : BARQ_KV_ERRBIT_BAD_INDEX;
        } else {
          cp = checked_id(a.c.free_cold[before - 1], a.c.num_cold);
          if (cp < 0) err |= BARQ_KV_ERRBIT_BAD_INDEX;
        }
        s_cold = cp;
      }
      __syncthreads();
      const int cp = s_cold;
      const int hp = row[jb];
      if (cp >= 0) {  // uniform
        quantise_page<KIND, VE>(a, hp, cp, s_kexp, s_vexp);
        __syncthreads();  // every thread has read the hot page before it is released
        if (threadIdx.x == 0) {
          row[jb] = BARQ_KV_COLD_ENTRY(cp);
          const int slot = atomicAdd(&p.ctrl[BARQ_KV_CTRL_FREE_TOP], 1);
          if (slot < p.num_pages) p.free_pages[slot] = hp;
          else err |= BARQ_KV_ERRBIT_BAD_INDEX;
        }
      }
      __syncthreads();
    }
  }
  if (err) atomicOr(&p.ctrl[BARQ_KV_CTRL_ERRORS], err);
}

// ---------------------------------------------------------------------------------------------
// Blocks quantised by a wave to each (K or V, head) of a block: the compress of pools whose pages
// divide into waves (quant_blocks_vectors below), and an append of any number of tokens that
// quantises what passes the residual window straight from the input.
//
// A unit = one head of a block's K (or V), NV vectors of 16 bytes per lane: lane l holds column
// l % vd (vd = vectors per head row) of tokens l / vd + i * 64 / vd.  Key maxima over the page's
// tokens and value maxima over head_dim then cross lanes of one wave only -- no LDS, no barrier --
// and units are independent, so a workgroup of up to 16 waves takes a block in one round trip of
// loads.  The compress also takes heads whose page is more than eight waves' vectors, a unit then
// being some of K's columns or some of V's tokens (split), and less than one wave's, a unit then being
// several heads (packed).  Such pools' page of 16 rows, launch and events included, against the kernel
// of any geometry: 2 x 128 at page 64 22.4 -> 12.0 us, 1 x 256 at page 32 18.0 -> 11.6, 1 x 128 at page
// 128 30.6 -> 12.0; 8 x 64 at page 4 10.2 -> 8.9, 16 x 64 at page 2 10.2 -> 8.7.
//
// Quantised blocks lead every row (the attention kernels and a crop count on it), also when the cold
// store runs out.  So in compress_blocks_kernel each row has one workgroup, which takes the pages of
// the row's hot blocks with one atomic and quantises as many as it got, the first ones.  Where the
// store cannot run out -- the append's plan below has counted, or the caller has (spread) --
// quant_blocks_kernel spreads a row's blocks over workgroups.  16 rows of the 8 x 128 bf16 shape, one
// page a row 10.7 us in order and 10.8 spread (launch and events included), four pages 20.7 and 11.4;
// one workgroup of 256 threads a row, its blocks one after the other through LDS, took 14.6 and 35.9.
//
// Tiles (row, i): i < nnew is the i-th block that receives new tokens -- a block the plan has
// just mapped to a cold page is quantised from the input, one that stays behind the frontier is
// copied to its hot page, one that was hot before (the row's partial block, blocks a crop
// re-opened) is quantised from its page and the input; i >= nnew are the row's older hot blocks.
// Blocks that were hot take their cold page and return their hot page through atomics on the stack
// tops, which no other part of the launch moves the other way.
//
// Bound: HBM (the input read once, codes and scales written once), then the round trips of a
// workgroup's only block.  A 16 x 1000-token prompt of the 8 x 128 bf16 shape: 25.6 us for 95 MB
// after a 7.1 us plan, against 16 chunks of an append and a compress each, 9.2 + 33 us.
// ---------------------------------------------------------------------------------------------

// Tiles per row that look for older hot blocks: an append of 64 tokens pushes four out of the window
// (page size 16).
constexpr int kOldTiles = 4;

struct QuantArgs {
  barq_kv_pool p;
  ColdPtrs c;
  const char* in[2];      // key, value states (append)
  int64_t isb, ish, ist;  // input strides, elements
  int32_t tokens;         // appended tokens, already counted in seq_lens (0: compress only)
  int32_t ahead;          // compress: tokens the rows are about to receive
  int32_t nnew;           // tiles per row of blocks that receive tokens
  int32_t vd_log2;        // vectors per head row
  int32_t mode_log2;      // split units: units per head; packed units: vectors of a head's page
  FastDiv div_page;
  FastDiv div_tiles;      // nnew + kOldTiles
};

// The lane, unknown to the optimiser: a unit's per-vector offsets are computed where they are used
// and not held across the loop over units (16 registers a vector).
__device__ __forceinline__ int opaque_lane() {
  int lane = threadIdx.x & (kWave - 1);
  asm volatile("" : "+v"(lane));
  return lane;
}

enum : int { kWholeUnit = 0, kSplitUnit = 1, kPackedUnit = 2 };

// Where a lane's vectors of a unit lie: columns from col of tokens t0 + i * step.
struct UnitLane {
  int col, t0, step;
  bool first;         // of the lanes that share a column
  int vectors;        // of a row in the unit
  int reach;          // lanes that share a column are less than this apart
};

// piece: which of a head's units a split one is.
template <int KIND, int NV, int MODE>
__device__ __forceinline__ UnitLane unit_lane(const QuantArgs& a, int kv, int piece) {
  constexpr int VE = 16 / (int)sizeof(typename Elem<KIND>::Bits);
  int lane = opaque_lane();
  UnitLane l;
  l.reach = MODE == kPackedUnit ? 1 << a.mode_log2 : kWave;
  if constexpr (MODE == kPackedUnit) lane &= l.reach - 1;
  const int vl = MODE == kSplitUnit && kv == 0 ? a.vd_log2 - a.mode_log2 : a.vd_log2;
  l.vectors = 1 << vl;
  l.col = (lane & (l.vectors - 1)) * VE;
  l.t0 = lane >> vl;
  l.step = kWave >> vl;
  l.first = l.t0 == 0;
  if constexpr (MODE == kSplitUnit) {
    if (kv == 0) l.col += (piece << vl) * VE;
    else l.t0 += piece * NV * l.step;
  }
  return l;
}

// Loads unit (kv, h) of the block whose positions start at s0: from hot page hp (if any), and
// positions from len on -- the launch's tokens -- from the input.  Lane offsets fit 32 bits.
template <int KIND, int NV, int MODE = kWholeUnit>
__device__ __forceinline__ void load_unit(const QuantArgs& a, int b, int kv, int h, int hp, int s0, int len,
                                          typename RawC<16>::T (&x)[NV], int piece = 0) {
  using Bits = typename Elem<KIND>::Bits;
  using V = typename RawC<16>::T;
  const barq_kv_pool& p = a.p;
  const UnitLane l = unit_lane<KIND, NV, MODE>(a, kv, piece);
  const int col = l.col, t0 = l.t0, step = l.step;
  const int HD = (int)(p.kv_heads * p.head_dim), P = (int)p.page_size;
  const Bits* in = (const Bits*)a.in[kv] + ((int64_t)b * a.isb + (int64_t)h * a.ish + (int64_t)(s0 - len) * a.ist);
  const uint32_t ist = (uint32_t)a.ist;
  if (hp < 0) {  // uniform: only new tokens
#pragma unroll
    for (int i = 0; i < NV; ++i)
      x[i] = __builtin_nontemporal_load((const V*)(in + ((uint32_t)(t0 + i * step) * ist + (uint32_t)col)));
    return;
  }
  const Bits* page = (const Bits*)(kv ? p.value_pages : p.key_pages) + ((int64_t)hp * P * HD + h * (int)p.head_dim);
#pragma unroll
  for (int i = 0; i < NV; ++i) x[i] = __builtin_nontemporal_load((const V*)(page + (uint32_t)((t0 + i * step) * HD + col)));
  if (s0 + P > len) {  // uniform: the block's last positions are new
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int t = t0 + i * step;
      const V y = *(const V*)(in + ((uint32_t)max(t, len - s0) * ist + (uint32_t)col));
      x[i] = s0 + t >= len ? y : x[i];
    }
  }
}

// Magnitudes as bit patterns, whose order is the values': a word holds two of a two-byte type or one
// fp32.
template <int KIND>
struct Mag {
  static constexpr bool kPacked = KIND != BARQ_KV_FP32;
  static constexpr uint32_t kMask = kPacked ? 0x7FFF7FFFu : 0x7FFFFFFFu;
  static constexpr uint32_t kInf = KIND == BARQ_KV_BF16 ? 0x7F80u : KIND == BARQ_KV_FP16 ? 0x7C00u : 0x7F800000u;
  __device__ static uint32_t max2(uint32_t a, uint32_t b) {
    if constexpr (kPacked) {
      using P2 = uint16_t __attribute__((ext_vector_type(2)));
      return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(P2, a), __builtin_bit_cast(P2, b)));
    } else {
      return max(a, b);
    }
  }
  __device__ static bool any_nonfinite(uint32_t m) {
    if constexpr (kPacked) return (m & 0xFFFFu) >= kInf || (m >> 16) >= kInf;
    return m >= kInf;
  }
  // the word's magnitudes, infinities and NaN as 0
  __device__ static uint32_t finite(uint32_t w) {
    const uint32_t m = w & kMask;
    if constexpr (kPacked) return ((m & 0xFFFFu) >= kInf ? 0u : m & 0xFFFFu) | ((m >> 16) >= kInf ? 0u : m & 0xFFFF0000u);
    return m >= kInf ? 0u : m;
  }
  // element e of word w as a float (e: 0 low, 1 high half)
  __device__ static float value(uint32_t w, int e) {
    if constexpr (KIND == BARQ_KV_BF16) return __uint_as_float(e ? w & 0xFFFF0000u : w << 16);
    if constexpr (KIND == BARQ_KV_FP16) return Elem<KIND>::to_float((uint16_t)(e ? w >> 16 : w));
    return __uint_as_float(w);
  }
};

// Codes and scales of unit (kv, h) into cold page cp.  The maxima run on magnitude bits (two
// elements an operation); the codes are e4m3_encode of x * 2^-e through the hardware conversion
// (e4m3_encode4's domain), infinities and NaN -- looked for only in units that hold one -- given
// the NaN code with their sign.  Each vector's code and scale words also go to emit(token, column, ...).
struct NoEmit {
  template <typename... A>
  __device__ void operator()(A&&...) const {}
};

template <int KIND, int NV, int MODE = kWholeUnit, typename Emit = NoEmit>
__device__ __forceinline__ void quantise_unit(const QuantArgs& a, int kv, int h, int cp,
                                              const typename RawC<16>::T (&x)[NV], const Emit& emit = Emit(),
                                              int piece = 0) {
  using M = Mag<KIND>;
  constexpr int VE = M::kPacked ? 8 : 4;  // elements of a vector; EW of a word
  constexpr int EW = VE / 4;
  const barq_kv_pool& p = a.p;
  const UnitLane l = unit_lane<KIND, NV, MODE>(a, kv, piece);
  const int col = l.col, t0 = l.t0, step = l.step;
  const int P = (int)p.page_size, H = (int)p.kv_heads, D = (int)p.head_dim;
  float inv[VE];      // keys: 2^-e of the columns' scale exponents e in [-127, 120] (products are exact)
  uint32_t top[NV];   // values: the vectors' token maxima
  uint32_t scales[VE / 4];  // keys: the columns' scale bytes
  bool special;
  if (kv == 0) {
    uint32_t m[4] = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < NV; ++i)
#pragma unroll
      for (int w = 0; w < 4; ++w) m[w] = M::max2(m[w], x[i][w] & M::kMask);
    special = __builtin_amdgcn_ballot_w64(M::any_nonfinite(M::max2(M::max2(m[0], m[1]), M::max2(m[2], m[3])))) != 0;
    if (special) {  // uniform
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        m[w] = 0;
#pragma unroll
        for (int i = 0; i < NV; ++i) m[w] = M::max2(m[w], M::finite(x[i][w]));
      }
    }
    for (int o = l.vectors; o < l.reach; o <<= 1) {
#pragma unroll
      for (int w = 0; w < 4; ++w) m[w] = M::max2(m[w], (uint32_t)__shfl_xor((int)m[w], o, kWave));
    }
    typename CodeVec<VE>::U sc;
#pragma unroll
    for (int e = 0; e < VE; ++e) {
      const int ex = group_exponent(M::value(m[e / EW], e % EW));
      inv[e] = __uint_as_float((uint32_t)(127 - ex) << 23);
      sc.b[e] = (uint8_t)(ex + 127);
    }
    if (l.first) *(typename CodeVec<VE>::Raw*)(a.c.key_scales + ((int64_t)cp * H + h) * D + col) = sc.v;
    __builtin_memcpy(scales, sc.b, VE);
  } else {
    uint32_t all = 0;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      top[i] = M::max2(M::max2(x[i][0] & M::kMask, x[i][1] & M::kMask), M::max2(x[i][2] & M::kMask, x[i][3] & M::kMask));
      all = M::max2(all, top[i]);
    }
    special = __builtin_amdgcn_ballot_w64(M::any_nonfinite(all)) != 0;
    if (special) {  // uniform
#pragma unroll
      for (int i = 0; i < NV; ++i)
        top[i] = M::max2(M::max2(M::finite(x[i][0]), M::finite(x[i][1])), M::max2(M::finite(x[i][2]), M::finite(x[i][3])));
    }
    uint8_t* __restrict__ vscales = a.c.value_scales + ((int64_t)cp * P * H + h);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      if constexpr (M::kPacked) top[i] = max(top[i] & 0xFFFFu, top[i] >> 16);
      for (int o = 1; o < l.vectors; o <<= 1) top[i] = max(top[i], (uint32_t)__shfl_xor((int)top[i], o, kWave));
      const int ex = group_exponent(M::value(top[i], 0));
      top[i] = (uint32_t)(127 - ex) << 23;  // 2^-e
      if (col == 0) vscales[(uint32_t)((t0 + i * step) * H)] = (uint8_t)(ex + 127);
    }
  }
  uint8_t* __restrict__ codes = a.c.codes[kv] + ((int64_t)cp * P * H + h) * D;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    __builtin_amdgcn_sched_barrier(0);  // one vector's floats at a time
    typename CodeVec<VE>::U out;
    uint32_t word[VE / 4];
#pragma unroll
    for (int q = 0; q < VE / 4; ++q) {
      float f[4];
#pragma unroll
      for (int k = 0; k < 4; ++k)
        f[k] = M::value(x[i][(4 * q + k) / EW], (4 * q + k) % EW) * (kv == 0 ? inv[4 * q + k] : __uint_as_float(top[i]));
      uint32_t nan = 0;
      if (special) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          if (fabsf(f[k]) <= 3.402823466e38f) continue;
          nan |= (((__float_as_uint(f[k]) >> 24) & 0x80u) | 0x7Fu) << (8 * k);
          f[k] = 0.0f;
        }
      }
      const int lo = __builtin_amdgcn_cvt_pk_fp8_f32(f[0], f[1], 0, false);
      word[q] = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(f[2], f[3], lo, true) | nan;
    }
    __builtin_memcpy(out.b, word, VE);
    *(typename CodeVec<VE>::Raw*)(codes + (uint32_t)((t0 + i * step) * H * D + col)) = out.v;
    emit(t0 + i * step, col, word, scales, 254u - (top[i] >> 23));
  }
}

template <int KIND, int NV>
__global__ void __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(NV <= 4 ? 8 : 4))) quant_blocks_kernel(const QuantArgs a) {
  using V = typename RawC<16>::T;
  using Bits = typename Elem<KIND>::Bits;
  __shared__ int s_cold;
  const barq_kv_pool& p = a.p;
  if (a.tokens > 0 && p.ctrl[BARQ_KV_CTRL_APPEND_OK] == 0) return;  // the append was abandoned
  const int b = (int)a.div_tiles.div(blockIdx.x);
  const int i = (int)blockIdx.x - b * (int)a.div_tiles.d;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int nwaves = (int)blockDim.x / kWave;
  const int P = (int)p.page_size, H = (int)p.kv_heads, D = (int)p.head_dim, mb = (int)p.max_blocks;
  const int end = p.seq_lens[b] + a.ahead;  // the row's length after the append (or ahead of it)
  const int len = end - a.tokens;           // positions from here on are the launch's tokens
  const int hw = p.high_water[b];
  const int frontier = min(end > a.c.window ? (int)a.div_page.div((uint32_t)(end - a.c.window)) : 0, mb);
  int32_t* row = p.block_table + (int64_t)b * mb;
  int err = 0;

  const bool new_tile = i < a.nnew;
  // Older blocks, wholly below len (compress: below the high-water mark), as far as the frontier;
  // this tile's every kOldTiles-th of them, 64 entries (one per lane) at a time.
  const int limit = a.tokens > 0 ? (int)a.div_page.div((uint32_t)len)
                                 : min(ceil_div_fd(max(hw, end), a.div_page), mb);
  int next = new_tile ? 0 : min(frontier, limit) - 1 - (i - a.nnew);
  int first = 0, found = -1;  // the lane's hot page, of block first - lane * kOldTiles
  uint64_t hot = 0;           // lanes whose block is still to do (the same bits in every wave)
  for (;;) {
    int j, hp = -1, cp = -1;
    bool moves = false;  // a hot block that leaves the window
    if (new_tile) {
      j = (int)a.div_page.div((uint32_t)len) + i;
      if (j * P >= end || j >= mb) break;
      const int entry = row[j];
      if (entry <= -2) {
        if (j * P >= len) cp = checked_id(-2 - entry, a.c.num_cold);
        if (cp < 0) err |= BARQ_KV_ERRBIT_BAD_INDEX;
      } else {
        hp = checked_id(entry, p.num_pages);
        moves = hp >= 0 && j < frontier && (!p.page_shares || p.page_shares[hp] == 0);
      }
    } else {
      while (hot == 0 && next >= 0) {
        const int jl = next - lane * kOldTiles;
        found = jl >= 0 ? checked_id(row[jl], p.num_pages) : -1;
        if (found >= 0 && p.page_shares && p.page_shares[found] != 0) found = -1;
        hot = __builtin_amdgcn_ballot_w64(found >= 0);
        first = next;
        next -= kOldTiles * kWave;
      }
      if (hot == 0) break;
      const int l = __builtin_ctzll(hot);
      hot &= hot - 1;
      j = first - l * kOldTiles;
      hp = __builtin_amdgcn_readlane(found, l);
      moves = true;
    }
    if (moves) {  // uniform
      if (threadIdx.x == 0) {
        const int before = atomicSub(&p.ctrl[BARQ_KV_CTRL_COLD_TOP], 1);
        int c = -1;
        if (before <= 0 || (int64_t)before > a.c.num_cold) {
          atomicAdd(&p.ctrl[BARQ_KV_CTRL_COLD_TOP], 1);
          err |= before <= 0 ? BARQ_KV_ERRBIT_POOL_EXHAUSTED : BARQ_KV_ERRBIT_BAD_INDEX;
        } else {
          c = checked_id(a.c.free_cold[before - 1], a.c.num_cold);
          if (c < 0) err |= BARQ_KV_ERRBIT_BAD_INDEX;
        }
        s_cold = c;
      }
      __syncthreads();
      cp = s_cold;  // (-1, the block stays hot: not the pages that the plan or the caller counted)
    }
#pragma unroll 1
    for (int u = wave; u < 2 * H; u += nwaves) {  // a wave's units: heads of K, then of V
      const int kv = u >= H ? 1 : 0, h = u - kv * H;
      V x[NV];
      if (cp >= 0) {
        load_unit<KIND, NV>(a, b, kv, h, hp, j * P, len, x);
        quantise_unit<KIND, NV>(a, kv, h, cp, x);
      } else if (hp >= 0 && new_tile) {  // the block's new tokens into its hot page
        const int lane = opaque_lane();
        const int lo = max(len - j * P, 0), hi = min(end - j * P, P);
        const int col = (lane & ((1 << a.vd_log2) - 1)) * (16 / (int)sizeof(Bits));
        const Bits* in = (const Bits*)a.in[kv] + ((int64_t)b * a.isb + (int64_t)h * a.ish + (int64_t)(j * P - len) * a.ist);
        Bits* page = (Bits*)(kv ? p.value_pages : p.key_pages) + ((int64_t)hp * P * H + h) * D;
#pragma unroll
        for (int k = 0; k < NV; ++k) {
          const int t = (lane >> a.vd_log2) + k * (kWave >> a.vd_log2);
          if (t >= lo && t < hi)
            x[k] = __builtin_nontemporal_load((const V*)(in + ((uint32_t)t * (uint32_t)a.ist + (uint32_t)col)));
        }
#pragma unroll
        for (int k = 0; k < NV; ++k) {
          const int t = (lane >> a.vd_log2) + k * (kWave >> a.vd_log2);
          if (t >= lo && t < hi) *(V*)(page + (uint32_t)(t * H * D + col)) = x[k];
        }
      }
    }
    if (moves) {
      __syncthreads();  // every wave has read the hot page, and s_cold, before they change
      if (threadIdx.x == 0 && cp >= 0) {
        row[j] = BARQ_KV_COLD_ENTRY(cp);
        const int slot = atomicAdd(&p.ctrl[BARQ_KV_CTRL_FREE_TOP], 1);
        if (slot < p.num_pages) p.free_pages[slot] = hp;
        else err |= BARQ_KV_ERRBIT_BAD_INDEX;
      }
    }
    if (new_tile) break;
  }
  if (err) atomicOr(&p.ctrl[BARQ_KV_CTRL_ERRORS], err);
}

// Compress of one row, a pass of kScan entries a lane at a time (every wave scans for itself); the waves
// of rows of more than two passes first share those out to find the ones that hold hot blocks (16 rows of
// 2040 blocks of the 2 x 64 shape, one page each: 11.7 -> 9.8 us, launch and events included).
constexpr int kScan = 4;

template <int KIND, int NV, int MODE = kWholeUnit>
__global__ void __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(4))) compress_blocks_kernel(const QuantArgs a) {
  using V = typename RawC<16>::T;
  __shared__ int s_top, s_avail;
  __shared__ unsigned long long s_look;
  const barq_kv_pool& p = a.p;
  const int b = (int)blockIdx.x;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int nwaves = (int)blockDim.x / kWave;
  const int P = (int)p.page_size, H = (int)p.kv_heads, mb = (int)p.max_blocks;
  const int len = p.seq_lens[b] + a.ahead;
  const int frontier = min(len > a.c.window ? (int)a.div_page.div((uint32_t)(len - a.c.window)) : 0,
                           min(ceil_div_fd(max(p.high_water[b], len), a.div_page), mb));
  int32_t* row = p.block_table + (int64_t)b * mb;
  const int passes = (frontier + kScan * kWave - 1) / (kScan * kWave);
  uint64_t look = ~0ull;  // passes to look at, of the first 64
  if (passes > 2) {       // uniform
    if (threadIdx.x == 0) s_look = 0;
    __syncthreads();
    for (int t = wave; t < min(passes, 64); t += nwaves) {
      int top = -1;
#pragma unroll
      for (int k = 0; k < kScan; ++k) top = max(top, row[min((t * kScan + k) * kWave + lane, frontier - 1)]);
      if (__builtin_amdgcn_ballot_w64(top >= 0) != 0 && lane == 0) atomicOr(&s_look, 1ull << t);
    }
    __syncthreads();
    look = s_look;
  }
  int err = 0;
  for (int t = 0; t < passes; ++t) {
    if (t < 64 && ((look >> t) & 1) == 0) continue;
    const int j0 = t * kScan * kWave;
    int found[kScan];      // the lane's hot page, of block j0 + kWave * k + lane
    uint64_t hot[kScan];   // lanes that have one
    int count = 0;
#pragma unroll
    for (int k = 0; k < kScan; ++k) {
      const int j = j0 + kWave * k + lane;
      found[k] = j < frontier ? row[j] : -1;
    }
#pragma unroll
    for (int k = 0; k < kScan; ++k) {
      found[k] = checked_id(found[k], p.num_pages);
      if (found[k] >= 0 && p.page_shares && p.page_shares[found[k]] != 0) found[k] = -1;
      hot[k] = __builtin_amdgcn_ballot_w64(found[k] >= 0);
      count += __builtin_popcountll(hot[k]);
    }
    if (count == 0) continue;  // uniform
    if (threadIdx.x == 0) {
      const int before = atomicSub(&p.ctrl[BARQ_KV_CTRL_COLD_TOP], count);
      int avail = 0;
      if ((int64_t)before > a.c.num_cold) err |= BARQ_KV_ERRBIT_BAD_INDEX;
      else avail = min(max(before, 0), count);
      if (avail < count) {
        atomicAdd(&p.ctrl[BARQ_KV_CTRL_COLD_TOP], count - avail);
        err |= err ? 0 : BARQ_KV_ERRBIT_POOL_EXHAUSTED;
      }
      s_top = before;
      s_avail = avail;
    }
    __syncthreads();
    const int avail = s_avail;
    const int32_t* cold = a.c.free_cold + (s_top - 1);  // the q-th hot block takes cold[-q]
    // Units (block, heads of K, then of V) dealt to the waves in turn.
    const int packed = MODE == kPackedUnit ? kWave >> a.mode_log2 : 1;  // heads of a unit
    const int units = MODE == kSplitUnit ? H << a.mode_log2 : MODE == kPackedUnit ? (H + packed - 1) / packed : H;
    int q = 0, u = wave;
#pragma unroll
    for (int k = 0; k < kScan; ++k) {
      uint64_t left = hot[k];
      for (; left != 0 && q < avail; ++q) {
        const int l = __builtin_ctzll(left);
        left &= left - 1;
        if (u < 2 * units) {
          const int hp = __builtin_amdgcn_readlane(found[k], l);
          const int cp = checked_id(cold[-q], a.c.num_cold);
#pragma unroll 1
          for (; u < 2 * units; u += nwaves) {
            const int kv = u >= units ? 1 : 0, n = u - kv * units;
            const int piece = MODE == kSplitUnit ? n & ((1 << a.mode_log2) - 1) : 0;
            const int h = MODE == kSplitUnit    ? n >> a.mode_log2
                          : MODE == kPackedUnit ? min(n * packed + (lane >> a.mode_log2), H - 1)  // past the last: it again
                                                : n;
            V x[NV];
            load_unit<KIND, NV, MODE>(a, b, kv, h, hp, 0, P, x, piece);
            if (cp >= 0) quantise_unit<KIND, NV, MODE>(a, kv, h, cp, x, NoEmit(), piece);
          }
        }
        u -= 2 * units;
      }
    }
    __syncthreads();  // every wave has read its hot pages, s_top and s_avail before they change
    if (wave == 0) {
      int first = 0;  // rank of the 64 entries' first hot block
#pragma unroll
      for (int k = 0; k < kScan; ++k) {
        const int rank = first + __builtin_popcountll(hot[k] & ((1ull << lane) - 1));
        first += __builtin_popcountll(hot[k]);
        const int cp = found[k] >= 0 && rank < avail ? checked_id(cold[-rank], a.c.num_cold) : -1;
        if (found[k] >= 0 && rank < avail && cp < 0) err |= BARQ_KV_ERRBIT_BAD_INDEX;
        const uint64_t done = __builtin_amdgcn_ballot_w64(cp >= 0);
        if (done == 0) continue;  // uniform
        int slot = 0;
        if (lane == 0) slot = atomicAdd(&p.ctrl[BARQ_KV_CTRL_FREE_TOP], __builtin_popcountll(done));
        slot = __builtin_amdgcn_readfirstlane(slot) + __builtin_popcountll(done & ((1ull << lane) - 1));
        if (cp >= 0) {
          row[j0 + kWave * k + lane] = BARQ_KV_COLD_ENTRY(cp);
          if (slot < p.num_pages) p.free_pages[slot] = found[k];
          else err |= BARQ_KV_ERRBIT_BAD_INDEX;
        }
      }
    }
    if (avail < count) break;  // uniform: what follows stays hot too
  }
  if (err) atomicOr(&p.ctrl[BARQ_KV_CTRL_ERRORS], err);
}

// Commit of such an append, before its blocks are written: one workgroup maps every row's new
// blocks -- those wholly before the window at the row's new end to cold pages, the rest to hot
// pages, each ranked in (row, block) order on its stack -- and advances the rows.  If a row passes
// its capacity or a stack holds too few pages -- the cold one also those of the rows' hot blocks that
// leave the window -- nothing changes but the error bits, and ctrl[BARQ_KV_CTRL_APPEND_OK] = 0 tells
// the launch that follows.
struct AppendPlanArgs {
  barq_kv_pool p;
  ColdPtrs c;
  int32_t batch;
  int32_t tokens;
  FastDiv div_page;
};

constexpr int kPlanThreads = 1024;

__global__ void __launch_bounds__(kPlanThreads) append_plan_kernel(const AppendPlanArgs a) {
  __shared__ int s_scan[2][kPlanThreads / kWave];
  __shared__ int s_incl[2][kPlanThreads];  // rank ends of the chunk's rows: cold, hot
  __shared__ int s_first[2][kPlanThreads];
  __shared__ int s_bad, s_old;
  const barq_kv_pool& p = a.p;
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1), wave = tid / kWave;
  const int mb = (int)p.max_blocks;
  const int top = p.ctrl[BARQ_KV_CTRL_FREE_TOP];
  const int ctop = p.ctrl[BARQ_KV_CTRL_COLD_TOP];
  if (tid == 0) s_bad = s_old = 0;
  __syncthreads();
  // pass 0 counts, pass 1 maps
  for (int pass = 0; pass < 2; ++pass) {
    int used[2] = {0, 0};
    int err = 0;
    for (int r0 = 0; r0 < a.batch; r0 += kPlanThreads) {
      const int r = r0 + tid;
      int n[2] = {0, 0}, first[2] = {0, 0};
      int len = 0, hw = 0;
      if (r < a.batch) {
        len = p.seq_lens[r];
        hw = p.high_water[r];
        const int f = ceil_div_fd(hw, a.div_page);
        const int full = ceil_div_fd(len + a.tokens, a.div_page);
        if (full > mb) err |= BARQ_KV_ERRBIT_CAPACITY;
        const int end = min(full, mb);
        const int behind = len + a.tokens - a.c.window;
        const int frontier = min(behind > 0 ? (int)a.div_page.div((uint32_t)behind) : 0, end);
        first[0] = f;
        n[0] = max(frontier - f, 0);
        first[1] = max(f, frontier);
        n[1] = max(end - first[1], 0);
      }
      int total[2];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int incl = wave_incl_scan(n[k]);
        if (lane == kWave - 1) s_scan[k][wave] = incl;
        __syncthreads();
        int before = 0, all = 0;
        for (int w = 0; w < kPlanThreads / kWave; ++w) {
          const int t = s_scan[k][w];
          if (w < wave) before += t;
          all += t;
        }
        s_incl[k][tid] = before + incl;
        s_first[k][tid] = first[k];
        total[k] = all;
      }
      __syncthreads();
      if (pass == 1) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          for (int q = tid; q < total[k]; q += kPlanThreads) {
            int lo = 0, hi = kPlanThreads - 1;
            while (lo < hi) {  // the first row whose rank end passes q
              const int mid = (lo + hi) >> 1;
              if (s_incl[k][mid] > q) hi = mid;
              else lo = mid + 1;
            }
            const int excl = lo > 0 ? s_incl[k][lo - 1] : 0;
            const int idx = (k == 0 ? ctop : top) - 1 - (used[k] + q);  // within the stack: pass 0 checked
            const int id = k == 0 ? checked_id(a.c.free_cold[idx], a.c.num_cold)
                                  : checked_id(p.free_pages[idx], p.num_pages);
            if (id < 0) err |= BARQ_KV_ERRBIT_BAD_INDEX;
            p.block_table[(int64_t)(r0 + lo) * mb + s_first[k][lo] + (q - excl)] =
                k == 0 && id >= 0 ? BARQ_KV_COLD_ENTRY(id) : id;
          }
        }
        if (r < a.batch) {
          p.seq_lens[r] = len + a.tokens;
          p.high_water[r] = max(hw, len + a.tokens);
        }
      }
      used[0] += total[0];
      used[1] += total[1];
      __syncthreads();  // s_scan / s_incl / s_first are rewritten by the next chunk of rows
    }
    if (pass == 0) {
      // Hot blocks that leave the window: at most the hot pages in use, and counted one by one only
      // where the cold stack might not hold that many.
      if (used[0] <= ctop && ctop - used[0] < (int)p.num_pages - top) {  // uniform
        int old = 0;
        for (int r = wave; r < a.batch; r += kPlanThreads / kWave) {
          const int behind = p.seq_lens[r] + a.tokens - a.c.window;
          const int n = min(min(behind > 0 ? (int)a.div_page.div((uint32_t)behind) : 0, ceil_div_fd(p.high_water[r], a.div_page)), mb);
          const int32_t* row = p.block_table + (int64_t)r * mb;
          for (int j = lane; j < n; j += kWave) {
            const int page = checked_id(row[j], p.num_pages);
            old += page >= 0 && (!p.page_shares || p.page_shares[page] == 0);
          }
        }
        if (old > 0) atomicAdd(&s_old, old);
        __syncthreads();
        used[0] += s_old;
      }
      if (used[0] > ctop || ctop > a.c.num_cold || used[1] > top || top > p.num_pages)
        err |= BARQ_KV_ERRBIT_POOL_EXHAUSTED;
      if (err) atomicOr(&s_bad, err);
      __syncthreads();
      if (s_bad) {  // uniform
        if (tid == 0) {
          p.ctrl[BARQ_KV_CTRL_APPEND_OK] = 0;
          atomicOr(&p.ctrl[BARQ_KV_CTRL_ERRORS], s_bad);
        }
        return;
      }
    } else {
      if (tid == 0) {
        p.ctrl[BARQ_KV_CTRL_COLD_TOP] = ctop - used[0];
        p.ctrl[BARQ_KV_CTRL_FREE_TOP] = top - used[1];
        p.ctrl[BARQ_KV_CTRL_APPEND_OK] = 1;
      }
      if (err) atomicOr(&p.ctrl[BARQ_KV_CTRL_ERRORS], err);
    }
  }
}

// ---------------------------------------------------------------------------------------------
// Gather with dequantisation: tile = (row, block, K or V); a tile's block is hot, cold or
// unmapped for all its positions, so the branch is uniform.  Vectors of VE elements along
// head_dim; output [B, H, S, D] with element strides.
// ---------------------------------------------------------------------------------------------

struct GatherArgs {
  barq_kv_pool p;
  ColdPtrs c;
  char* out[2];
  int64_t osb, osh, oss;  // elements
  int32_t batch;
  int32_t seq_out;
  int32_t nblk;           // output blocks per row
  int32_t from_device;
  FastDiv div_head;       // page_size * head_dim / VE vectors per head
  FastDiv div_dv;         // head_dim / VE
  FastDiv div_nblk;
};

template <int BYTES>
struct Raw;
template <>
struct Raw<16> { using T = uint32_t __attribute__((ext_vector_type(4))); };
template <>
struct Raw<8> { using T = uint32_t __attribute__((ext_vector_type(2))); };
template <>
struct Raw<4> { using T = uint32_t; };
template <>
struct Raw<2> { using T = uint16_t; };
template <>
struct Raw<1> { using T = uint8_t; };

template <int KIND, int VE>
struct Vec {
  using E = Elem<KIND>;
  using Bits = typename E::Bits;
  static constexpr int kBytes = VE * (int)sizeof(Bits);
  using Out = typename Raw<kBytes>::T;
  using Codes = typename Raw<VE>::T;
  union OutU {
    Out v;
    Bits e[VE];
  };
  union CodeU {
    Codes v;
    uint8_t b[VE];
  };
};

// Hardware decode of 8 codes (words w0, w1) with their 8 scale bytes (sk0, sk1): gfx950's OCP
// E4M3 conversion (exact for every finite code) times 2^(s - 127), exact in fp32 while the scale
// bytes stay in [64, 191], rounded to the output type as from_float does.  hw_decodable tells
// when it applies: NaN codes (the hardware drops their sign) and other scales take
// dequant_vec's other paths.
__device__ __forceinline__ bool hw_decodable(uint32_t w0, uint32_t w1, uint32_t sk0, uint32_t sk1) {
  const uint32_t mid = ((sk0 >> 1) ^ sk0) & ((sk1 >> 1) ^ sk1) & 0x40404040u;
  const uint32_t n0 = (w0 & 0x7F7F7F7Fu) ^ 0x7F7F7F7Fu, n1 = (w1 & 0x7F7F7F7Fu) ^ 0x7F7F7F7Fu;
  const uint32_t nan = (((n0 - 0x01010101u) & ~n0) | ((n1 - 0x01010101u) & ~n1)) & 0x80808080u;
  return mid == 0x40404040u && nan == 0;
}

// gfx950's scaled conversion: the two E4M3 codes of half HI of w times the fp32 scale s, rounded
// once to bf16.  Checked on the GPU for every code pair and every scale byte 1 .. 254 (s = 2^(b -
// 127)): identical to rounding the exact product, signed zeros included.
template <bool HI>
__device__ __forceinline__ uint32_t cvt2_bf16(uint32_t w, float s) {
  return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, s, HI));
}
__device__ __forceinline__ float e8m0_scale(uint32_t b) { return __uint_as_float(b << 23); }

template <int KIND>
__device__ __forceinline__ typename Vec<KIND, 8>::Out hw_decode(uint32_t w0, uint32_t w1, uint32_t sk0, uint32_t sk1) {
  using V = Vec<KIND, 8>;
  using E = Elem<KIND>;
  using Bits = typename E::Bits;
  typename V::OutU val;
  if constexpr (KIND == BARQ_KV_BF16) {
    // two conversions per pair of codes, one with each code's scale, and a half of each kept
    uint32_t r[4];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const uint32_t w = j ? w1 : w0, sw = j ? sk1 : sk0;
      const uint32_t a0 = cvt2_bf16<false>(w, e8m0_scale(sw & 0xFFu));
      const uint32_t b0 = cvt2_bf16<false>(w, e8m0_scale((sw >> 8) & 0xFFu));
      const uint32_t a1 = cvt2_bf16<true>(w, e8m0_scale((sw >> 16) & 0xFFu));
      const uint32_t b1 = cvt2_bf16<true>(w, e8m0_scale(sw >> 24));
      r[2 * j] = (a0 & 0xFFFFu) | (b0 & 0xFFFF0000u);
      r[2 * j + 1] = (a1 & 0xFFFFu) | (b1 & 0xFFFF0000u);
    }
    return typename V::Out{r[0], r[1], r[2], r[3]};
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const uint32_t w = j ? w1 : w0, sw = j ? sk1 : sk0;
    const auto lo = __builtin_amdgcn_cvt_pk_f32_fp8((int)w, false);
    const auto hi = __builtin_amdgcn_cvt_pk_f32_fp8((int)w, true);
    const float f[4] = {lo[0] * __uint_as_float((sw & 0xFFu) << 23),
                        lo[1] * __uint_as_float(((sw >> 8) & 0xFFu) << 23),
                        hi[0] * __uint_as_float(((sw >> 16) & 0xFFu) << 23),
                        hi[1] * __uint_as_float((sw >> 24) << 23)};
    // The hardware reads code 0x80 as +0: every code's sign bit goes back on its value.
    if constexpr (KIND == BARQ_KV_BF16) {  // exact values: the top halves
      const uint32_t p0 = __builtin_amdgcn_perm(__float_as_uint(f[1]), __float_as_uint(f[0]), 0x07060302u) |
                          ((w << 8) & 0x8000u) | ((w << 16) & 0x80000000u);
      const uint32_t p1 = __builtin_amdgcn_perm(__float_as_uint(f[3]), __float_as_uint(f[2]), 0x07060302u) |
                          ((w >> 8) & 0x8000u) | (w & 0x80000000u);
      val.e[4 * j] = (Bits)p0;
      val.e[4 * j + 1] = (Bits)(p0 >> 16);
      val.e[4 * j + 2] = (Bits)p1;
      val.e[4 * j + 3] = (Bits)(p1 >> 16);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        val.e[4 * j + e] = (Bits)(E::from_float(f[e]) | (((w >> (8 * e + 7)) & 1u) << 15));
    }
  }
  return val.v;
}

// hw_decode for one scale byte over all 8 codes (a value vector: one scale per position and head).
template <int KIND>
__device__ __forceinline__ typename Vec<KIND, 8>::Out hw_decode_one(uint32_t w0, uint32_t w1, uint32_t sb) {
  if constexpr (KIND == BARQ_KV_BF16) {
    const float s = e8m0_scale(sb);
    return typename Vec<KIND, 8>::Out{cvt2_bf16<false>(w0, s), cvt2_bf16<true>(w0, s), cvt2_bf16<false>(w1, s),
                                      cvt2_bf16<true>(w1, s)};
  } else {
    return hw_decode<KIND>(w0, w1, sb * 0x01010101u, sb * 0x01010101u);
  }
}

// VE elements from their E4M3 codes and scales: keys with VE per-channel scale bytes (ksc),
// values with one per-token scale byte (vsc).  Exact: code * 2^(s - 127) rounded once to the
// element type.
template <int KIND, int VE>
__device__ __forceinline__ typename Vec<KIND, VE>::Out dequant_vec(typename Vec<KIND, VE>::CodeU codes,
                                                                  typename Vec<KIND, VE>::CodeU ksc, uint32_t vsc,
                                                                  int kv) {
  using V = Vec<KIND, VE>;
  using E = Elem<KIND>;
  typename V::OutU val;
  if constexpr (VE == 8 && KIND != BARQ_KV_FP32) {
    const uint32_t w0 = codes.v.x, w1 = codes.v.y;
    const uint32_t sk0 = kv == 0 ? ksc.v.x : vsc * 0x01010101u;
    const uint32_t sk1 = kv == 0 ? ksc.v.y : vsc * 0x01010101u;
    if (hw_decodable(w0, w1, sk0, sk1)) return hw_decode<KIND>(w0, w1, sk0, sk1);
    uint32_t s0, s1, s2, s3;  // scale pairs, spread like the code pairs
    bool fast = codes_normal(w0) && codes_normal(w1);
    if (kv == 0) {
#pragma unroll
      for (int e = 0; e < VE; ++e) fast = fast && scale_fast<KIND>(ksc.b[e]);
      s0 = spread_lo(ksc.v.x);
      s1 = spread_hi(ksc.v.x);
      s2 = spread_lo(ksc.v.y);
      s3 = spread_hi(ksc.v.y);
    } else {
      fast = fast && scale_fast<KIND>(vsc);
      s0 = s1 = s2 = s3 = vsc | (vsc << 16);
    }
    if (fast) {
      uint32_t r[4] = {fast_pair<KIND>(spread_lo(w0), s0), fast_pair<KIND>(spread_hi(w0), s1),
                       fast_pair<KIND>(spread_lo(w1), s2), fast_pair<KIND>(spread_hi(w1), s3)};
      return *(typename V::Out*)r;
    }
  }
  if (kv == 0) {
#pragma unroll
    for (int e = 0; e < VE; ++e) val.e[e] = E::from_float(ldexpf(e4m3_decode(codes.b[e]), (int)ksc.b[e] - 127));
  } else {
#pragma unroll
    for (int e = 0; e < VE; ++e) val.e[e] = E::from_float(ldexpf(e4m3_decode(codes.b[e]), (int)vsc - 127));
  }
  return val.v;
}

template <int KIND, int VE>
__global__ void __launch_bounds__(kGatherThreads) gather_cold_kernel(const GatherArgs a) {
  using V = Vec<KIND, VE>;
  using E = Elem<KIND>;
  using Bits = typename E::Bits;
  __shared__ int s_seq;
  const barq_kv_pool& p = a.p;
  const int kv = blockIdx.x & 1;
  const int bj = blockIdx.x >> 1;
  const int b = (int)a.div_nblk.div((uint32_t)bj);
  const int j = bj - b * a.nblk;
  const int P = (int)p.page_size, H = (int)p.kv_heads, D = (int)p.head_dim;
  const int pos0 = j * P;
  // The row's mark and the block's entry are read together with the lengths (one round trip).
  const int hw = p.high_water[b];
  const int stored = p.block_table[(int64_t)b * p.max_blocks + j];
  // The extent (longest row) matters only to a block reaching past its row's length: the others
  // hold data at every position and skip the batch-wide read.
  const bool need_extent = a.from_device && pos0 + P > p.seq_lens[b];
  if (need_extent) {  // uniform
    if (threadIdx.x < kWave) {
      int m = 0;
      for (int i = threadIdx.x; i < a.batch; i += kWave) m = max(m, p.seq_lens[i]);
#pragma unroll
      for (int o = kWave / 2; o > 0; o >>= 1) m = max(m, __shfl_xor(m, o, kWave));
      if (threadIdx.x == 0) s_seq = min(m, a.seq_out);
    }
    __syncthreads();
  }
  const int S = need_extent ? s_seq : a.seq_out;
  if (pos0 >= S) return;  // uniform
  const int entry = pos0 < hw ? stored : -1;
  const int hot = checked_id(entry, p.num_pages);
  const int cold = entry <= -2 ? checked_id(-2 - entry, a.c.num_cold) : -1;
  if (entry <= -2 && cold < 0 && threadIdx.x == 0) atomicOr(&p.ctrl[BARQ_KV_CTRL_ERRORS], BARQ_KV_ERRBIT_BAD_INDEX);
  const int dv_n = (int)a.div_dv.d;
  const int nvec = H * P * dv_n;
  Bits* out = (Bits*)a.out[kv] + (int64_t)b * a.osb;
  const int live = min(S, hw) - pos0;  // positions of this block with data
  const int end = min(S - pos0, P);    // positions of this block in the output
  const int slot = hot >= 0 ? hot : cold;
  // Every load of a round is issued before any value is used (one round trip per round).
  for (int v0 = threadIdx.x; v0 < nvec; v0 += kGatherThreads * kUnroll) {
    typename V::OutU val[kUnroll];
    int64_t at[kUnroll], el[kUnroll];
    int tok[kUnroll], head[kUnroll], col[kUnroll];
    bool in[kUnroll], has[kUnroll];
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      const int v = v0 + u * kGatherThreads;
      const int h = (int)a.div_head.div((uint32_t)v);
      const int rem = v - h * (int)a.div_head.d;
      const int t = (int)a.div_dv.div((uint32_t)rem);
      const int dv = rem - t * dv_n;
      in[u] = v < nvec && t < end;
      has[u] = in[u] && t < live && slot >= 0;
      at[u] = (int64_t)h * a.osh + (int64_t)(pos0 + t) * a.oss + (int64_t)dv * VE;
      el[u] = (((int64_t)slot * P + t) * H + h) * D + (int64_t)dv * VE;
      tok[u] = t;
      head[u] = h;
      col[u] = dv * VE;
      val[u].v = typename V::Out(0);
    }
    if (hot >= 0) {  // uniform
      const char* base = kv ? (const char*)p.value_pages : (const char*)p.key_pages;
#pragma unroll
      for (int u = 0; u < kUnroll; ++u)
        if (has[u]) val[u].v = __builtin_nontemporal_load((const typename V::Out*)(base + el[u] * (int64_t)sizeof(Bits)));
    } else if (cold >= 0) {  // uniform
      typename V::CodeU codes[kUnroll], ksc[kUnroll];
      uint32_t vsc[kUnroll];
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
        codes[u].v = typename V::Codes(0);
        ksc[u].v = typename V::Codes(0);
        vsc[u] = 0;
        if (!has[u]) continue;
        codes[u].v = __builtin_nontemporal_load((const typename V::Codes*)(a.c.codes[kv] + el[u]));
        if (kv == 0)
          ksc[u].v = *(const typename V::Codes*)(a.c.key_scales + ((int64_t)cold * H + head[u]) * D + col[u]);
        else
          vsc[u] = a.c.value_scales[((int64_t)cold * P + tok[u]) * H + head[u]];
      }
#pragma unroll
      for (int u = 0; u < kUnroll; ++u)
        if (has[u]) val[u].v = dequant_vec<KIND, VE>(codes[u], ksc[u], vsc[u], kv);
    }
#pragma unroll
    for (int u = 0; u < kUnroll; ++u)
      if (in[u]) __builtin_nontemporal_store(val[u].v, (typename V::Out*)(out + at[u]));
  }
}

// dequant_vec's exact path for 8 codes (words w0, w1) and their scale bytes (sk0, sk1), one
// element at a time: the rare path of the lanes kernels, holding one element's registers.
template <int KIND>
__device__ __forceinline__ typename Vec<KIND, 8>::Out exact8(uint32_t w0, uint32_t w1, uint32_t sk0, uint32_t sk1) {
  uint32_t r0 = 0, r1 = 0, r2 = 0, r3 = 0;
#pragma unroll 1
  for (int e = 0; e < 8; ++e) {
    const int sh = 8 * (e & 3);
    const uint32_t code = ((e < 4 ? w0 : w1) >> sh) & 0xFFu;
    const int sc = (int)(((e < 4 ? sk0 : sk1) >> sh) & 0xFFu);
    const uint32_t bits = (uint32_t)Elem<KIND>::from_float(ldexpf(e4m3_decode(code), sc - 127)) << (16 * (e & 1));
    const int word = e >> 1;
    r0 |= word == 0 ? bits : 0u;
    r1 |= word == 1 ? bits : 0u;
    r2 |= word == 2 ? bits : 0u;
    r3 |= word == 3 ? bits : 0u;
  }
  return typename Vec<KIND, 8>::Out{r0, r1, r2, r3};
}

// ---------------------------------------------------------------------------------------------
// An append to empty rows -- a prompt -- by a caller that knows they are empty and the tops of both
// stacks: every row takes the same number of cold pages and of hot pages after them, so a block's page
// is one stack entry and no launch has to plan the append first.  With an output (dense states as a
// gather would return them: cold blocks as their codes read) a wave stores its unit's codes, scales and
// dequantised elements from the registers it was quantised in.  Units are independent: workgroups are a
// few of a block's units, the block's first also writing its table entry (and row 0's the tops).
//
// Bound: HBM (input read once, codes and output written once).  A 16 x 1000-token prompt of the 8 x 128
// bf16 shape: 31 us for 163 MB (5.3 TB/s) against 7.1 (plan) + 25.6 + 17.7 (gather, codes from cache);
// without output 20.7 against 32.7.
// ---------------------------------------------------------------------------------------------

struct FreshArgs {
  QuantArgs q;            // tokens: the rows' new length
  char* out[2];           // key, value output, or null
  int64_t osb, osh;       // output strides, elements
  uint32_t oss;
  int32_t ncold, nblk;    // blocks of a row: cold ones first
  int32_t top, ctop;      // free pages and free cold pages before the launch
  FastDiv div_groups;     // workgroups of a block
  FastDiv div_nblk;
};

constexpr int kFreshWaves = 8;  // a page's value scales from one workgroup while kv_heads <= 8

template <int KIND, int NV>
__global__ void __launch_bounds__(kFreshWaves * kWave) __attribute__((amdgpu_waves_per_eu(NV <= 4 ? 6 : 4))) fresh_blocks_kernel(const FreshArgs f) {
  using V = typename RawC<16>::T;
  using Bits = typename Elem<KIND>::Bits;
  const QuantArgs& a = f.q;
  const barq_kv_pool& p = a.p;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int bj = (int)f.div_groups.div(blockIdx.x);
  const int g = (int)blockIdx.x - bj * (int)f.div_groups.d;
  const int b = (int)f.div_nblk.div((uint32_t)bj);
  const int j = bj - b * f.nblk;
  const int P = (int)p.page_size, H = (int)p.kv_heads, D = (int)p.head_dim;
  const bool to_cold = j < f.ncold;
  // within the stacks: the host checked their tops
  const int32_t* entry = to_cold ? a.c.free_cold + (f.ctop - 1 - (b * f.ncold + j))
                                 : p.free_pages + (f.top - 1 - (b * (f.nblk - f.ncold) + j - f.ncold));
  const int stored = *entry;
  const int u = g * kFreshWaves + wave;  // the wave's unit: heads of K, then of V
  const int kv = u >= H ? 1 : 0, h = u - kv * H;
  V x[NV];
  if (u < 2 * H && to_cold) load_unit<KIND, NV>(a, b, kv, h, -1, j * P, 0, x);
  const int id = checked_id(stored, to_cold ? a.c.num_cold : p.num_pages);
  if (g == 0 && threadIdx.x == 0) {
    p.block_table[(int64_t)b * p.max_blocks + j] = to_cold && id >= 0 ? BARQ_KV_COLD_ENTRY(id) : id;
    if (id < 0) atomicOr(&p.ctrl[BARQ_KV_CTRL_ERRORS], BARQ_KV_ERRBIT_BAD_INDEX);
    if (j == 0) {
      p.seq_lens[b] = a.tokens;
      p.high_water[b] = a.tokens;
    }
    if (bj == 0) {
      const int batch = (int)(gridDim.x / (f.div_groups.d * f.div_nblk.d));
      p.ctrl[BARQ_KV_CTRL_COLD_TOP] = f.ctop - batch * f.ncold;
      p.ctrl[BARQ_KV_CTRL_FREE_TOP] = f.top - batch * (f.nblk - f.ncold);
    }
  }
  if (u >= 2 * H) return;
  Bits* out = f.out[kv] ? (Bits*)f.out[kv] + ((int64_t)b * f.osb + (int64_t)h * f.osh + (int64_t)j * P * f.oss) : nullptr;
  if (to_cold && id >= 0) {  // uniform
    constexpr int VE = 16 / (int)sizeof(Bits);
    if (out) {  // uniform
      quantise_unit<KIND, NV, kWholeUnit>(a, kv, h, id, x, [&](int t, int col, const uint32_t (&w)[VE / 4], const uint32_t (&ks)[VE / 4], uint32_t vs) {
        V v;
        if constexpr (KIND == BARQ_KV_FP32) {
          typename Vec<KIND, VE>::CodeU c, k;
          c.v = w[0];
          k.v = ks[0];
          v = dequant_vec<KIND, VE>(c, k, vs, kv);
        } else {
          const uint32_t sk0 = kv ? vs * 0x01010101u : ks[0], sk1 = kv ? sk0 : ks[1];
          if (__builtin_amdgcn_ballot_w64(!hw_decodable(w[0], w[1], sk0, sk1)) == 0)  // uniform
            v = kv ? hw_decode_one<KIND>(w[0], w[1], vs) : hw_decode<KIND>(w[0], w[1], sk0, sk1);
          else
            v = exact8<KIND>(w[0], w[1], sk0, sk1);
        }
        __builtin_nontemporal_store(v, (V*)(out + ((uint32_t)t * f.oss + (uint32_t)col)));
      });
    } else {
      quantise_unit<KIND, NV>(a, kv, h, id, x);
    }
    return;
  }
  const int lane = opaque_lane();
  const int col = (lane & ((1 << a.vd_log2) - 1)) * (16 / (int)sizeof(Bits));
  const int t0 = lane >> a.vd_log2, step = kWave >> a.vd_log2;
  const int n = min(a.tokens - j * P, P);
  const Bits* in = (const Bits*)a.in[kv] + ((int64_t)b * a.isb + (int64_t)h * a.ish + (int64_t)j * P * a.ist);
  Bits* page = (Bits*)(kv ? p.value_pages : p.key_pages) + ((int64_t)max(id, 0) * P * H + h) * D;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int t = t0 + k * step;
    x[k] = V(0);
    if (t < n && id >= 0) x[k] = __builtin_nontemporal_load((const V*)(in + ((uint32_t)t * (uint32_t)a.ist + (uint32_t)col)));
  }
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int t = t0 + k * step;
    if (t >= n) continue;
    if (id >= 0) *(V*)(page + (uint32_t)(t * H * D + col)) = x[k];
    if (out) __builtin_nontemporal_store(x[k], (V*)(out + ((uint32_t)t * f.oss + (uint32_t)col)));
  }
}

// One wave's round of a cold tile in the lanes kernels (VALUES: the V page, whose scales are
// per position and head; else K, per-channel scales ksc): positions t0 .. t0 + 8 / LPP - 1 of
// the page, decoded below `live`, zeros up to `end`; the lane's columns col[c] (element offsets
// in a token row) go to ocol[c] of the output rows at o.  The round's codes and scales load
// together and unconditionally (positions clamped into the page): a load under a condition
// leaves a phi of zero and the loaded value, into whose block the compiler moves the scale
// arithmetic, waiting there for each load before the next is issued.  A vector decodes on the
// hardware path when every lane's does (scales in [64, 191], no NaN code: the usual case), else
// element by element; with dequant_vec inlined for the whole round the kernels held 4 waves per
// SIMD instead of 5.  `spaced` (uniform): each store waits for the previous one, one store in
// flight per wave.
template <int KIND, int LPP, bool VALUES>
__device__ __forceinline__ void cold_round(const GatherArgs& a, int cold, int t0, int live, int end, int lane,
                                           const int (&col)[LPP], const int64_t (&ocol)[LPP],
                                           const typename Vec<KIND, 8>::CodeU (&ksc)[LPP],
                                           typename Elem<KIND>::Bits* o, bool spaced) {
  using V = Vec<KIND, 8>;
  constexpr int kNPos = 8 / LPP;
  const barq_kv_pool& p = a.p;
  const int P = (int)p.page_size, H = (int)p.kv_heads, D = (int)p.head_dim;
  const int HD = H * D;
  const int dvn = D / 8;
  const uint8_t* codes = a.c.codes[VALUES ? 1 : 0] + (int64_t)cold * P * HD;
  const uint8_t* vscales = a.c.value_scales + (int64_t)cold * P * H;
  typename V::CodeU cv[kNPos][LPP];
  uint32_t vsc[kNPos][LPP];
#pragma unroll
  for (int i = 0; i < kNPos; ++i) {
    const int t = min(t0 + i, P - 1);
#pragma unroll
    for (int c = 0; c < LPP; ++c) {
      cv[i][c].v = __builtin_nontemporal_load((const typename V::Codes*)(codes + (int64_t)t * HD + col[c]));
      vsc[i][c] = VALUES ? vscales[t * H + (c * kWave + lane) / dvn] : 0u;
    }
  }
#pragma unroll
  for (int i = 0; i < kNPos; ++i)
#pragma unroll
    for (int c = 0; c < LPP; ++c) {
      if (t0 + i >= end) continue;
      const uint32_t w0 = cv[i][c].v.x, w1 = cv[i][c].v.y;
      const uint32_t sk0 = VALUES ? vsc[i][c] * 0x01010101u : ksc[c].v.x;
      const uint32_t sk1 = VALUES ? vsc[i][c] * 0x01010101u : ksc[c].v.y;
      const bool dead = t0 + i >= live;
      typename V::Out v;
      if (__builtin_amdgcn_ballot_w64(!(dead || hw_decodable(w0, w1, sk0, sk1))) == 0) {  // uniform
        if constexpr (VALUES)
          v = hw_decode_one<KIND>(w0, w1, vsc[i][c]);
        else
          v = hw_decode<KIND>(w0, w1, sk0, sk1);
      } else
        v = exact8<KIND>(w0, w1, sk0, sk1);
      if (dead) v = typename V::Out(0);
      if (spaced) wait_vm<0>();
      __builtin_nontemporal_store(v, (typename V::Out*)(o + (int64_t)i * a.oss + ocol[c]));
    }
}

// The gather for 8-element vectors (2-byte elements) when a token's kv_heads * head_dim
// elements are 64 * LPP vectors: a wave moves whole positions, lane l taking vectors l, l + 64,
// ... of each, so a lane's columns -- and its key scales -- are fixed for the tile and only the
// position varies (wave-uniform).  Each wave holds 8 vectors per lane in flight (8 / LPP
// positions a round); per-channel key scales are read once per tile.
template <int KIND, int LPP>
__global__ void __launch_bounds__(kGatherThreads) gather_cold_lanes_kernel(const GatherArgs a) {
  using V = Vec<KIND, 8>;
  using E = Elem<KIND>;
  using Bits = typename E::Bits;
  constexpr int kNPos = 8 / LPP;  // positions a wave moves per round
  constexpr int kWavesPerTile = kGatherThreads / kWave;
  __shared__ int s_seq;
  const barq_kv_pool& p = a.p;
  const int kv = blockIdx.x & 1;
  const int bj = blockIdx.x >> 1;
  const int b = (int)a.div_nblk.div((uint32_t)bj);
  const int j = bj - b * a.nblk;
  const int P = (int)p.page_size, H = (int)p.kv_heads, D = (int)p.head_dim;
  const int pos0 = j * P;
  const int hw = p.high_water[b];
  const int stored = p.block_table[(int64_t)b * p.max_blocks + j];
  // The extent (longest row) matters only to a block reaching past its row's length: the others
  // hold data at every position and skip the batch-wide read.
  const bool need_extent = a.from_device && pos0 + P > p.seq_lens[b];
  if (need_extent) {  // uniform
    if (threadIdx.x < kWave) {
      int m = 0;
      for (int i = threadIdx.x; i < a.batch; i += kWave) m = max(m, p.seq_lens[i]);
#pragma unroll
      for (int o = kWave / 2; o > 0; o >>= 1) m = max(m, __shfl_xor(m, o, kWave));
      if (threadIdx.x == 0) s_seq = min(m, a.seq_out);
    }
    __syncthreads();
  }
  const int S = need_extent ? s_seq : a.seq_out;
  if (pos0 >= S) return;  // uniform
  const int entry = pos0 < hw ? stored : -1;
  const int hot = checked_id(entry, p.num_pages);
  const int cold = entry <= -2 ? checked_id(-2 - entry, a.c.num_cold) : -1;
  if (entry <= -2 && cold < 0 && threadIdx.x == 0) atomicOr(&p.ctrl[BARQ_KV_CTRL_ERRORS], BARQ_KV_ERRBIT_BAD_INDEX);
  const int live = min(S, hw) - pos0;
  const int end = min(S - pos0, P);
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int HD = H * D;
  const int dvn = D / 8;
  // this lane's columns: element offsets within a token row and within an output position
  int col[LPP];
  int64_t ocol[LPP];
#pragma unroll
  for (int c = 0; c < LPP; ++c) {
    const int vi = c * kWave + lane;
    const int h = vi / dvn;
    col[c] = vi * 8;
    ocol[c] = (int64_t)h * a.osh + (int64_t)(vi - h * dvn) * 8;
  }
  Bits* out = (Bits*)a.out[kv] + (int64_t)b * a.osb + (int64_t)pos0 * a.oss;
  typename V::CodeU ksc[LPP];
  if (cold >= 0 && kv == 0) {
#pragma unroll
    for (int c = 0; c < LPP; ++c) ksc[c].v = *(const typename V::Codes*)(a.c.key_scales + (int64_t)cold * HD + col[c]);
  }
  for (int t0 = wave * kNPos; t0 < end; t0 += kWavesPerTile * kNPos) {
    Bits* o = out + (int64_t)t0 * a.oss;
    if (hot >= 0) {  // uniform: a copy, every load of the round in flight before the stores
      const char* base = (kv ? (const char*)p.value_pages : (const char*)p.key_pages) +
                         ((int64_t)hot * P + t0) * HD * (int64_t)sizeof(Bits);
      typename V::OutU val[kNPos][LPP];
#pragma unroll
      for (int i = 0; i < kNPos; ++i)
#pragma unroll
        for (int c = 0; c < LPP; ++c) {
          val[i][c].v = typename V::Out(0);
          if (t0 + i < live)
            val[i][c].v = __builtin_nontemporal_load(
                (const typename V::Out*)(base + ((int64_t)i * HD + col[c]) * (int64_t)sizeof(Bits)));
        }
#pragma unroll
      for (int i = 0; i < kNPos; ++i)
#pragma unroll
        for (int c = 0; c < LPP; ++c)
          if (t0 + i < end) __builtin_nontemporal_store(val[i][c].v, (typename V::Out*)(o + (int64_t)i * a.oss + ocol[c]));
    } else if (cold >= 0) {  // uniform
      if (kv)
        cold_round<KIND, LPP, true>(a, cold, t0, live, end, lane, col, ocol, ksc, o, false);
      else
        cold_round<KIND, LPP, false>(a, cold, t0, live, end, lane, col, ocol, ksc, o, false);
    } else {
#pragma unroll
      for (int i = 0; i < kNPos; ++i)
#pragma unroll
        for (int c = 0; c < LPP; ++c)
          if (t0 + i < end) __builtin_nontemporal_store(typename V::Out(0), (typename V::Out*)(o + (int64_t)i * a.oss + ocol[c]));
    }
  }
}

// The dequantising update in one launch, for tokens <= window (the blocks that leave the window
// were quantised just before, from the lengths the rows are about to reach): the tiles of
// gather_cold_lanes_kernel, whose rows also receive `tokens` new positions.  Every tile reads
// the launch's starting state -- the row's length and mark, its block's entry, the output extent
// (longest row + tokens), and for a block the append maps first the page its rank takes from the
// stack -- then arrives; the last tile to arrive commits the append (barq_commit, as the stream
// kernels do).  New positions are taken from the input, written to the output and to their hot
// page; a tile holding none runs gather_cold_lanes_kernel's copy or decode unchanged.
struct UpdateArgs {
  GatherArgs g;
  const char* in[2];      // key, value states
  int64_t isb, ish, ist;  // input strides, elements
  int32_t tokens;
  int32_t nsub;           // arrival sub-counters in use
  int32_t spaced;         // every tile resident at once: one store in flight per wave (3 % faster
                          // at C2); launches of several rounds keep their stores back to back
  FastDiv div_page;
};

// The row state of a caller that knows it exactly (barq_internal::update_cold_known): no tile reads it
// from the device, none arrives, and the first workgroup commits.  An arrival is a round trip to a
// counter that the tile's first wave makes before its loads: 16 rows of 648 positions (8 x 128 bf16,
// 64 MB) took 17.9 us with arrivals and take 15.5 without.  (Six waves a SIMD spill, 19.5 us; four or
// three tiles a CU at a time, 16.1 - 16.3; up to 12 positions a tile, cut evenly, 19.2.)
struct KnownRows {
  int32_t len[kWave];
  int32_t hw[kWave];
  int32_t top;
};

template <int KIND, int LPP, bool KNOWN>
__device__ __forceinline__ void update_cold_tile(const UpdateArgs& u, const KnownRows* ks) {
  using V = Vec<KIND, 8>;
  using E = Elem<KIND>;
  using Bits = typename E::Bits;
  constexpr int kNPos = 8 / LPP;  // positions a wave moves per round
  constexpr int kWavesPerTile = kGatherThreads / kWave;
  const GatherArgs& a = u.g;
  const barq_kv_pool& p = a.p;
  const int kv = blockIdx.x & 1;
  const int bj = blockIdx.x >> 1;
  const int b = (int)a.div_nblk.div((uint32_t)bj);
  const int j = bj - b * a.nblk;
  const int P = (int)p.page_size, H = (int)p.kv_heads, D = (int)p.head_dim;
  const int T = u.tokens;
  const int mb = (int)p.max_blocks;
  const int pos0 = j * P;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);

  // The launch's starting state (batch <= 64: one row per lane).
  const int len = KNOWN ? ks->len[b] : p.seq_lens[b];
  const int hw = KNOWN ? ks->hw[b] : p.high_water[b];
  const int stored = p.block_table[(int64_t)b * mb + j];
  // The extent (longest row + tokens) matters only to a block reaching past its row's new end:
  // the others hold data at every position and skip the batch-wide read (every tile reading the
  // same lengths serialises on one L2 channel).
  int S = a.seq_out;
  if (!KNOWN && a.from_device && pos0 + P > len + T)
    S = min(barq_commit::wave_max(lane < a.batch ? p.seq_lens[lane] + T : 0), a.seq_out);
  const barq_commit::NewBlocks nb = barq_commit::new_blocks(len, hw, T, mb, u.div_page);
  const bool fresh_block = j >= nb.first && j < nb.first + nb.count;
  int newpage = -1;
  if (fresh_block) {
    const int top = KNOWN ? ks->top : p.ctrl[BARQ_KV_CTRL_FREE_TOP];
    const int rl = lane < b ? (KNOWN ? ks->len[lane] : p.seq_lens[lane]) : 0;
    const int rh = lane < b ? (KNOWN ? ks->hw[lane] : p.high_water[lane]) : 0;
    const int base = barq_commit::wave_sum(lane < b ? barq_commit::new_blocks(rl, rh, T, mb, u.div_page).count : 0);
    const int idx = top - 1 - (base + j - nb.first);
    newpage = idx >= 0 ? checked_id(p.free_pages[idx], p.num_pages) : -1;
  }
  if constexpr (!KNOWN) {
    __builtin_amdgcn_s_waitcnt(0);  // every wave holds its metadata before the tile arrives
    __syncthreads();
    if (wave == 0) barq_commit::arrive_and_commit(p, u.nsub, a.batch, T, a.seq_out, u.div_page);
  }
  if (pos0 >= S) return;  // uniform

  const bool old_block = pos0 < hw;  // mapped before this append
  const int entry = old_block ? stored : -1;
  const int hot = old_block ? checked_id(entry, p.num_pages) : newpage;
  const int cold = entry <= -2 ? checked_id(-2 - entry, a.c.num_cold) : -1;
  if (entry <= -2 && cold < 0 && threadIdx.x == 0) atomicOr(&p.ctrl[BARQ_KV_CTRL_ERRORS], BARQ_KV_ERRBIT_BAD_INDEX);
  const int live = min(S, hw) - pos0;  // old data: positions below the mark
  const int end = min(S - pos0, P);
  const int f_lo = len - pos0;         // new positions of the tile: [f_lo, f_lo + T) within [0, end)
  const bool fresh_tile = f_lo < end && f_lo + T > 0;
  const int HD = H * D;
  const int dvn = D / 8;
  int col[LPP];
  int64_t ocol[LPP], icol[LPP];
#pragma unroll
  for (int c = 0; c < LPP; ++c) {
    const int vi = c * kWave + lane;
    const int h = vi / dvn;
    col[c] = vi * 8;
    ocol[c] = (int64_t)h * a.osh + (int64_t)(vi - h * dvn) * 8;
    icol[c] = (int64_t)h * u.ish + (int64_t)(vi - h * dvn) * 8;
  }
  Bits* out = (Bits*)a.out[kv] + (int64_t)b * a.osb + (int64_t)pos0 * a.oss;
  char* page_base = hot >= 0 ? (kv ? (char*)p.value_pages : (char*)p.key_pages) +
                                   (int64_t)hot * P * HD * (int64_t)sizeof(Bits)
                             : nullptr;
  if (fresh_tile) {
    // New positions from the input (to the output and their page), old ones from the hot page.
    const Bits* in = (const Bits*)u.in[kv] + (int64_t)b * u.isb;
    if (cold >= 0 && threadIdx.x == 0) atomicOr(&p.ctrl[BARQ_KV_CTRL_ERRORS], BARQ_KV_ERRBIT_BAD_INDEX);
    for (int t0 = wave * kNPos; t0 < end; t0 += kWavesPerTile * kNPos) {
      typename V::OutU val[kNPos][LPP];
#pragma unroll
      for (int i = 0; i < kNPos; ++i) {
        const int t = t0 + i;
        const bool fresh = (unsigned)(t - f_lo) < (unsigned)T;
#pragma unroll
        for (int c = 0; c < LPP; ++c) {
          val[i][c].v = typename V::Out(0);
          if (t < end && fresh)
            val[i][c].v = __builtin_nontemporal_load(
                (const typename V::Out*)(in + (int64_t)(t - f_lo) * u.ist + icol[c]));
          else if (t < live && hot >= 0)
            val[i][c].v = __builtin_nontemporal_load(
                (const typename V::Out*)(page_base + ((int64_t)t * HD + col[c]) * (int64_t)sizeof(Bits)));
        }
      }
#pragma unroll
      for (int i = 0; i < kNPos; ++i) {
        const int t = t0 + i;
        if (t >= end) continue;
        const bool fresh = (unsigned)(t - f_lo) < (unsigned)T;
#pragma unroll
        for (int c = 0; c < LPP; ++c) {
          __builtin_nontemporal_store(val[i][c].v, (typename V::Out*)(out + (int64_t)t * a.oss + ocol[c]));
          if (fresh && hot >= 0)
            *(typename V::Out*)(page_base + ((int64_t)t * HD + col[c]) * (int64_t)sizeof(Bits)) = val[i][c].v;
        }
      }
    }
    return;
  }
  typename V::CodeU ksc[LPP];
  if (cold >= 0 && kv == 0) {
#pragma unroll
    for (int c = 0; c < LPP; ++c) ksc[c].v = *(const typename V::Codes*)(a.c.key_scales + (int64_t)cold * HD + col[c]);
  }
  for (int t0 = wave * kNPos; t0 < end; t0 += kWavesPerTile * kNPos) {
    Bits* o = out + (int64_t)t0 * a.oss;
    if (hot >= 0) {  // uniform: a copy, every load of the round in flight before the stores
      const char* base = page_base + (int64_t)t0 * HD * (int64_t)sizeof(Bits);
      typename V::OutU val[kNPos][LPP];
#pragma unroll
      for (int i = 0; i < kNPos; ++i)
#pragma unroll
        for (int c = 0; c < LPP; ++c) {
          val[i][c].v = typename V::Out(0);
          if (t0 + i < live)
            val[i][c].v = __builtin_nontemporal_load(
                (const typename V::Out*)(base + ((int64_t)i * HD + col[c]) * (int64_t)sizeof(Bits)));
        }
#pragma unroll
      for (int i = 0; i < kNPos; ++i)
#pragma unroll
        for (int c = 0; c < LPP; ++c)
          if (t0 + i < end) {
            if (u.spaced) wait_vm<0>();
            __builtin_nontemporal_store(val[i][c].v, (typename V::Out*)(o + (int64_t)i * a.oss + ocol[c]));
          }
    } else if (cold >= 0) {  // uniform
      if (kv)
        cold_round<KIND, LPP, true>(a, cold, t0, live, end, lane, col, ocol, ksc, o, u.spaced);
      else
        cold_round<KIND, LPP, false>(a, cold, t0, live, end, lane, col, ocol, ksc, o, u.spaced);
    } else {
#pragma unroll
      for (int i = 0; i < kNPos; ++i)
#pragma unroll
        for (int c = 0; c < LPP; ++c)
          if (t0 + i < end) __builtin_nontemporal_store(typename V::Out(0), (typename V::Out*)(o + (int64_t)i * a.oss + ocol[c]));
    }
  }
}

template <int KIND, int LPP>
__global__ void __launch_bounds__(kGatherThreads) __attribute__((amdgpu_waves_per_eu(LPP <= 2 ? 5 : 3))) update_cold_lanes_kernel(const UpdateArgs u) {
  update_cold_tile<KIND, LPP, false>(u, nullptr);
}

// The commit follows the first tile's data: no tile reads what it writes (a block of new positions takes
// its page from the stack, whose entries stay).
template <int KIND, int LPP>
__global__ void __launch_bounds__(kGatherThreads) __attribute__((amdgpu_waves_per_eu(LPP <= 2 ? 5 : 3))) update_cold_known_kernel(const UpdateArgs u, const KnownRows ks) {
  update_cold_tile<KIND, LPP, true>(u, &ks);
  if (blockIdx.x != 0 || threadIdx.x >= kWave) return;
  const barq_kv_pool& p = u.g.p;
  const int lane = threadIdx.x, batch = u.g.batch;
  const int len = lane < batch ? ks.len[lane] : 0, hw = lane < batch ? ks.hw[lane] : 0;
  const int news = barq_commit::wave_sum(
      lane < batch ? barq_commit::new_blocks(len, hw, u.tokens, (int)p.max_blocks, u.div_page).count : 0);
  const int idx = ks.top - 1 - lane;
  barq_commit::commit_from_lanes(p, batch, u.tokens, u.g.seq_out, u.div_page, len, hw, ks.top,
                                 news > 0 && idx >= 0 ? p.free_pages[idx] : -1);
}

// ---------------------------------------------------------------------------------------------
// Row release with a cold store: one workgroup, a row at a time; hot pages (shares-aware) go back
// to free_pages, cold pages to free_cold, each in (row, block) order.
// ---------------------------------------------------------------------------------------------

struct FreeArgs {
  barq_kv_pool p;
  ColdPtrs c;
  const int32_t* rows;
  int32_t n;
  FastDiv div_page;
};

__global__ void __launch_bounds__(kThreads) free_rows_cold_kernel(const FreeArgs a) {
  __shared__ int lds_scan[kWaves];
  const barq_kv_pool& p = a.p;
  const int hot_top = p.ctrl[BARQ_KV_CTRL_FREE_TOP];
  const int cold_top = p.ctrl[BARQ_KV_CTRL_COLD_TOP];
  const int mb = (int)p.max_blocks;
  int hot_pushed = 0, cold_pushed = 0, err = 0;
  for (int i = 0; i < a.n; ++i) {
    const int r = a.rows[i];
    if (r < 0 || r >= (int)p.max_batch) {
      err |= BARQ_KV_ERRBIT_BAD_INDEX;
      continue;
    }
    const int cnt = min(ceil_div_fd(p.high_water[r], a.div_page), mb);
    int32_t* row = p.block_table + (int64_t)r * mb;
    for (int j0 = 0; j0 < cnt; j0 += kThreads) {
      const int j = j0 + (int)threadIdx.x;
      int hot = -1, cold = -1;
      if (j < cnt) {
        const int e = row[j];
        hot = checked_id(e, p.num_pages);
        if (e <= -2) cold = checked_id(-2 - e, a.c.num_cold);
        if (hot >= 0 && p.page_shares && atomicSub(&p.page_shares[hot], 1) != 0) hot = -1;
        else if (hot >= 0 && p.page_shares) p.page_shares[hot] = 0;
        if (cold >= 0 && a.c.shares && atomicSub(&a.c.shares[cold], 1) != 0) cold = -1;
        else if (cold >= 0 && a.c.shares) a.c.shares[cold] = 0;
        row[j] = -1;
      }
      int hot_n = 0, cold_n = 0;
      const int hk = block_exclusive_scan(hot >= 0, lds_scan, &hot_n);
      const int ck = block_exclusive_scan(cold >= 0, lds_scan, &cold_n);
      if (hot >= 0) {
        const int64_t slot = (int64_t)hot_top + hot_pushed + hk;
        if (slot < p.num_pages) p.free_pages[slot] = hot;
        else err |= BARQ_KV_ERRBIT_BAD_INDEX;
      }
      if (cold >= 0) {
        const int64_t slot = (int64_t)cold_top + cold_pushed + ck;
        if (slot < a.c.num_cold) a.c.free_cold[slot] = cold;
        else err |= BARQ_KV_ERRBIT_BAD_INDEX;
      }
      hot_pushed += hot_n;
      cold_pushed += cold_n;
    }
    __syncthreads();  // every thread has read the row's mark before it is cleared
    if (threadIdx.x == 0) {
      p.seq_lens[r] = 0;
      p.high_water[r] = 0;
    }
  }
  if (threadIdx.x == 0) {
    p.ctrl[BARQ_KV_CTRL_FREE_TOP] = (int)std::min<int64_t>((int64_t)hot_top + hot_pushed, p.num_pages);
    p.ctrl[BARQ_KV_CTRL_COLD_TOP] = (int)std::min<int64_t>((int64_t)cold_top + cold_pushed, a.c.num_cold);
  }
  if (err) atomicOr(&p.ctrl[BARQ_KV_CTRL_ERRORS], err);
}

__global__ void cold_reset_kernel(ColdPtrs c, int32_t* ctrl) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < c.num_cold) c.free_cold[i] = (int32_t)(c.num_cold - 1 - i);
  if (i < c.num_cold && c.shares) c.shares[i] = 0;
  if (i == 0) ctrl[BARQ_KV_CTRL_COLD_TOP] = (int32_t)c.num_cold;
}

// ---------------------------------------------------------------------------------------------
// Crop with a cold store: workgroup per row.  The row's quantised blocks from the one holding its
// new length on are re-opened: a page popped from free_pages receives the block's dequantised K
// and V (code * 2^e rounded to the element type, as the gather reads it), the block maps it, and
// the cold page loses the reference.
// ---------------------------------------------------------------------------------------------

struct CropArgs {
  barq_kv_pool p;
  ColdPtrs c;
  int32_t batch;
  int32_t max_length;
  FastDiv div_page;
};

template <int KIND>
__global__ void __launch_bounds__(kThreads) crop_cold_kernel(const CropArgs a) {
  using E = Elem<KIND>;
  using Bits = typename E::Bits;
  __shared__ int lds_scan[kWaves];
  __shared__ int s_block[kThreads];  // the chunk's re-opened blocks ...
  __shared__ int s_hot[kThreads];    // ... and the pages they take (-1: none left)
  __shared__ int s_base;
  const barq_kv_pool& p = a.p;
  const int r = blockIdx.x;
  const int mb = (int)p.max_blocks;
  const int P = (int)p.page_size, H = (int)p.kv_heads, D = (int)p.head_dim;
  const int HD = H * D;
  const int len = min(p.seq_lens[r], a.max_length);
  const int first = (int)a.div_page.div((uint32_t)len);
  const int nb = min(ceil_div_fd(p.high_water[r], a.div_page), mb);
  int32_t* row = p.block_table + (int64_t)r * mb;
  int err = 0;
  for (int j0 = first; j0 < nb; j0 += kThreads) {
    const int j = j0 + (int)threadIdx.x;
    int c = -1;
    if (j < nb) {
      const int e = row[j];
      if (e <= -2) c = checked_id(-2 - e, a.c.num_cold);
    }
    int count = 0;
    const int k = block_exclusive_scan(c >= 0, lds_scan, &count);
    if (threadIdx.x == 0 && count > 0) {
      const int before = atomicSub(&p.ctrl[BARQ_KV_CTRL_FREE_TOP], count);
      const int got = max(0, min(before, count));
      if (got < count) {
        atomicAdd(&p.ctrl[BARQ_KV_CTRL_FREE_TOP], count - got);
        err |= BARQ_KV_ERRBIT_POOL_EXHAUSTED;
      }
      s_base = before - got;  // pages [s_base, s_base + got) of the stack, the top one first
      s_hot[0] = got;         // read before the per-block entries below are written
    }
    __syncthreads();
    const int got = s_hot[0], base = s_base;
    __syncthreads();
    if (c >= 0) {
      s_block[k] = j;
      s_hot[k] = k < got ? checked_id(p.free_pages[base + got - 1 - k], p.num_pages) : -1;
      if (k < got && s_hot[k] < 0) err |= BARQ_KV_ERRBIT_BAD_INDEX;
    }
    __syncthreads();
    for (int q = 0; q < min(count, got); ++q) {
      const int jb = s_block[q], hp = s_hot[q];
      const int cp = -2 - row[jb];  // every thread reads the entry before thread 0 rewrites it
      __syncthreads();
      if (hp < 0) continue;  // uniform
      Bits* kp = (Bits*)p.key_pages + (int64_t)hp * P * HD;
      Bits* vp = (Bits*)p.value_pages + (int64_t)hp * P * HD;
      const uint8_t* kc = a.c.codes[0] + (int64_t)cp * P * HD;
      const uint8_t* vc = a.c.codes[1] + (int64_t)cp * P * HD;
      for (int i = threadIdx.x; i < P * HD; i += kThreads) {
        const int t = i / HD, hd = i - t * HD, h = hd / D;
        const int ek = (int)a.c.key_scales[(int64_t)cp * HD + hd] - 127;
        const int ev = (int)a.c.value_scales[((int64_t)cp * P + t) * H + h] - 127;
        kp[i] = E::from_float(ldexpf(e4m3_decode(kc[i]), ek));
        vp[i] = E::from_float(ldexpf(e4m3_decode(vc[i]), ev));
      }
      __syncthreads();  // the cold page is read in full before it can return to the stack
      if (threadIdx.x == 0) {
        row[jb] = hp;
        if (!a.c.shares || atomicSub(&a.c.shares[cp], 1) == 0) {
          if (a.c.shares) a.c.shares[cp] = 0;
          const int slot = atomicAdd(&p.ctrl[BARQ_KV_CTRL_COLD_TOP], 1);
          if (slot < a.c.num_cold) a.c.free_cold[slot] = cp;
          else err |= BARQ_KV_ERRBIT_BAD_INDEX;
        }
      }
    }
    __syncthreads();
  }
  __syncthreads();  // every thread has read the row's length before it is lowered
  if (threadIdx.x == 0 && r < a.batch) p.seq_lens[r] = len;
  if (err) atomicOr(&p.ctrl[BARQ_KV_CTRL_ERRORS], err);
}

// ---------------------------------------------------------------------------------------------
// Host side.
// ---------------------------------------------------------------------------------------------

bool pool_ok(const barq_kv_pool* p) {
  if (!p || !p->key_pages || !p->value_pages || !p->block_table || !p->seq_lens || !p->high_water ||
      !p->free_pages || !p->ctrl)
    return false;
  if (p->num_pages < 1 || p->num_pages > kI32Max || p->max_batch < 1 || p->max_batch > kI32Max ||
      p->max_blocks < 1 || p->page_size < 1 || p->kv_heads < 1 || p->head_dim < 1)
    return false;
  if (p->max_batch * p->max_blocks > kI32Max || p->max_blocks * p->page_size > kI32Max) return false;
  return p->elem_bytes == 2 || p->elem_bytes == 4;
}

bool cold_ok(const barq_kv_pool* p, const barq_kv_cold* c) {
  if (!pool_ok(p) || !c || !c->key_codes || !c->value_codes || !c->key_scales || !c->value_scales ||
      !c->free_cold)
    return false;
  if (c->num_cold < 1 || c->num_cold > kI32Max - 2 || c->window < 0 || c->window > kI32Max) return false;
  const int64_t want = c->element_type == BARQ_KV_FP32 ? 4 : 2;
  if (c->element_type < BARQ_KV_BF16 || c->element_type > BARQ_KV_FP32 || p->elem_bytes != want) return false;
  return p->page_size * p->kv_heads <= kMaxTokenHeads && p->kv_heads * p->head_dim <= kMaxChannels;
}

ColdPtrs cold_ptrs(const barq_kv_cold* c) {
  ColdPtrs r;
  r.codes[0] = (uint8_t*)c->key_codes;
  r.codes[1] = (uint8_t*)c->value_codes;
  r.key_scales = (uint8_t*)c->key_scales;
  r.value_scales = (uint8_t*)c->value_scales;
  r.free_cold = c->free_cold;
  r.shares = c->cold_shares;
  r.num_cold = c->num_cold;
  r.window = (int32_t)c->window;
  return r;
}

int launch(const void* fn, dim3 grid, void* arg, hipStream_t stream) {
  void* args[] = {arg};
  return hipLaunchKernel(fn, grid, dim3(kThreads), args, 0, stream) == hipSuccess ? BARQ_KV_OK
                                                                                 : BARQ_KV_ERR_LAUNCH;
}

template <int KIND>
const void* compress_fn_t(int ve) {
  if constexpr (KIND != BARQ_KV_FP32) {
    if (ve == 8) return (const void*)&compress_kernel<KIND, 8>;
  }
  switch (ve) {
    case 4: return (const void*)&compress_kernel<KIND, 4>;
    case 2: return (const void*)&compress_kernel<KIND, 2>;
    default: return (const void*)&compress_kernel<KIND, 1>;
  }
}

const void* compress_fn(int64_t kind, int ve) {
  return kind == BARQ_KV_BF16   ? compress_fn_t<BARQ_KV_BF16>(ve)
         : kind == BARQ_KV_FP16 ? compress_fn_t<BARQ_KV_FP16>(ve)
                                : compress_fn_t<BARQ_KV_FP32>(ve);
}

// How a compress takes a pool: vectors per lane of a unit (0: not at all) and the kind of units.
struct QuantUnits {
  int nv = 0, mode = kWholeUnit, log2 = 0;
};

template <int KIND>
const void* compress_blocks_fn_t(const QuantUnits& q) {
  if (q.mode == kSplitUnit) return (const void*)&compress_blocks_kernel<KIND, 8, kSplitUnit>;
  if (q.mode == kPackedUnit) return (const void*)&compress_blocks_kernel<KIND, 1, kPackedUnit>;
  switch (q.nv) {
    case 1: return (const void*)&compress_blocks_kernel<KIND, 1>;
    case 2: return (const void*)&compress_blocks_kernel<KIND, 2>;
    case 4: return (const void*)&compress_blocks_kernel<KIND, 4>;
    default: return (const void*)&compress_blocks_kernel<KIND, 8>;
  }
}

template <int KIND>
const void* quant_blocks_fn_t(int nv) {
  switch (nv) {
    case 1: return (const void*)&quant_blocks_kernel<KIND, 1>;
    case 2: return (const void*)&quant_blocks_kernel<KIND, 2>;
    case 4: return (const void*)&quant_blocks_kernel<KIND, 4>;
    default: return (const void*)&quant_blocks_kernel<KIND, 8>;
  }
}

// A compress takes head rows of a power of two of 16-byte vectors, up to a wave's 64, in pages of a power
// of two of tokens, every page, code and key-scale address aligned to its vector: a head's page of 1, 2,
// 4 or 8 waves' vectors as a unit, less than one wave's packed, 16 to 64 waves' split (K by columns, so
// a row has as many vectors as the head has units).
QuantUnits quant_units(const barq_kv_pool* p, const barq_kv_cold* c) {
  QuantUnits q;
  const int64_t ve = 16 / p->elem_bytes;
  const uint64_t bits = (uint64_t)(uintptr_t)p->key_pages | (uint64_t)(uintptr_t)p->value_pages;
  const uint64_t cbits = (uint64_t)(uintptr_t)c->key_codes | (uint64_t)(uintptr_t)c->value_codes |
                         (uint64_t)(uintptr_t)c->key_scales;
  if (p->head_dim % ve || (bits & 15) || (cbits & (uint64_t)(ve - 1))) return q;
  const int64_t vd = p->head_dim / ve, n = p->page_size * vd;
  if (vd > kWave || (vd & (vd - 1)) || (n & (n - 1)) || n > kWave * kWave || n > 8 * kWave * vd) return q;
  q.nv = (int)std::min<int64_t>(std::max<int64_t>(n / kWave, 1), 8);
  q.mode = n < kWave ? kPackedUnit : n > 8 * kWave ? kSplitUnit : kWholeUnit;
  if (q.mode == kPackedUnit) q.log2 = __builtin_ctzll((unsigned long long)n);
  if (q.mode == kSplitUnit) q.log2 = __builtin_ctzll((unsigned long long)(n / (8 * kWave)));
  return q;
}

// The vectors per lane where an append quantises from its input too: whole units only.
int quant_blocks_vectors(const barq_kv_pool* p, const barq_kv_cold* c) {
  const QuantUnits q = quant_units(p, c);
  return q.mode == kWholeUnit ? q.nv : 0;
}

// Quantises blocks of `batch` rows: behind an append of `tokens`, already committed, or for the rows'
// lengths `ahead` tokens on, in order or (whole units) spread.
int launch_quant_blocks(const barq_kv_pool* pool, const barq_kv_cold* cold, const QuantUnits& q, int64_t batch, int64_t tokens,
                        int64_t ahead, bool spread, const void* ks, const void* vs, int64_t sb, int64_t sh,
                        int64_t st, hipStream_t stream) {
  QuantArgs a;
  a.p = *pool;
  a.c = cold_ptrs(cold);
  a.in[0] = (const char*)ks;
  a.in[1] = (const char*)vs;
  a.isb = sb;
  a.ish = sh;
  a.ist = st;
  a.tokens = (int32_t)tokens;
  a.ahead = (int32_t)ahead;
  const int64_t P = pool->page_size;
  // `tokens` positions from anywhere in a block
  const int64_t nnew = tokens > 0 ? (tokens + P - 2) / P + 1 : 0;
  a.nnew = (int32_t)nnew;
  const int64_t vd = pool->head_dim * pool->elem_bytes / 16;
  a.vd_log2 = __builtin_ctzll((unsigned long long)vd);
  a.mode_log2 = q.log2;
  a.div_page = FastDiv::make((uint32_t)P);
  a.div_tiles = FastDiv::make((uint32_t)(nnew + kOldTiles));
  const bool tiled = tokens > 0 || (spread && q.mode == kWholeUnit);
  const int64_t tiles = tiled ? batch * (nnew + kOldTiles) : batch;
  if (tiles > kI32Max) return BARQ_KV_ERR_INVALID;
  const auto fn_of = [&](auto kind) {
    return tiled ? quant_blocks_fn_t<decltype(kind)::value>(q.nv) : compress_blocks_fn_t<decltype(kind)::value>(q);
  };
  const void* fn = cold->element_type == BARQ_KV_BF16   ? fn_of(std::integral_constant<int, BARQ_KV_BF16>{})
                   : cold->element_type == BARQ_KV_FP16 ? fn_of(std::integral_constant<int, BARQ_KV_FP16>{})
                                                        : fn_of(std::integral_constant<int, BARQ_KV_FP32>{});
  const int64_t H = pool->kv_heads, packed = q.mode == kPackedUnit ? kWave >> q.log2 : 1;
  const int threads = kWave * (int)std::min<int64_t>(16, 2 * (q.mode == kSplitUnit ? H << q.log2 : (H + packed - 1) / packed));
  void* args[] = {&a};
  return hipLaunchKernel(fn, dim3((uint32_t)tiles), dim3((uint32_t)threads), args, 0, stream) == hipSuccess
             ? BARQ_KV_OK
             : BARQ_KV_ERR_LAUNCH;
}

template <int KIND>
const void* fresh_blocks_fn_t(int nv) {
  switch (nv) {
    case 1: return (const void*)&fresh_blocks_kernel<KIND, 1>;
    case 2: return (const void*)&fresh_blocks_kernel<KIND, 2>;
    case 4: return (const void*)&fresh_blocks_kernel<KIND, 4>;
    default: return (const void*)&fresh_blocks_kernel<KIND, 8>;
  }
}

template <int KIND>
const void* update_fn_t(int lpp, bool known) {
  if (known)
    return lpp == 1   ? (const void*)&update_cold_known_kernel<KIND, 1>
           : lpp == 2 ? (const void*)&update_cold_known_kernel<KIND, 2>
                      : (const void*)&update_cold_known_kernel<KIND, 4>;
  return lpp == 1   ? (const void*)&update_cold_lanes_kernel<KIND, 1>
         : lpp == 2 ? (const void*)&update_cold_lanes_kernel<KIND, 2>
                    : (const void*)&update_cold_lanes_kernel<KIND, 4>;
}

template <int KIND>
int launch_gather(int ve, int lpp, dim3 grid, GatherArgs* a, hipStream_t s) {
  const void* fn = (const void*)&gather_cold_kernel<KIND, 1>;
  if constexpr (KIND != BARQ_KV_FP32) {  // 8 two-byte elements: a 16-byte vector
    if (ve == 8) fn = (const void*)&gather_cold_kernel<KIND, 8>;
    if (ve == 8 && lpp == 1) fn = (const void*)&gather_cold_lanes_kernel<KIND, 1>;
    if (ve == 8 && lpp == 2) fn = (const void*)&gather_cold_lanes_kernel<KIND, 2>;
    if (ve == 8 && lpp == 4) fn = (const void*)&gather_cold_lanes_kernel<KIND, 4>;
  }
  if (ve == 4) fn = (const void*)&gather_cold_kernel<KIND, 4>;
  if (ve == 2) fn = (const void*)&gather_cold_kernel<KIND, 2>;
  void* args[] = {a};
  return hipLaunchKernel(fn, grid, dim3(kGatherThreads), args, 0, s) == hipSuccess ? BARQ_KV_OK : BARQ_KV_ERR_LAUNCH;
}

}  // namespace

extern "C" {

int barq_kv_cold_reset(const barq_kv_pool* pool, const barq_kv_cold* cold, void* stream) {
  if (!cold_ok(pool, cold)) return BARQ_KV_ERR_INVALID;
  const int64_t blocks = (cold->num_cold + kThreads - 1) / kThreads;
  hipLaunchKernelGGL(cold_reset_kernel, dim3((uint32_t)blocks), dim3(kThreads), 0, (hipStream_t)stream,
                     cold_ptrs(cold), pool->ctrl);
  return hipGetLastError() == hipSuccess ? BARQ_KV_OK : BARQ_KV_ERR_LAUNCH;
}

}  // extern "C"

namespace {

// barq_kv_compress for the lengths the rows [0, batch) will have after `ahead` more tokens; spread: the
// caller has counted enough cold pages.
int compress_launch(const barq_kv_pool* pool, const barq_kv_cold* cold, int64_t batch, int64_t ahead, bool spread,
                    void* stream) {
  if (!cold_ok(pool, cold) || batch < 0 || batch > pool->max_batch) return BARQ_KV_ERR_INVALID;
  if (batch == 0) return BARQ_KV_OK;
  if (const QuantUnits q = quant_units(pool, cold); q.nv)
    return launch_quant_blocks(pool, cold, q, batch, 0, ahead, spread, nullptr, nullptr, 0, 0, 0, (hipStream_t)stream);
  CompressArgs a;
  a.p = *pool;
  a.c = cold_ptrs(cold);
  a.batch = (int32_t)batch;
  a.ahead = (int32_t)ahead;
  a.div_page = FastDiv::make((uint32_t)pool->page_size);
  a.div_dim = FastDiv::make((uint32_t)pool->head_dim);
  // widest vector along head_dim that every page row, code row and scale row admits
  const int64_t eb = pool->elem_bytes, D = pool->head_dim;
  const uint64_t bits = (uint64_t)(uintptr_t)pool->key_pages | (uint64_t)(uintptr_t)pool->value_pages;
  const uint64_t cbits = (uint64_t)(uintptr_t)cold->key_codes | (uint64_t)(uintptr_t)cold->value_codes |
                         (uint64_t)(uintptr_t)cold->key_scales;
  int ve = eb == 2 ? 8 : 4;
  while (ve > 1 && (D % ve || (bits & (uint64_t)(ve * eb - 1)) || (cbits & (uint64_t)(ve - 1)))) ve >>= 1;
  a.div_groups = FastDiv::make((uint32_t)(pool->kv_heads * D / ve));
  return launch(compress_fn(cold->element_type, ve), dim3((uint32_t)batch), &a, (hipStream_t)stream);
}

// The update in two launches -- compress for the lengths the rows reach, then
// update_cold_lanes_kernel -- when it applies: tokens in [1, window], batch <= 64, two-byte
// elements whose token rows are 64, 128 or 256 vectors of 16 bytes, every address and stride
// 16-byte aligned (codes and key scales 8-byte), the output reaching the new tokens.  Returns -1
// (nothing launched) when it does not.
// Workgroups of a kGatherThreads-thread kernel resident at once on the current device (cached per
// slot and device; 0 when the runtime does not say).  Host threads may race on the cache, which
// only ever stores the one value a device gives.
int resident_tiles(const void* fn, int slot) {
  constexpr int kMaxDevices = 64;
  constexpr int kSlots = 12;
  static std::atomic<int> cached[kSlots][kMaxDevices];  // 0 = not queried yet
  int dev = 0;
  if (slot < 0 || slot >= kSlots || hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return 0;
  int v = cached[slot][dev].load(std::memory_order_relaxed);
  if (v == 0) {
    int per_cu = 0, cus = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, kGatherThreads, 0) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || per_cu <= 0 ||
        cus <= 0)
      return 0;
    v = per_cu * cus;
    cached[slot][dev].store(v, std::memory_order_relaxed);
  }
  return v;
}

// barq_kv_update_cold's BARQ_KV_QUANT_DIRECT append.
int append_direct(const barq_kv_pool* pool, const barq_kv_cold* cold, const void* key_states, const void* value_states,
                  int64_t batch, int64_t tokens, int64_t stride_b, int64_t stride_h, int64_t stride_t, void* stream) {
  if (!cold_ok(pool, cold) || batch < 0 || batch > pool->max_batch || tokens < 0) return BARQ_KV_ERR_INVALID;
  if (tokens > pool->max_blocks * pool->page_size) return BARQ_KV_ERR_INVALID;
  if (batch == 0 || tokens == 0) return BARQ_KV_OK;
  if (!key_states || !value_states || stride_b < 0 || stride_h < 0 || stride_t < 0) return BARQ_KV_ERR_INVALID;
  const int nv = quant_blocks_vectors(pool, cold);
  const int64_t eb = pool->elem_bytes;
  const uint64_t bits = (uint64_t)(uintptr_t)key_states | (uint64_t)(uintptr_t)value_states |
                        (uint64_t)(stride_b * eb) | (uint64_t)(stride_h * eb) | (uint64_t)(stride_t * eb);
  // lane offsets within a block of the input fit 32 bits
  if (nv == 0 || (bits & 15) || stride_t > kI32Max / (pool->page_size * eb)) return BARQ_KV_ERR_UNSUPPORTED;
  AppendPlanArgs a;
  a.p = *pool;
  a.c = cold_ptrs(cold);
  a.batch = (int32_t)batch;
  a.tokens = (int32_t)tokens;
  a.div_page = FastDiv::make((uint32_t)pool->page_size);
  void* args[] = {&a};
  if (hipLaunchKernel((const void*)&append_plan_kernel, dim3(1), dim3(kPlanThreads), args, 0,
                      (hipStream_t)stream) != hipSuccess)
    return BARQ_KV_ERR_LAUNCH;
  return launch_quant_blocks(pool, cold, QuantUnits{nv}, batch, tokens, 0, true, key_states, value_states, stride_b, stride_h, stride_t,
                             (hipStream_t)stream);
}

int update_cold_fused(const barq_kv_pool* pool, const barq_kv_cold* cold, const void* ks, const void* vs,
                      int64_t batch, int64_t tokens, int64_t sb, int64_t sh, int64_t st, void* ko, void* vo,
                      int64_t seq_out, int64_t osb, int64_t osh, int64_t oss, int64_t flags, void* stream,
                      const KnownRows* known = nullptr) {
  if (!cold_ok(pool, cold) || pool->elem_bytes != 2 || cold->element_type == BARQ_KV_FP32) return -1;
  if (batch < 1 || batch > kWave || batch > pool->max_batch || tokens < 1 || tokens > cold->window) return -1;
  const int64_t P = pool->page_size, H = pool->kv_heads, D = pool->head_dim;
  const int64_t cap = pool->max_blocks * P;
  if (seq_out < tokens || seq_out > cap) return -1;
  if (!ks || !vs || !ko || !vo || sb < 0 || sh < 0 || st < 0 || osb < 0 || osh < 0 || oss < 0) return -1;
  const uint64_t bits = (uint64_t)(uintptr_t)ko | (uint64_t)(uintptr_t)vo | (uint64_t)(osb * 2) |
                        (uint64_t)(osh * 2) | (uint64_t)(oss * 2) | (uint64_t)(D * 2) |
                        (uint64_t)(uintptr_t)pool->key_pages | (uint64_t)(uintptr_t)pool->value_pages |
                        (uint64_t)(uintptr_t)ks | (uint64_t)(uintptr_t)vs | (uint64_t)(sb * 2) |
                        (uint64_t)(sh * 2) | (uint64_t)(st * 2);
  const uint64_t code_bits = (uint64_t)(uintptr_t)cold->key_codes | (uint64_t)(uintptr_t)cold->value_codes |
                             (uint64_t)(uintptr_t)cold->key_scales | (uint64_t)D;
  if ((bits & 15) || (code_bits & 7)) return -1;
  const int64_t hd8 = H * D / 8;
  if (D % 8 != 0 || hd8 % kWave != 0 || (hd8 / kWave != 1 && hd8 / kWave != 2 && hd8 / kWave != 4) ||
      P * H * D > kI32Max)
    return -1;
  const int lpp = (int)(hd8 / kWave);
  if (!(flags & BARQ_KV_NO_COMPRESS)) {
    const int rc = compress_launch(pool, cold, batch, tokens, false, stream);
    if (rc != BARQ_KV_OK) return rc;
  }
  UpdateArgs u;
  GatherArgs& a = u.g;
  a.p = *pool;
  a.c = cold_ptrs(cold);
  a.out[0] = (char*)ko;
  a.out[1] = (char*)vo;
  a.osb = osb;
  a.osh = osh;
  a.oss = oss;
  a.batch = (int32_t)batch;
  a.seq_out = (int32_t)seq_out;
  a.nblk = (int32_t)((seq_out + P - 1) / P);
  a.from_device = (flags & BARQ_KV_SEQ_FROM_DEVICE) ? 1 : 0;
  a.div_head = FastDiv::make((uint32_t)(P * (D / 8)));
  a.div_dv = FastDiv::make((uint32_t)(D / 8));
  a.div_nblk = FastDiv::make((uint32_t)a.nblk);
  u.in[0] = (const char*)ks;
  u.in[1] = (const char*)vs;
  u.isb = sb;
  u.ish = sh;
  u.ist = st;
  u.tokens = (int32_t)tokens;
  const int64_t tiles = batch * a.nblk * 2;
  u.nsub = (int32_t)std::min<int64_t>(tiles, BARQ_KV_CTRL_SUBCOUNTERS);
  u.div_page = FastDiv::make((uint32_t)P);
  const bool f16 = cold->element_type == BARQ_KV_FP16;
  const void* fn = f16 ? update_fn_t<BARQ_KV_FP16>(lpp, known != nullptr) : update_fn_t<BARQ_KV_BF16>(lpp, known != nullptr);
  const int64_t resident = resident_tiles(fn, ((lpp == 1 ? 0 : lpp == 2 ? 1 : 2) * 2 + (f16 ? 1 : 0)) * 2 + (known ? 1 : 0));
  u.spaced = resident > 0 && tiles <= resident ? 1 : 0;
  KnownRows rows{};
  if (known) rows = *known;
  void* args[] = {&u, &rows};
  return hipLaunchKernel(fn, dim3((uint32_t)tiles), dim3(kGatherThreads), args, 0, (hipStream_t)stream) == hipSuccess
             ? BARQ_KV_OK
             : BARQ_KV_ERR_LAUNCH;
}

}  // namespace

extern "C" {

int barq_kv_compress(const barq_kv_pool* pool, const barq_kv_cold* cold, int64_t batch, void* stream) {
  return compress_launch(pool, cold, batch, 0, false, stream);
}

int barq_kv_gather_cold(const barq_kv_pool* pool, const barq_kv_cold* cold, void* key_out,
                        void* value_out, int64_t batch, int64_t seq_out, int64_t osb, int64_t osh,
                        int64_t oss, int64_t flags, void* stream) {
  if (!cold_ok(pool, cold) || batch < 0 || batch > pool->max_batch) return BARQ_KV_ERR_INVALID;
  if (flags & ~(int64_t)BARQ_KV_SEQ_FROM_DEVICE) return BARQ_KV_ERR_INVALID;
  const int64_t cap = pool->max_blocks * pool->page_size;
  if (seq_out < 0 || seq_out > cap) return BARQ_KV_ERR_INVALID;
  if (batch == 0 || seq_out == 0) return BARQ_KV_OK;
  if (!key_out || !value_out || osb < 0 || osh < 0 || oss < 0) return BARQ_KV_ERR_INVALID;
  const int64_t eb = pool->elem_bytes, D = pool->head_dim;
  // widest vector of VE elements every address and stride admits
  const uint64_t bits = (uint64_t)(uintptr_t)key_out | (uint64_t)(uintptr_t)value_out | (uint64_t)(osb * eb) |
                        (uint64_t)(osh * eb) | (uint64_t)(oss * eb) | (uint64_t)(D * eb) |
                        (uint64_t)(uintptr_t)pool->key_pages | (uint64_t)(uintptr_t)pool->value_pages;
  const uint64_t code_bits = (uint64_t)(uintptr_t)cold->key_codes | (uint64_t)(uintptr_t)cold->value_codes |
                             (uint64_t)(uintptr_t)cold->key_scales | (uint64_t)D;
  int ve = eb == 2 ? 8 : 4;
  while (ve > 1 && ((bits & (uint64_t)(ve * eb - 1)) || (code_bits & (uint64_t)(ve - 1)))) ve >>= 1;
  GatherArgs a;
  a.p = *pool;
  a.c = cold_ptrs(cold);
  a.out[0] = (char*)key_out;
  a.out[1] = (char*)value_out;
  a.osb = osb;
  a.osh = osh;
  a.oss = oss;
  a.batch = (int32_t)batch;
  a.seq_out = (int32_t)seq_out;
  a.nblk = (int32_t)((seq_out + pool->page_size - 1) / pool->page_size);
  a.from_device = (flags & BARQ_KV_SEQ_FROM_DEVICE) ? 1 : 0;
  a.div_head = FastDiv::make((uint32_t)(pool->page_size * (D / ve)));
  a.div_dv = FastDiv::make((uint32_t)(D / ve));
  a.div_nblk = FastDiv::make((uint32_t)a.nblk);
  const int64_t tiles = batch * a.nblk * 2;
  if (tiles > kI32Max) return BARQ_KV_ERR_INVALID;
  // Whole positions per wave: a token row of 64 * lpp vectors, and 32-bit offsets within a page
  const int64_t hd8 = pool->kv_heads * D / 8;
  const int lpp = (ve == 8 && D % 8 == 0 && hd8 % kWave == 0 &&
                   (hd8 / kWave == 1 || hd8 / kWave == 2 || hd8 / kWave == 4) &&
                   pool->page_size * pool->kv_heads * D <= kI32Max)
                      ? (int)(hd8 / kWave) : 0;
  hipStream_t s = (hipStream_t)stream;
  switch (cold->element_type) {
    case BARQ_KV_BF16: return launch_gather<BARQ_KV_BF16>(ve, lpp, dim3((uint32_t)tiles), &a, s);
    case BARQ_KV_FP16: return launch_gather<BARQ_KV_FP16>(ve, lpp, dim3((uint32_t)tiles), &a, s);
    default: return launch_gather<BARQ_KV_FP32>(ve, lpp, dim3((uint32_t)tiles), &a, s);
  }
}

int barq_kv_update_cold(const barq_kv_pool* pool, const barq_kv_cold* cold, const void* key_states,
                        const void* value_states, int64_t batch, int64_t tokens, int64_t stride_b,
                        int64_t stride_h, int64_t stride_t, void* key_out, void* value_out,
                        int64_t seq_out, int64_t osb, int64_t osh, int64_t oss, int64_t flags,
                        void* stream) {
  if (!cold_ok(pool, cold)) return BARQ_KV_ERR_INVALID;
  if (flags & ~(int64_t)(BARQ_KV_SEQ_FROM_DEVICE | BARQ_KV_NO_COMPRESS | BARQ_KV_QUANT_DIRECT)) return BARQ_KV_ERR_INVALID;
  if (flags & BARQ_KV_QUANT_DIRECT) {
    if (flags & BARQ_KV_NO_COMPRESS) return BARQ_KV_ERR_INVALID;
    if (seq_out < 0 || seq_out > pool->max_blocks * pool->page_size || (seq_out > 0 && (!key_out || !value_out)))
      return BARQ_KV_ERR_INVALID;
    const int rc = append_direct(pool, cold, key_states, value_states, batch, tokens, stride_b, stride_h, stride_t, stream);
    return rc != BARQ_KV_OK ? rc
                            : barq_kv_gather_cold(pool, cold, key_out, value_out, batch, seq_out, osb, osh, oss,
                                                  flags & BARQ_KV_SEQ_FROM_DEVICE, stream);
  }
  const int fused = update_cold_fused(pool, cold, key_states, value_states, batch, tokens, stride_b, stride_h,
                                      stride_t, key_out, value_out, seq_out, osb, osh, oss, flags, stream);
  if (fused >= 0) return fused;
  int rc = barq_kv_append(pool, key_states, value_states, batch, tokens, stride_b, stride_h, stride_t, stream);
  if (rc == BARQ_KV_OK && !(flags & BARQ_KV_NO_COMPRESS)) rc = barq_kv_compress(pool, cold, batch, stream);
  if (rc == BARQ_KV_OK)
    rc = barq_kv_gather_cold(pool, cold, key_out, value_out, batch, seq_out, osb, osh, oss,
                             flags & BARQ_KV_SEQ_FROM_DEVICE, stream);
  return rc;
}

int barq_kv_crop_cold(const barq_kv_pool* pool, const barq_kv_cold* cold, int64_t batch, int64_t max_length,
                      void* stream) {
  if (!cold_ok(pool, cold) || batch < 0 || batch > pool->max_batch) return BARQ_KV_ERR_INVALID;
  if (batch == 0) return BARQ_KV_OK;
  CropArgs a;
  a.p = *pool;
  a.c = cold_ptrs(cold);
  a.batch = (int32_t)batch;
  a.max_length = (int32_t)std::max<int64_t>(0, std::min<int64_t>(max_length, kI32Max));
  a.div_page = FastDiv::make((uint32_t)pool->page_size);
  const void* fn = cold->element_type == BARQ_KV_BF16   ? (const void*)&crop_cold_kernel<BARQ_KV_BF16>
                   : cold->element_type == BARQ_KV_FP16 ? (const void*)&crop_cold_kernel<BARQ_KV_FP16>
                                                        : (const void*)&crop_cold_kernel<BARQ_KV_FP32>;
  return launch(fn, dim3((uint32_t)batch), &a, (hipStream_t)stream);
}

int barq_kv_free_rows_cold(const barq_kv_pool* pool, const barq_kv_cold* cold, const int32_t* rows,
                           int64_t num_rows, void* stream) {
  if (!cold_ok(pool, cold) || num_rows < 0 || num_rows > pool->max_batch) return BARQ_KV_ERR_INVALID;
  if (num_rows == 0) return BARQ_KV_OK;
  if (!rows) return BARQ_KV_ERR_INVALID;
  FreeArgs a;
  a.p = *pool;
  a.c = cold_ptrs(cold);
  a.rows = rows;
  a.n = (int32_t)num_rows;
  a.div_page = FastDiv::make((uint32_t)pool->page_size);
  return launch((const void*)&free_rows_cold_kernel, dim3(1), &a, (hipStream_t)stream);
}

}  // extern "C"

namespace barq_internal {

int append_fresh_cold(const barq_kv_pool* pool, const barq_kv_cold* cold, const void* key_states,
                      const void* value_states, int64_t batch, int64_t tokens, int64_t stride_b, int64_t stride_h,
                      int64_t stride_t, void* key_out, void* value_out, int64_t osb, int64_t osh, int64_t oss,
                      int64_t free_top, int64_t cold_top, void* stream) {
  if (!cold_ok(pool, cold) || batch < 1 || batch > pool->max_batch || tokens < 1 || !key_states || !value_states ||
      stride_b < 0 || stride_h < 0 || stride_t < 0 || osb < 0 || osh < 0 || oss < 0 || !key_out != !value_out)
    return BARQ_KV_ERR_INVALID;
  const int64_t P = pool->page_size, eb = pool->elem_bytes;
  const int nv = quant_blocks_vectors(pool, cold);
  uint64_t bits = (uint64_t)(uintptr_t)key_states | (uint64_t)(uintptr_t)value_states | (uint64_t)(stride_b * eb) |
                  (uint64_t)(stride_h * eb) | (uint64_t)(stride_t * eb);
  if (key_out)
    bits |= (uint64_t)(uintptr_t)key_out | (uint64_t)(uintptr_t)value_out | (uint64_t)(osb * eb) |
            (uint64_t)(osh * eb) | (uint64_t)(oss * eb);
  // lane offsets within a block of the states and of the output fit 32 bits
  if (nv == 0 || (bits & 15) || std::max(stride_t, oss) > kI32Max / (P * eb)) return BARQ_KV_ERR_UNSUPPORTED;
  const int64_t nblk = (tokens + P - 1) / P;
  const int64_t ncold = std::max<int64_t>(tokens - cold->window, 0) / P;
  const int64_t groups = (2 * pool->kv_heads + kFreshWaves - 1) / kFreshWaves;
  // What a caller's count could get wrong is left to the path that reads the stacks' tops.
  if (nblk > pool->max_blocks || cold_top > cold->num_cold || free_top > pool->num_pages ||
      batch * ncold > cold_top || batch * (nblk - ncold) > free_top || batch * nblk * groups > kI32Max)
    return BARQ_KV_ERR_UNSUPPORTED;
  FreshArgs f;
  QuantArgs& a = f.q;
  a.p = *pool;
  a.c = cold_ptrs(cold);
  a.in[0] = (const char*)key_states;
  a.in[1] = (const char*)value_states;
  a.isb = stride_b;
  a.ish = stride_h;
  a.ist = stride_t;
  a.tokens = (int32_t)tokens;
  a.ahead = 0;
  a.nnew = (int32_t)nblk;
  a.vd_log2 = __builtin_ctzll((unsigned long long)(pool->head_dim * eb / 16));
  a.mode_log2 = 0;
  a.div_page = FastDiv::make((uint32_t)P);
  a.div_tiles = FastDiv::make((uint32_t)nblk);
  f.out[0] = (char*)key_out;
  f.out[1] = (char*)value_out;
  f.osb = osb;
  f.osh = osh;
  f.oss = (uint32_t)oss;
  f.ncold = (int32_t)ncold;
  f.nblk = (int32_t)nblk;
  f.top = (int32_t)free_top;
  f.ctop = (int32_t)cold_top;
  f.div_groups = FastDiv::make((uint32_t)groups);
  f.div_nblk = FastDiv::make((uint32_t)nblk);
  const void* fn = cold->element_type == BARQ_KV_BF16   ? fresh_blocks_fn_t<BARQ_KV_BF16>(nv)
                   : cold->element_type == BARQ_KV_FP16 ? fresh_blocks_fn_t<BARQ_KV_FP16>(nv)
                                                        : fresh_blocks_fn_t<BARQ_KV_FP32>(nv);
  void* args[] = {&f};
  return hipLaunchKernel(fn, dim3((uint32_t)(batch * nblk * groups)), dim3(kFreshWaves * kWave), args, 0,
                         (hipStream_t)stream) == hipSuccess
             ? BARQ_KV_OK
             : BARQ_KV_ERR_LAUNCH;
}

int compress_spread(const barq_kv_pool* pool, const barq_kv_cold* cold, int64_t batch, int64_t ahead, void* stream) {
  return compress_launch(pool, cold, batch, ahead, true, stream);
}

int update_cold_known(const barq_kv_pool* pool, const barq_kv_cold* cold, const void* ks, const void* vs, int64_t batch,
                      int64_t tokens, int64_t sb, int64_t sh, int64_t st, void* ko, void* vo, int64_t seq_out,
                      int64_t osb, int64_t osh, int64_t oss, int64_t flags, const int32_t* seq_lens,
                      const int32_t* high_water, int64_t free_top, void* stream) {
  if ((flags & ~(int64_t)BARQ_KV_NO_COMPRESS) || !seq_lens || !high_water) return BARQ_KV_ERR_INVALID;
  if (batch < 1 || batch > kWave) return BARQ_KV_ERR_UNSUPPORTED;
  if (!pool || free_top < 0 || free_top > pool->num_pages) return BARQ_KV_ERR_INVALID;
  KnownRows rows{};
  for (int64_t r = 0; r < batch; ++r) {
    rows.len[r] = seq_lens[r];
    rows.hw[r] = high_water[r];
    if (rows.len[r] < 0 || rows.hw[r] < rows.len[r]) return BARQ_KV_ERR_INVALID;
  }
  rows.top = (int32_t)free_top;
  const int rc = update_cold_fused(pool, cold, ks, vs, batch, tokens, sb, sh, st, ko, vo, seq_out, osb, osh, oss, flags,
                                   stream, &rows);
  return rc < 0 ? BARQ_KV_ERR_UNSUPPORTED : rc;
}

}  // namespace barq_internal
