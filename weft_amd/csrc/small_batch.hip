// Small-batch mul_mat: 2 .. 64 activation rows against every weight format
// (the same products as the GEMVs and the prefill GEMMs; formats and GGML
// line numbers in decode_staged.hip and decode_q4k.hip), any number of rows
// where no prefill GEMM takes the weights, and up to 64 of MUL_MAT_ID's pairs
// grouped by expert.
//
// What bounds it: one read of the weights, and the latency of that one read.
// The GEMVs walk a batch four activation rows at a time and pay eight v_dot4
// per 32 weights and row; the prefill GEMMs' 64 x 128 tiles leave most CUs
// idle below a few hundred rows (N = 4096: 32 workgroups).  Here a workgroup
// takes 16 weight rows and up to 32 tokens, its waves split K, and each wave's
// products run on
// v_mfma_i32_16x16x32_i8: one instruction per 32-value block for 16 rows x
// 16 tokens, whatever the batch.  A block's scale is applied to its 16 x 16
// product on VALU (4 values per lane), so the arithmetic per weight hardly
// grows with the batch.
//
// A wave walks units of 256 values: it reads the rows' and the tokens' record
// bytes of the unit as 16-byte chunks, adjacent lanes adjacent chunks (an
// operand-shaped read, 16 rows by 8 bytes, costs the address unit a cache
// line per lane), the next unit's while it computes one, and stages them in
// its own LDS region, from which the operands come at constant offsets.  Records of any alignment are
// read with unaligned loads; what is left of a record past its whole chunks
// comes as a field of its own, so nothing outside the records is read.  No
// barrier until the end, where the waves' partial sums meet in LDS in wave
// order, so an output does not depend on timing.  Operand layout: lane l
// holds weight row l % 16 (the MFMA's column) and k = 8 (l / 16) .. + 7 of
// the block; its products are tokens 4 (l / 16) .. + 3 of that row, so the
// row's scales are per lane and the tokens' scales are broadcast reads.
//
// MUL_MAT_ID with up to 64 (token, slot) pairs: the same kernel, a workgroup
// per weight tile and pair that groups the pairs of one expert itself.
//
// The activation is quantized into Xq (GGML's records) by the format's
// quantize kernel first and read from L2 as records.
#include <algorithm>
#include <type_traits>

#include "kernels.h"
#include "runtime.h"
#include "weft_common.h"

namespace weft {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

// as decode_quantized's format codes, and Q4_K
enum class SF { Q4_0, MXFP4, IQ2_XXS, Q6_K, Q5_K, NVFP4, Q4_1, IQ2_XS, Q4_K };

enum class Act { Q8_0, Q8_1, Q8_K };

template <SF F>
struct Traits {
  // bytes of 256 weights; the activation's records; alignment of a record
  static constexpr int kUnit = F == SF::Q4_0      ? 8 * kQ4_0Bytes
                               : F == SF::MXFP4   ? 8 * kMxfp4Bytes
                               : F == SF::IQ2_XXS ? kIq2xxsBytes
                               : F == SF::Q6_K    ? kQ6_KBytes
                               : F == SF::Q5_K    ? kQ5_KBytes
                               : F == SF::NVFP4   ? 4 * kNvfp4Bytes
                               : F == SF::Q4_1    ? 8 * kQ4_1Bytes
                               : F == SF::IQ2_XS  ? kIq2xsBytes
                                                  : kQ4_KBytes;
  static constexpr Act kAct = F == SF::Q4_0 || F == SF::MXFP4 || F == SF::NVFP4 ? Act::Q8_0
                              : F == SF::Q4_1                                   ? Act::Q8_1
                                                                                : Act::Q8_K;
  static constexpr bool kQ8K = kAct == Act::Q8_K;
  static constexpr int kElems = kQ8K ? 256 : F == SF::NVFP4 ? 64 : 32;       // values per record
  static constexpr int kRec = kUnit / (256 / kElems);                         // bytes per record
  static constexpr int kXRec = kQ8K ? kQ8_KBytes : kAct == Act::Q8_1 ? kQ8_1Bytes : kQ8_0Bytes;
  // a unit's bytes [kHead, kHead + 16 kChunks) are copied as chunks; the rest
  // is one field of kExt bytes at kExtAt (Q6_K's d, MXFP4's last 8 codes,
  // IQ2's d; IQ2_XS has its 8 scales besides)
  static constexpr bool kIq2 = F == SF::IQ2_XXS || F == SF::IQ2_XS;
  static constexpr int kHead = kIq2 ? 2 : 0;
  static constexpr int kChunks = (F == SF::IQ2_XS ? 64 : kUnit - kHead) / 16;
  static constexpr int kExt = F == SF::MXFP4 ? 8 : F == SF::Q6_K || kIq2 ? 2 : 0;
  static constexpr int kExtAt = F == SF::MXFP4 ? 128 : F == SF::Q6_K ? 208 : 0;
  static constexpr int kExt2 = F == SF::IQ2_XS ? 8 : 0;
  static_assert(kHead + 16 * kChunks + kExt2 + (kIq2 ? 0 : kExt) == kUnit, "the unit is chunks and fields");
  // LDS bytes per row: the chunks at an odd number of 16 bytes (16 rows'
  // reads at one offset then fall on distinct banks)
  static constexpr int kPitch = 16 * (kChunks | 1);
  // a token's unit: Q8_K without its d (a field of its own), whole records
  static constexpr int kXUnit = kQ8K ? kQ8_KBytes : 8 * kXRec;  // 292, 272, 288
  static constexpr int kXHead = kQ8K ? 4 : 0;
  static constexpr int kXChunks = (kXUnit - kXHead) / 16;       // 18, 17, 18
  static constexpr int kXPitch = 16 * (kXChunks | 1);
  static_assert(kXHead + 16 * kXChunks == kXUnit, "a token's unit is whole chunks");
  static constexpr bool kTable = F == SF::MXFP4 || F == SF::NVFP4;
  static constexpr int kGridWords = F == SF::IQ2_XS ? 1024 : 512;
  static constexpr int kTableBytes = kIq2 ? 4 * kGridWords + 2048 : kTable ? 1024 : 0;
};

struct Args {
  const uint8_t* W;
  const uint8_t* Xq;
  const int8_t* tab0;  // IQ2 grid, MXFP4 / NVFP4 codebook
  const void* tab1;    // IQ2 signs, MXFP4 / NVFP4 scale table
  float* Y;
  int N, K, M;
  int mtiles;       // dense: token tiles
  uint32_t ldw;     // bytes between weight rows (24 bits)
  long long ldy;    // floats between output rows
  PairArgs pair;    // MUL_MAT_ID mode: at most 64 pairs
  int n_pairs;
  bool wide;        // Xq is the caller's own
};

// chunk loads per lane of 16 rows
constexpr int loads_per_lane(int chunks) { return (16 * chunks + kWave - 1) / kWave; }

// bytes of one wave's LDS: one weight tile's window (with slack for the last
// dword of a run) and its fields, the tokens' records, and their scales as
// floats (Q8_K: one a unit; else one a block, Q8_1: block sums too)
template <SF F>
constexpr int w_lds() {
  using T = Traits<F>;
  return 16 * T::kPitch + 16 + (T::kExt + T::kExt2 ? 16 * 16 : 0);
}
template <SF F, int MT>
constexpr int wave_lds() {
  using T = Traits<F>;
  return w_lds<F>() + 16 * MT * T::kXPitch + (T::kQ8K ? 64 * MT : 512 * MT * (T::kAct == Act::Q8_1 ? 2 : 1));
}
// waves of a workgroup, at most: 16 leave a lane 128 registers, which two
// token tiles do not fit
template <int MT>
constexpr int max_waves() {
  return MT == 1 ? 16 : 8;
}

// c / d for c < 1024 in full-rate 24-bit arithmetic (the 32-bit products of a
// general division run at a quarter of it)
template <int d>
__device__ __forceinline__ uint32_t small_div(uint32_t c) {
  return __umul24(c, 65536 / d + 1) >> 16;
}

// n dwords at LDS byte o + off (o a multiple of 4, off any constant)
template <int off, int n>
__device__ __forceinline__ void run(const char* base, int o, uint32_t (&v)[n]) {
  constexpr int sh = off & 3;
  const uint32_t* w = reinterpret_cast<const uint32_t*>(base + o + (off - sh));
  if constexpr (sh == 0) {
#pragma unroll
    for (int i = 0; i < n; ++i) v[i] = w[i];
  } else {
    uint32_t t[n + 1];
#pragma unroll
    for (int i = 0; i <= n; ++i) t[i] = w[i];
#pragma unroll
    for (int i = 0; i < n; ++i) v[i] = __builtin_amdgcn_alignbyte(t[i + 1], t[i], sh);
  }
}
// the u16 / byte at LDS byte o + off
__device__ __forceinline__ uint32_t half_at(const char* base, int o) {
  return *reinterpret_cast<const uint16_t*>(base + o);
}
__device__ __forceinline__ uint32_t byte_at(const char* base, int o) {
  return *reinterpret_cast<const uint8_t*>(base + o);
}

__device__ __forceinline__ long pack(uint32_t lo, uint32_t hi) { return (long)(((uint64_t)hi << 32) | lo); }

// 16 bytes of global memory at any address
struct __attribute__((packed, aligned(1))) Chunk {
  uint32_t w[4];
};
__device__ __forceinline__ uint4 load_chunk(const uint8_t* p) {
  const Chunk c = *reinterpret_cast<const Chunk*>(p);
  return make_uint4(c.w[0], c.w[1], c.w[2], c.w[3]);
}
__device__ __forceinline__ uint32_t load_half(const uint8_t* p) {
  struct __attribute__((packed, aligned(1))) H {
    uint16_t v;
  };
  return reinterpret_cast<const H*>(p)->v;
}
__device__ __forceinline__ void load_8(const uint8_t* p, uint32_t& lo, uint32_t& hi) {
  struct __attribute__((packed, aligned(1))) D {
    uint32_t lo, hi;
  };
  const D d = *reinterpret_cast<const D*>(p);
  lo = d.lo;
  hi = d.hi;
}

// bytewise a - 8 for nibbles, no borrow between bytes
__device__ __forceinline__ uint32_t minus8(uint32_t a) { return ((a | 0x80808080u) - 0x08080808u) ^ 0x80808080u; }

// four nibbles (one per byte) -> bytes of the 16-entry codebook c
__device__ __forceinline__ uint32_t lookup(uint32_t n, const uint32_t (&c)[4]) {
  const uint32_t sel = n & 0x07070707u;
  const uint32_t lo = __builtin_amdgcn_perm(c[1], c[0], sel);
  const uint32_t hi = __builtin_amdgcn_perm(c[3], c[2], sel);
  // byte i of lo or hi by the code's bit 3
  return __builtin_amdgcn_perm(hi, lo, 0x03020100u | ((n >> 1) & 0x04040404u));
}

__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// What every row's decode shares: the lane's operand part, the codebook, the
// IQ2 tables (entry picks the lane's 8 weights of a grid and sign row).
struct Shared {
  int q;
  uint32_t cb[4];
  const char* tables;
  const uint2 *grid, *sgn;
  bool canon;

  __device__ __forceinline__ void entry(uint32_t gi, uint32_t si, uint32_t& w0, uint32_t& w1) const {
    const uint2 g = grid[gi], m = sgn[si];
    w0 = (g.x ^ m.x) + (m.x & 0x01010101u);
    w1 = (g.y ^ m.y) + (m.y & 0x01010101u);
    if (!canon) {
      // a scalar branch the compiler keeps (selects would carry both forms)
      w0 = mul8x4(g.x, m.x);
      w1 = mul8x4(g.y, m.y);
      asm volatile("" : "+v"(w0), "+v"(w1));
    }
  }
};

// One weight row's unit in LDS (chunks at byte o of win, fields at ext) as
// this lane reads it: begin() takes the unit's header and fields, block<s>() the lane's 8 weights of block s
// as int8 and the block's scales (c0 of its first 16 values, c1 of the last
// 16 where the format has two).
template <SF F>
struct Row {
  float dw = 0.f, dmin = 0.f;
  uint32_t h[4], hx[4], b[4];
  uint32_t mn03, mn47;

  __device__ __forceinline__ void begin(const char* win, int o, const char* ext, const Shared& sh) {
    if constexpr (F == SF::Q4_K || F == SF::Q5_K) {
      run<0>(win, o, h);
      dw = fp16_to_fp32(h[0] & 0xffffu);
      dmin = fp16_to_fp32(h[0] >> 16);
      mn03 = h[2] & 0x3f3f3f3fu;
      mn47 = ((h[3] >> 4) & 0x0f0f0f0fu) | (((h[2] >> 6) & 0x03030303u) << 4);
      h[3] = (h[3] & 0x0f0f0f0fu) | (((h[1] >> 6) & 0x03030303u) << 4);  // scales 4 .. 7
      h[1] &= 0x3f3f3f3fu;                                              // scales 0 .. 3
      if constexpr (F == SF::Q5_K) {
        uint32_t t[2];
        run<16>(win, o + 8 * sh.q, t);
        hx[0] = t[0];
        hx[1] = t[1];
      }
    } else if constexpr (F == SF::Q6_K) {
      run<192>(win, o, h);
      dw = fp16_to_fp32(half_at(ext, 0));
    } else if constexpr (F == SF::IQ2_XXS || F == SF::IQ2_XS) {
      dw = 0.125f * fp16_to_fp32(half_at(ext, 0));
      if constexpr (F == SF::IQ2_XS) {
        uint32_t t[2];
        run<8>(ext, 0, t);
        hx[0] = t[0];
        hx[1] = t[1];
      }
    } else if constexpr (F == SF::MXFP4) {
      uint32_t t[2];
      run<0>(ext, 0, t);
      hx[0] = t[0];
      hx[1] = t[1];
    }
  }

  template <int s>
  __device__ __forceinline__ void block(const char* win, int o, const Shared& sh, uint32_t& w0, uint32_t& w1, int& c0,
                                        int& c1, float& f0, float& f1) {
    const int q = sh.q;
    if constexpr (F == SF::Q4_K || F == SF::Q5_K) {
      if constexpr (s % 2 == 0) {
        uint32_t t[2];
        run<(F == SF::Q5_K ? 48 : 16) + 16 * s>(win, o + 8 * q, t);
        b[0] = t[0];
        b[1] = t[1];
      }
      w0 = (b[0] >> (4 * (s & 1))) & 0x0f0f0f0fu;
      w1 = (b[1] >> (4 * (s & 1))) & 0x0f0f0f0fu;
      if constexpr (F == SF::Q5_K) {
        w0 |= ((hx[0] >> s) & 0x01010101u) << 4;
        w1 |= ((hx[1] >> s) & 0x01010101u) << 4;
      }
      c0 = (int)((h[s < 4 ? 1 : 3] >> (8 * (s & 3))) & 63u);
    } else if constexpr (F == SF::Q6_K) {
      constexpr int hf = s / 4, j = s % 4;
      if constexpr (j == 0) {
        uint32_t t[2];
        run<64 * hf>(win, o + 8 * q, t);
        b[0] = t[0];
        b[1] = t[1];
        run<64 * hf + 32>(win, o + 8 * q, t);
        b[2] = t[0];
        b[3] = t[1];
        run<128 + 32 * hf>(win, o + 8 * q, t);
        hx[0] = t[0];
        hx[1] = t[1];
      }
      uint32_t w[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const uint32_t lo = (b[2 * (j & 1) + i] >> (4 * (j >> 1))) & 0x0f0f0f0fu;
        const uint32_t hi = ((hx[i] >> (2 * j)) & 0x03030303u) << 4;
        w[i] = (((lo | hi) | 0x80808080u) - 0x20202020u) ^ 0x80808080u;  // q6 - 32
      }
      w0 = w[0];
      w1 = w[1];
      const uint32_t s2 = h[2 * hf + (j >> 1)] >> (16 * (j & 1));
      c0 = (int)(int8_t)(s2 & 0xffu);
      c1 = (int)(int8_t)((s2 >> 8) & 0xffu);
    } else if constexpr (F == SF::IQ2_XXS) {
      uint32_t t[2];
      run<8 * s>(win, o, t);
      sh.entry((t[0] >> (8 * q)) & 0xffu, (t[1] >> (7 * q)) & 127u, w0, w1);
      c0 = 2 * (int)(t[1] >> 28) + 1;
    } else if constexpr (F == SF::IQ2_XS) {
      const uint32_t e = half_at(win, o + 8 * s + 2 * q), sc = (hx[s / 4] >> (8 * (s % 4))) & 0xffu;
      sh.entry(e & 511u, e >> 9, w0, w1);
      c0 = 2 * (int)(sc & 15u) + 1;
      c1 = 2 * (int)(sc >> 4) + 1;
    } else if constexpr (F == SF::NVFP4) {
      uint32_t t[2];
      run<36 * (s / 2) + 4 + 16 * (s & 1)>(win, o + 8 * (q >> 1), t);
      w0 = lookup(t[0] >> (4 * (q & 1)), sh.cb);
      w1 = lookup(t[1] >> (4 * (q & 1)), sh.cb);
      const uint32_t e = half_at(win, o + 36 * (s / 2) + 2 * (s & 1));
      f0 = reinterpret_cast<const float*>(sh.tables)[e & 0xffu];
      f1 = reinterpret_cast<const float*>(sh.tables)[e >> 8];
    } else {
      constexpr int rec = Traits<F>::kRec, at = rec * s;
      uint32_t t[2];
      if constexpr (F == SF::MXFP4 && s == 7) {
        run<at + rec - 16>(win, o, t);  // the first 8 code bytes; the last 8 are the field
        t[0] = q & 1 ? hx[0] : t[0];
        t[1] = q & 1 ? hx[1] : t[1];
      } else {
        run<at + rec - 16>(win, o + 8 * (q & 1), t);
      }
      w0 = t[0] >> (4 * (q >> 1));
      w1 = t[1] >> (4 * (q >> 1));
      if constexpr (F == SF::MXFP4) {
        w0 = lookup(w0, sh.cb);
        w1 = lookup(w1, sh.cb);
        f0 = reinterpret_cast<const float*>(sh.tables)[byte_at(win, o + at)];
      } else {
        w0 &= 0x0f0f0f0fu;
        w1 &= 0x0f0f0f0fu;
        f0 = fp16_to_fp32(half_at(win, o + at));
        if constexpr (F == SF::Q4_0) {
          w0 = minus8(w0);
          w1 = minus8(w1);
        } else {
          f1 = fp16_to_fp32(half_at(win, o + at + 2));
        }
      }
    }
  }
};

// a compile-time loop: f(integral_constant<0>) .. f(integral_constant<7>)
template <class Fn>
__device__ __forceinline__ void for_blocks(Fn f) {
  f(std::integral_constant<int, 0>{});
  f(std::integral_constant<int, 1>{});
  f(std::integral_constant<int, 2>{});
  f(std::integral_constant<int, 3>{});
  f(std::integral_constant<int, 4>{});
  f(std::integral_constant<int, 5>{});
  f(std::integral_constant<int, 6>{});
  f(std::integral_constant<int, 7>{});
}

// MT token tiles of 16.  kWide (Q4_K, Q5_K): a caller's Q8_K records, whose
// bsums may be any int16; a quantizer's are at most 2048, exact in f16 (the
// wide form makes calls 1 to 7 % longer)
template <SF F, int MT, bool kGroup, bool kWide>
__global__ void __launch_bounds__((64 * max_waves<MT>())) small_gemm_kernel(Args a) {
  using T = Traits<F>;
  static_assert(T::kTableBytes + 64 + max_waves<MT>() * wave_lds<F, MT>() <= 158 * 1024, "fits the LDS");
  extern __shared__ __align__(16) char lds[];
  __shared__ uint32_t tflag[16];
  __shared__ int pairs[kGroup ? 16 : 1][16][2];  // each wave's copy: activation row and index of the tile's pairs
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int nwaves = __builtin_amdgcn_readfirstlane(blockDim.x / kWave);
  const int col = lane & 15, q = lane >> 4;

  // Workgroups are dealt to the eight XCDs in turn: the token tiles of one
  // weight tile (dense) stay on one XCD, whose L2 then serves their weights.
  int m0 = 0, mrows, n0;
  const uint8_t* W = a.W;
  if constexpr (kGroup) {
    // MUL_MAT_ID (ggml-cpu/ggml-cpu.c:1454-1698): lane p holds pair p's
    // expert; the workgroups of pair y take up to 16 pairs of y's expert from
    // y on, unless an earlier pair of it already does
    const PairArgs& p = a.pair;
    const int t = lane / p.n_ids, s = lane - t * p.n_ids, y = (int)blockIdx.y;
    const int id = lane < a.n_pairs ? p.ids[t * p.ids_s1 + s * p.ids_s0] : -1;
    const int e = __builtin_amdgcn_readlane(id, y);
    const uint64_t same = __builtin_amdgcn_ballot_w64(id == e);
    const int rank = __popcll(same & ((1ull << lane) - 1));  // of this lane's pair, if it is one of them
    const int first = __builtin_amdgcn_readlane(rank, y);
    if (e < 0 || e >= p.n_as || (first & 15) != 0) return;  // no barrier yet
    mrows = min(16, (int)__popcll(same) - first);
    if (id == e && rank >= first && rank < first + 16) {
      pairs[wave][rank - first][0] = t * p.ne11 + s % p.ne11;
      pairs[wave][rank - first][1] = lane;
    }
    wave_lds_fence();
    W += e * p.w_es;
    n0 = (int)blockIdx.x * 16;
  } else {
    const int b = (int)blockIdx.x, j = b >> 3, mt = j % a.mtiles;
    n0 = ((j / a.mtiles) * 8 + (b & 7)) * 16;
    if (n0 >= a.N) return;  // no barrier yet
    m0 = mt * 16 * MT;
    mrows = min(16 * MT, a.M - m0);
  }

  char* tables = lds;
  char* win = lds + T::kTableBytes + wave * wave_lds<F, MT>();
  char* ext = win + 16 * T::kPitch + 16;
  char* xwin = win + w_lds<F>();
  float* dxs = reinterpret_cast<float*>(xwin + 16 * MT * T::kXPitch);  // [tile][block][token]

  const int nunits = a.K >> 8;
  const uint32_t ldw = a.ldw;
  const uint32_t xrb = (uint32_t)nunits * T::kXUnit;

  // this lane's chunks: row and place are fixed, the unit moves.  Chunks past
  // the tile's last one repeat it (same bytes to the same place).
  constexpr int kWL = loads_per_lane(T::kChunks), kXL = loads_per_lane(T::kXChunks);
  uint32_t woff[kWL], wrow[kWL];
  int wdst[kWL];
#pragma unroll
  for (int j = 0; j < kWL; ++j) {
    const uint32_t c = min(lane + kWave * j, 16 * T::kChunks - 1), r = small_div<T::kChunks>(c);
    const uint32_t p = c - __umul24(r, T::kChunks);
    wrow[j] = r;
    woff[j] = __umul24(r, ldw) + T::kHead + 16 * p;
    wdst[j] = (int)(__umul24(r, T::kPitch) + 16 * p);
  }
  uint32_t xoff[MT][kXL], doff[MT];
  int xdst[kXL];
  auto act_row = [&](int r) -> uint32_t {
    r = min(r, mrows - 1);
    if constexpr (kGroup)
      return (uint32_t)pairs[wave][r][0];
    else
      return (uint32_t)(m0 + r);
  };
#pragma unroll
  for (int j = 0; j < kXL; ++j) {
    const uint32_t c = min(lane + kWave * j, 16 * T::kXChunks - 1), r = small_div<T::kXChunks>(c);
    const uint32_t p = c - __umul24(r, T::kXChunks);
#pragma unroll
    for (int t = 0; t < MT; ++t) xoff[t][j] = __umul24(act_row(16 * t + (int)r), xrb) + T::kXHead + 16 * p;
    xdst[j] = (int)(__umul24(r, T::kXPitch) + 16 * p);
  }
  if constexpr (T::kQ8K) {
#pragma unroll
    for (int t = 0; t < MT; ++t) doff[t] = __umul24(act_row(16 * t + col), xrb);
  }

  // chunks of the tokens a tile holds: the rest is neither read nor staged
  // (their products go nowhere)
  int xchunks[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) xchunks[t] = min(16, mrows - 16 * t) * T::kXChunks;

  uint4 wreg[kWL], xreg[MT][kXL];
  uint32_t ereg[4];
  float dreg[MT];
  auto fetch_w = [&](int u) {
    // rows of the tile past the matrix's last one repeat it
    const uint8_t* base = W + (size_t)n0 * ldw + (size_t)u * T::kUnit;
    const uint32_t last = (uint32_t)(a.N - 1 - n0);
    if (last >= 15u) {
#pragma unroll
      for (int j = 0; j < kWL; ++j) wreg[j] = load_chunk(base + woff[j]);
    } else {
#pragma unroll
      for (int j = 0; j < kWL; ++j)
        wreg[j] = load_chunk(base + (woff[j] - __umul24(wrow[j] - min(wrow[j], last), ldw)));
    }
    if constexpr (T::kExt != 0) {
      if (lane < 16) {
        const uint8_t* e = base + __umul24(min((uint32_t)lane, last), ldw);
        if constexpr (T::kExt == 2) {
          ereg[0] = load_half(e + T::kExtAt);
        } else {
          load_8(e + T::kExtAt, ereg[0], ereg[1]);
        }
        if constexpr (T::kExt2 != 0) load_8(e + 66, ereg[2], ereg[3]);
      }
    }
  };
  auto fetch_x = [&](int u) {
    const uint8_t* base = a.Xq + (size_t)u * T::kXUnit;
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      if constexpr (T::kQ8K) {
        if (lane < 16) dreg[t] = *reinterpret_cast<const float*>(base + doff[t]);
      }
#pragma unroll
      for (int j = 0; j < kXL; ++j)
        if (kWave * j < xchunks[t]) xreg[t][j] = load_chunk(base + xoff[t][j]);
    }
  };

  if (wave < nunits) {
    fetch_x(wave);
    fetch_w(wave);
  }

  // lookup tables (all waves), and whether the IQ2 ones suit the sign masks
  Shared sh;
  sh.q = q;
  sh.tables = tables;
  if constexpr (T::kIq2) {
    bool bad = false;
    for (int i = threadIdx.x; i < T::kGridWords; i += blockDim.x) {
      const uint32_t g = reinterpret_cast<const uint32_t*>(a.tab0)[i];
      reinterpret_cast<uint32_t*>(tables)[i] = g;
      bad |= !iq2_grid_word_ok(g);
    }
    for (int i = threadIdx.x; i < 256; i += blockDim.x) {
      const uint32_t sg = reinterpret_cast<const uint32_t*>(a.tab1)[i];
      reinterpret_cast<uint32_t*>(tables + 4 * T::kGridWords)[i] = ((sg >> 7) & 0x01010101u) * 0xffu;
      reinterpret_cast<uint32_t*>(tables + 4 * T::kGridWords + 1024)[i] = sg;
      bad |= !iq2_sign_word_ok(sg);
    }
    iq2_flag_wave(tflag, bad);
    __syncthreads();
    sh.canon = iq2_flags_clear(tflag, nwaves);
    sh.grid = reinterpret_cast<const uint2*>(tables);
    sh.sgn = reinterpret_cast<const uint2*>(tables + 4 * T::kGridWords + (sh.canon ? 0 : 1024));
  } else if constexpr (T::kTable) {
    const uint8_t* c = reinterpret_cast<const uint8_t*>(a.tab0);
#pragma unroll
    for (int i = 0; i < 4; ++i) sh.cb[i] = ld_u32_a1(c + 4 * i);
    for (int i = threadIdx.x; i < 256; i += blockDim.x)
      reinterpret_cast<float*>(tables)[i] = reinterpret_cast<const float*>(a.tab1)[i];
    __syncthreads();
  }

  float y[MT][4];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) y[t][r] = 0.f;
  const v4i zero = {};
  const bool h0 = q < 2;

  for (int u = wave; u < nunits; u += nwaves) {
    const bool more = u + nwaves < nunits;
    // this unit into the windows, the next one's loads
#pragma unroll
    for (int t = 0; t < MT; ++t) {
#pragma unroll
      for (int j = 0; j < kXL; ++j)
        if (kWave * j < xchunks[t]) *reinterpret_cast<uint4*>(xwin + 16 * t * T::kXPitch + xdst[j]) = xreg[t][j];
      if constexpr (T::kQ8K) {
        if (lane < 16) dxs[16 * t + lane] = dreg[t];
      }
    }
#pragma unroll
    for (int j = 0; j < kWL; ++j) *reinterpret_cast<uint4*>(win + wdst[j]) = wreg[j];
    if constexpr (T::kExt != 0) {
      if (lane < 16)
        *reinterpret_cast<uint4*>(ext + 16 * lane) = make_uint4(
            ereg[0], T::kExt == 8 ? ereg[1] : 0u, T::kExt2 ? ereg[2] : 0u, T::kExt2 ? ereg[3] : 0u);
    }
    if (more) {
      fetch_x(u + nwaves);
      fetch_w(u + nwaves);
    }
    wave_lds_fence();
    // NVFP4: whether a token's block scale of the unit is not finite
    bool odd_dx = false;
    if constexpr (!T::kQ8K) {
      // the tokens' block scales as floats: lane (token col, blocks q, q + 4)
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int at = (16 * t + col) * T::kXPitch + (q + 4 * i) * T::kXRec;
          const uint32_t d = half_at(xwin, at);
          dxs[128 * t + 16 * (q + 4 * i) + col] = fp16_to_fp32(d);
          if constexpr (F == SF::NVFP4) odd_dx |= 16 * t + col < mrows && (d & 0x7c00u) == 0x7c00u;
          if constexpr (T::kAct == Act::Q8_1)
            dxs[128 * (MT + t) + 16 * (q + 4 * i) + col] = fp16_to_fp32(half_at(xwin, at + 2));
        }
    }
    if constexpr (!T::kQ8K) wave_lds_fence();
    if constexpr (F == SF::NVFP4) odd_dx = __builtin_amdgcn_ballot_w64(odd_dx) != 0;
    const int xo = col * T::kXPitch + 8 * q, o = col * T::kPitch;
    Row<F> row;
    row.begin(win, o, ext + 16 * col, sh);
    int S[MT][4];     // Q8_K formats: the unit's exact integer sums
    float yu[MT][4];  // the others: the unit's fp32 sum (a chain of eight, then one of units: less rounding)
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        S[t][r] = 0;
        yu[t][r] = 0.f;
      }
    // one block's terms; apart (NVFP4): each half's by itself, in GGML's order
    auto block_terms = [&](auto blk, auto apart) {
      constexpr int s = decltype(blk)::value;
      long x[MT];
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        uint32_t v[2];
        run<T::kQ8K ? 32 * s : T::kXRec * s + T::kXRec - 32>(xwin, xo + 16 * t * T::kXPitch, v);
        x[t] = pack(v[0], v[1]);
      }
      uint32_t w0, w1;
      int c0 = 0, c1 = 0;
      float f0 = 0.f, f1 = 0.f;
      row.template block<s>(win, o, sh, w0, w1, c0, c1, f0, f1);
      constexpr bool kHalves = F == SF::Q6_K || F == SF::IQ2_XS || F == SF::NVFP4;
      const long wa = kHalves ? pack(h0 ? w0 : 0u, h0 ? w1 : 0u) : pack(w0, w1);
      const long wb = pack(h0 ? 0u : w0, h0 ? 0u : w1);
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const v4i I = __builtin_amdgcn_mfma_i32_16x16x32_i8(x[t], wa, zero, 0, 0, 0);
        v4i I2 = {};
        if constexpr (kHalves) I2 = __builtin_amdgcn_mfma_i32_16x16x32_i8(x[t], wb, zero, 0, 0, 0);
        if constexpr (T::kQ8K) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            S[t][r] += __mul24(I[r], c0);
            if constexpr (kHalves) S[t][r] += __mul24(I2[r], c1);
            // summed here: all blocks' products kept for one tree spill
            asm volatile("" : "+v"(S[t][r]));
          }
        } else {
          float(&yt)[4] = yu[t];
          const float4 d4 = *reinterpret_cast<const float4*>(dxs + 128 * t + 16 * s + 4 * q);
          const float dx[4] = {d4.x, d4.y, d4.z, d4.w};
          if constexpr (F == SF::MXFP4) {
#pragma unroll
            for (int r = 0; r < 4; ++r) yt[r] = ggml_scaled_term(yt[r], dx[r], f0, (float)I[r]);
          } else if constexpr (F == SF::Q4_0) {
#pragma unroll
            for (int r = 0; r < 4; ++r) yt[r] = fmaf(f0 * dx[r], (float)I[r], yt[r]);
          } else if constexpr (F == SF::NVFP4) {
            if constexpr (decltype(apart)::value) {
#pragma unroll
              for (int r = 0; r < 4; ++r)
                yt[r] = ggml_scaled_term(ggml_scaled_term(yt[r], dx[r], f0, (float)I[r]), dx[r], f1, (float)I2[r]);
            } else {
              // a UE4M3 scale has four bits, so its product with I is exact (of a
              // caller's table: rounded once)
#pragma unroll
              for (int r = 0; r < 4; ++r)
                yt[r] = fmaf(dx[r], fmaf(f1, (float)I2[r], f0 * (float)I[r]), yt[r]);
            }
          } else {
            const float4 s4 = *reinterpret_cast<const float4*>(dxs + 128 * (MT + t) + 16 * s + 4 * q);
            const float xs[4] = {s4.x, s4.y, s4.z, s4.w};
#pragma unroll
            for (int r = 0; r < 4; ++r) yt[r] = fmaf(f1, xs[r], fmaf(f0 * dx[r], (float)I[r], yt[r]));
          }
#pragma unroll
          for (int r = 0; r < 4; ++r) asm volatile("" : "+v"(yt[r]));
        }
      }
    };
    // Where a token's scale is not finite (NVFP4): an infinite dx is NaN with a
    // half that is zero and with two halves of unlike signs (ggml-cpu/quants.c:
    // 279-313), which the sum of the halves would hide.  A loop of its own, as a
    // choice at every block made every call 3 to 9 % longer.
    bool apart = false;
    if constexpr (F == SF::NVFP4) {
      apart = odd_dx;
      if (apart) for_blocks([&](auto blk) { block_terms(blk, std::true_type{}); });
    }
    if (!apart) for_blocks([&](auto blk) { block_terms(blk, std::false_type{}); });
    if constexpr (T::kQ8K) {
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        float(&yt)[4] = y[t];
        const float4 d4 = *reinterpret_cast<const float4*>(dxs + 16 * t + 4 * q);
        const float dx[4] = {d4.x, d4.y, d4.z, d4.w};
        if constexpr (F == SF::Q4_K || F == SF::Q5_K) {
          // Mn = sum_j m_{j/2} bsum_j: exact in f16 operands and fp32 sums
          uint32_t bs[2];  // bsums 4 q .. + 3 of token col
          run<256>(xwin, xo + 16 * t * T::kXPitch, bs);
          const uint32_t mw = (q < 2 ? row.mn03 : row.mn47) >> (16 * (q & 1));
          const _Float16 ma = (_Float16)(float)(mw & 63u), mb = (_Float16)(float)((mw >> 8) & 63u);
          const short b[4] = {(short)(bs[0] & 0xffffu), (short)(bs[0] >> 16), (short)(bs[1] & 0xffffu),
                              (short)(bs[1] >> 16)};
          const v4f fz = {};
          v4f mn;
          if constexpr (kWide) {
            // as 16 hi + lo in two of 32 places: lo's mins are m, hi's 16 m (at most 1008)
            const v8h am = {(_Float16)(short)(b[0] & 15), (_Float16)(short)(b[1] & 15), (_Float16)(short)(b[2] & 15),
                            (_Float16)(short)(b[3] & 15), (_Float16)(short)(b[0] >> 4), (_Float16)(short)(b[1] >> 4),
                            (_Float16)(short)(b[2] >> 4), (_Float16)(short)(b[3] >> 4)};
            const _Float16 k16 = (_Float16)16.f;
            const v8h bm = {ma, ma, mb, mb, k16 * ma, k16 * ma, k16 * mb, k16 * mb};
            mn = __builtin_amdgcn_mfma_f32_16x16x32_f16(am, bm, fz, 0, 0, 0);
          } else {
            const v4h am = {(_Float16)b[0], (_Float16)b[1], (_Float16)b[2], (_Float16)b[3]};
            const v4h bm = {ma, ma, mb, mb};
            mn = __builtin_amdgcn_mfma_f32_16x16x16f16(am, bm, fz, 0, 0, 0);
          }
#pragma unroll
          for (int r = 0; r < 4; ++r) yt[r] = fmaf(dx[r], row.dw * (float)S[t][r] - row.dmin * mn[r], yt[r]);
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r) yt[r] = fmaf(row.dw * dx[r], (float)S[t][r], yt[r]);
        }
      }
    } else {
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) y[t][r] += yu[t][r];
    }
    wave_lds_fence();  // every lane is done with the windows
  }

  // the waves' partial sums, added in wave order
  __syncthreads();
  constexpr int kOut = MT * 256;
  float* part = reinterpret_cast<float*>(lds);
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) part[wave * kOut + (t * 4 + r) * kWave + lane] = y[t][r];
  __syncthreads();
  for (int i = threadIdx.x; i < kOut; i += blockDim.x) {
    const int c = i & 15, row = 16 * (i >> 8) + 4 * ((i >> 4) & 3) + ((i >> 6) & 3);
    if (row >= mrows || n0 + c >= a.N) continue;
    double v = 0.;  // up to 16 sums: one rounding instead of one each
    for (int w = 0; w < nwaves; ++w) v += part[w * kOut + i];
    long long at;
    if constexpr (kGroup) {
      const int p = pairs[wave][row][1], t = p / a.pair.n_ids;
      at = t * a.pair.y_s2 + (p - t * a.pair.n_ids) * a.pair.y_s1;
    } else {
      at = (long long)(m0 + row) * a.ldy;
    }
    a.Y[at + n0 + c] = (float)v;
  }
}

template <SF F, int MT, bool kGroup>
void launch_tile(const Args& a, int gx, int gy) {
  // Waves share out a workgroup's units: four when the launch gives every CU
  // two workgroups, else twice as many per halving, so that about eight waves
  // a CU load at once.  Measured, Q4_K, 8 tokens: 11008 x 4096 (688
  // workgroups) 13.4 / 13.7 / 16.6 us a call at 4 / 8 / 16 waves, 4096 x 4096
  // (256) 10.2 / 8.1 / 8.1.  (MUL_MAT_ID's count is of all pairs, though of
  // those of one expert only one in sixteen works: the others are launched too.)
  // All of them at the same time, though: with two token tiles a CU's LDS holds
  // one workgroup of eight waves, three of four and six of two, and a second
  // round costs as much as the first.  So eight waves only where every
  // workgroup has a CU (Q4_K, 32 tokens, 5120 x 4096: 15.1 us at eight, 13.9 at
  // four), and two where four leave a rest that two do not, up to 3072 values
  // (IQ2_XXS, 32 tokens, 16384 x 1536: 17.4 us at four, 14.2 at two; at 11008
  // values two are up to 15 % slower).
  const int wgs = gx * gy;
  auto lds_bytes = [](int waves) { return (size_t)Traits<F>::kTableBytes + (size_t)waves * wave_lds<F, MT>(); };
  auto one_round = [&](int waves) {
    return (size_t)wgs <= (size_t)cu_count() * (160 * 1024 / (lds_bytes(waves) + 64));
  };
  int nwaves = 4;
  while (nwaves < max_waves<MT>() && wgs * nwaves < 8 * cu_count() && one_round(2 * nwaves)) nwaves *= 2;
  if (MT == 2 && a.K <= 3072 && !one_round(4) && one_round(2)) nwaves = 2;
  nwaves = std::min(nwaves, a.K / 256);  // every wave has a unit
  const size_t bytes = std::max(lds_bytes(nwaves), (size_t)nwaves * MT * 1024);
  const dim3 grid((unsigned)gx, (unsigned)gy);
  constexpr bool kBsums = F == SF::Q4_K || F == SF::Q5_K;
  if (kBsums && a.wide)
    small_gemm_kernel<F, MT, kGroup, kBsums><<<grid, nwaves * kWave, bytes, current_stream()>>>(a);
  else
    small_gemm_kernel<F, MT, kGroup, false><<<grid, nwaves * kWave, bytes, current_stream()>>>(a);
  check_launch(kGroup ? "small_mfma_gemm_grouped" : "small_mfma_gemm");
}

template <SF F, int MT>
void launch_dense(Args a) {
  a.mtiles = (a.M + 16 * MT - 1) / (16 * MT);
  const int gx = (a.N + 127) / 128 * 8 * a.mtiles;  // eight weight tiles (one an XCD) a step
  launch_tile<F, MT, false>(a, gx, 1);
}
template <SF F>
void launch_dense(const Args& a) {
  return a.M <= 16 ? launch_dense<F, 1>(a) : launch_dense<F, 2>(a);
}

template <SF F>
void launch_pairs(const Args& a) {
  launch_tile<F, 1, true>(a, (a.N + 15) / 16, a.n_pairs);
}

template <SF F>
void launch(const Args& a) {
  return a.n_pairs > 0 ? launch_pairs<F>(a) : launch_dense<F>(a);
}
void launch_fmt(int fmt, const Args& a) {
  switch (fmt) {
    case 0: return launch<SF::Q4_0>(a);
    case 1: return launch<SF::MXFP4>(a);
    case 2: return launch<SF::IQ2_XXS>(a);
    case 3: return launch<SF::Q6_K>(a);
    case 4: return launch<SF::Q5_K>(a);
    case 5: return launch<SF::NVFP4>(a);
    case 6: return launch<SF::Q4_1>(a);
    case 7: return launch<SF::IQ2_XS>(a);
    default: return launch<SF::Q4_K>(a);
  }
}

struct FmtInfo {
  size_t elems, rec, w_align, x_align;  // of a record; alignment of W and of Xq
  size_t x_elems, x_rec;                // of the activation's records
  size_t x_row(size_t K) const { return K / x_elems * x_rec; }
};
template <SF F>
FmtInfo info_of(size_t w_align) {
  using T = Traits<F>;
  return {(size_t)T::kElems, (size_t)T::kRec, w_align, T::kQ8K ? 4u : 2u, T::kQ8K ? 256u : 32u, (size_t)T::kXRec};
}
FmtInfo fmt_info(int fmt) {
  switch (fmt) {
    case 0: return info_of<SF::Q4_0>(2);
    case 1: return info_of<SF::MXFP4>(1);
    case 2: return info_of<SF::IQ2_XXS>(2);
    case 3: return info_of<SF::Q6_K>(1);
    case 4: return info_of<SF::Q5_K>(2);
    case 5: return info_of<SF::NVFP4>(1);
    case 6: return info_of<SF::Q4_1>(2);
    case 7: return info_of<SF::IQ2_XS>(2);
    default: return info_of<SF::Q4_K>(2);
  }
}
bool tables_ok(int fmt, const int8_t* tab0, const void* tab1) {
  if (fmt == 1 || fmt == 5) return tab0 != nullptr && tab1 != nullptr && aligned(tab1, 4);
  if (fmt == 2 || fmt == 7) return tab0 != nullptr && tab1 != nullptr && aligned(tab0, 4) && aligned(tab1, 4);
  return true;
}

}  // namespace

// row strides of the weights and of the quantized activation stay in 24 bits
static constexpr size_t kMaxRow = (size_t)1 << 24;

// Whether the small-batch kernel takes a product of M activation rows: every
// record alignment and row stride and every K of whole 256-value units does;
// bound tiles (weft_hip_set_tile_binding) choose launches of the GEMVs and
// the prefill GEMMs, so they keep those.
static bool small_ok(int fmt, const uint8_t* W, const uint8_t* Xq, const int8_t* tab0, const void* tab1,
                     const float* Y, size_t N, size_t K, size_t M, const RowStrides& st) {
  const FmtInfo f = fmt_info(fmt);
  const TileBindings& tb = tile_bindings();
  return N > 0 && K > 0 && K % 256 == 0 && tb.nc == 0 && tb.mr == 0 && tb.mc == 0 && W != nullptr &&
         Xq != nullptr && Y != nullptr && N <= (size_t)INT32_MAX - 256 && K <= (size_t)INT32_MAX &&
         M < ((size_t)1 << 24) && (M + 15) / 16 * ((N + 127) / 128) < ((size_t)1 << 27) &&
         M * f.x_row(K) < ((size_t)1 << 32) && std::max(st.ldw, K / f.elems * f.rec) < kMaxRow &&
         f.x_row(K) < kMaxRow && aligned(W, f.w_align) && aligned(Xq, f.x_align) && aligned(Y, 4) &&
         tables_ok(fmt, tab0, tab1) && strides_ok(st, K / f.elems * f.rec, f.w_align, K, N, N, 1);
}

// Whether the small-batch kernel is the faster one (figures: one call, replayed
// from a graph).
//
// Below 16 rows the other is a GEMV of four rows a pass, with the quantization
// in the same launch.  A batch of one pass is that one launch against two, about
// 4 against 7 us of host time where both are short, until the pass is longer:
// from 28M products of weights and rows on (Q4_0, 3 rows: 2048 x 2048 5.6 against
// 6.2 us, 4096 x 2048 6.2 against 6.1, 4096 x 4096 8.9 against 8.3), from 16M
// where it is long itself (Q5_K, Q6_K, NVFP4: Q5_K, 4 rows, 4096 x 1024 7.1
// against 5.6), of 16384 activation values, which every workgroup quantizes (Q4_0,
// 4 rows, 64 x 4096 7.7 against 7.0), or of 8192 weight rows.  Q4_K's pass is 6.5
// us from the start.  Past those, Q4_K / Q5_K win from 2 rows (11008 x 4096: 11.9
// against 13.8 us, 12.6 against 14.1), the rest from 3 (Q4_0 13.7 against 14.9; at
// 2, 13.6 against 12.7), MXFP4 and the formats with two scales a block from 4
// (NVFP4 18.3 against 17.0 at 3).  A quantized src1 is one launch either way.
//
// From 16 rows the other is the prefill GEMM, which takes one K loop of a 64 x
// 128 tile whatever N is until the tiles fill the chip, while this kernel's time
// grows with the weight rows times the token tiles; both grow with K.  The
// limits are where the two lines measured at 4096 and 11008 x 4096, 16 .. 64
// rows, cross (MXFP4, 64 rows: 20.7 against 33.0 us at 4096 rows, 41.0 against
// 35.3 at 11008); at 512 .. 14336 values, 16 .. 64 rows and row counts up to
// them no call was more than 4 % slower but for two, which have limits of their
// own: MXFP4 past 3072 values, where a second round of workgroups is not worth
// it (13000 x 11008, 32 rows: 65.3 against 58.1), and Q4_K at 17 .. 32 rows of
// 512 values, whose GEMM then has tiles of 32 x 64 (5632 x 512 7.0 against 6.4;
// 5120 x 768 to x 4096 0 to 10 % faster here but for 1536 values, 3 % slower).
static bool small_wins(int fmt, size_t N, size_t K, size_t M, bool gemm, bool quantize) {
  static constexpr uint8_t kFrom[9] = {3, 4, 3, 4, 2, 4, 3, 4, 2};
  static constexpr uint16_t kLimit[9] = {21000, 14000, 20000, 17000, 27000, 28000, 21000, 18000, 8192};
  if (M < kFrom[fmt]) return false;
  const size_t pass = M >= 3 && (fmt == 3 || fmt == 4 || fmt == 5) ? (size_t)16 << 20 : (size_t)28 << 20;
  if (quantize && M <= 4 && fmt != 8 && M * K < 16384 && N < 8192 && M * N * K < pass) return false;
  if (M < 16 || !gemm) return true;
  if (M > kSmallBatchRows) return false;
  size_t limit = kLimit[fmt];
  if (fmt == 1 && K > 3072) limit = 12288;
  if (fmt == 8 && M > 32) limit = limit * 3 / 2;  // its GEMM is 1.5 times longer past 32 rows
  if (fmt == 8 && M > 16 && M <= 32 && K <= 512) limit = 4096;
  // one token tile of 16 costs five eighths of one of 32
  const size_t w = M <= 16 ? N * 5 / 8 : N * ((M + 31) / 32);
  return w <= limit;
}

static bool small_run(int fmt, const uint8_t* W, const uint8_t* Xq, const int8_t* tab0, const void* tab1,
                      float* Y, size_t N, size_t K, size_t M, const RowStrides& st, bool gemm, bool wide) {
  if (!small_wins(fmt, N, K, M, gemm, !wide) || st.ldy < N || st.ldy >= ((size_t)1 << 38) ||
      !small_ok(fmt, W, Xq, tab0, tab1, Y, N, K, M, st)) return false;
  const FmtInfo f = fmt_info(fmt);
  const Args a{W, Xq, tab0, tab1, Y, (int)N, (int)K, (int)M, 1, (uint32_t)(N > 1 ? st.ldw : K / f.elems * f.rec),
               (long long)st.ldy, PairArgs{}, 0, wide};
  launch_fmt(fmt, a);
  return true;
}
bool small_batch_quantized(int fmt, const uint8_t* W, const uint8_t* Xq, const int8_t* tab0, const void* tab1,
                           float* Y, size_t N, size_t K, size_t M, const RowStrides& st, bool gemm) {
  return small_run(fmt, W, Xq, tab0, tab1, Y, N, K, M, st, gemm, true);
}

// Whether MUL_MAT_ID's pair GEMV, one launch that reads an expert's weights once
// for every pair of it, is the faster one: large matrices that it reads faster
// than this kernel does, of which few pairs share an expert.  The first token's
// pairs never do; `rest` of the others may.  Q4_K, whose GEMV keeps a row of up to
// 4096 values in registers (one call, experts past the Infinity Cache): 14336 x
// 4096, 2 pairs 14.8 us against 19.7 here, 16 experts of it, 2 a token, 2 / 4 / 6
// tokens 44 / 46 / 67 against 47 / 49 / 68, 8 tokens 83 against 75; 6144 x 8192, 8
// experts, 2 tokens 26.5 against 29.3, 8192 x 4096, 3 pairs of 4 14.5 and 16.2; 4096 x 4096 equal from 2 pairs on, 28672 x
// 1024, 2 pairs 14 against 11.  NVFP4,
// whose weights take this kernel longest, where a token has one expert: 11008 x
// 4096, 2 / 3 pairs 21.3 / 30.6 against 25.6 / 34.2.  Of the other formats the
// GEMV is at most as fast but for single shapes at 2 pairs.
static bool pair_gemv_wins(int fmt, size_t N, size_t K, const PairArgs& pr, int n_pairs) {
  const size_t values = N * K;
  const int rest = n_pairs - pr.n_ids;
  if (fmt == 5) return pr.n_ids == 1 && K > 2048 && values >= (size_t)40 << 20 && (rest == 1 || 8 * rest <= pr.n_as);
  if (fmt != 8 || K < 2048 || K > 8192) return false;
  if (K > 2048 && K <= 4096 && values >= (size_t)40 << 20) return rest <= 10 && 2 * rest <= pr.n_as;
  if (values >= (size_t)32 << 20) return rest <= 2 ? 2 * rest <= pr.n_as : rest == 3 && 4 * rest <= pr.n_as;
  return n_pairs == 2 && values >= (size_t)24 << 20;
}

bool small_pairs_ok(int fmt, const uint8_t* W, const uint8_t* Xq, const int8_t* tab0, const void* tab1,
                    const float* Y, size_t N, size_t K, const RowStrides& st, const PairArgs& pr, int n_pairs,
                    size_t x_rows) {
  return n_pairs >= 2 && n_pairs <= 64 && !pair_gemv_wins(fmt, N, K, pr, n_pairs) && pr.w_es % (long long)fmt_info(fmt).w_align == 0 &&
         small_ok(fmt, W, Xq, tab0, tab1, Y, N, K, x_rows, st);
}
void small_pairs(int fmt, const uint8_t* W, const uint8_t* Xq, const int8_t* tab0, const void* tab1, float* Y,
                 size_t N, size_t K, const RowStrides& st, const PairArgs& pr, int n_pairs, bool caller_xq) {
  const FmtInfo f = fmt_info(fmt);
  const Args a{W, Xq, tab0, tab1, Y, (int)N, (int)K, 16, 1, (uint32_t)(N > 1 ? st.ldw : K / f.elems * f.rec),
               0, pr, n_pairs, caller_xq};
  launch_fmt(fmt, a);
}

bool small_batch(int fmt, const uint8_t* W, const float* X, uint8_t* Xq, const int8_t* tab0, const void* tab1,
                 float* Y, size_t N, size_t K, size_t M, const RowStrides& st, bool gemm) {
  if (X == nullptr || !aligned(X, 4) || !small_wins(fmt, N, K, M, gemm, true) || st.ldx < K || st.ldy < N ||
      st.ldx >= ((size_t)1 << 38) || st.ldy >= ((size_t)1 << 38) || !small_ok(fmt, W, Xq, tab0, tab1, Y, N, K, M, st))
    return false;
  switch (fmt) {
    case 0:
    case 1:
    case 5: quantize_q8_0_rows(X, st.ldx, Xq, M, K); break;
    case 6: quantize_q8_1_rows(X, st.ldx, Xq, M, K); break;
    default: quantize_q8_k_rows(X, st.ldx, Xq, M, K); break;
  }
  return small_run(fmt, W, Xq, tab0, tab1, Y, N, K, M, st, gemm, false);
}

}  // namespace weft
