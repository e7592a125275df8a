// Q6_K and Q5_K x Q8_K prefill GEMMs on int8 MFMA (production_mul_mat_q6_k,
// production_mul_mat_q5_k; examples/kernels/mul_mat/q6_k.py:9-37,
// q5_k.py:9-37), with a grouped MUL_MAT_ID mode.
//
// Q6_K (ggml-cpu/quants.c:800-853):
//   Y[m,n] = sum_b (dw[n,b] dx[m,b]) * sum_{j<16} sc[n,b,j] * P[m,n,b,j]
//   P = sum_{k in 16-group j} q8[m,k] * (q6[n,k] - 32)                (exact int32)
// The signed 8-bit scale times the 6-bit value, p = sc (q6 - 32), does not fit
// an int8 operand (|p| <= 4096), but it is two of them exactly, p = 256 H + L
// with L its signed low byte: two v_mfma_i32_32x32x32_i8 per 32-group, whose
// int32 tiles run over the half superblock, S = lo + 256 hi.  Lane half kg of
// the operand holds exactly the 16 elements of scale group 2 s + kg, so a
// lane multiplies by one scale: v_pk_mad_u16 gives p + 128 for two values, of
// which a byte permute takes the high bytes (H) and the low ones (L + 128).
// What bounds it is VALU issue beside the MFMAs: about 11 instructions per
// four weights and 3 per output and half superblock.  Before, each 16-group's
// product tile took its scale on VALU (two masked MFMAs per 32-group and two
// multiply-adds per output): 633 VALU instructions per wave and half
// superblock, now about 300.
//
// Q5_K (ggml-cpu/quants.c:720-798):
//   Y[m,n] = sum_b (dw dx) * S - (dmin dx) * Mn
//   S  = sum_{g<8} sc[n,b,g] * sum_{k in 32-group g} q8 * q5            (exact int32)
//   Mn = sum_{j<16} m[n,b,j/2] * bsum[m,b,j]                             (exact)
// q5 in [0, 31] is the weight operand as it is; one MFMA per 32-group and
// one multiply-add of its 6-bit scale per output.  Mn comes from one
// v_mfma_f32_32x32x8_f16 per half superblock: Q8_K's bsums are sums of 16
// int8 (|bsum| <= 2032) and the mins 6-bit, so both are exact f16 operands
// and the fp32 result is exact (|Mn| < 2^21).
//
// The superblock's fp32 factors dx dw (and dx dmin) of every output come from
// one bf16 outer-product MFMA per tile each (dx = h + m + l in bf16 parts
// against the fp16 scale's two bf16 parts: six exact products summed in
// fp32), so the combine is a convert and one FMA per output (two for Q5_K).
//
// Tiling: 64 tokens x 128 weight rows per workgroup, 8 waves; wave w takes
// weight rows 32 (w % 4) .. +31 and the half superblock w / 4 (elements
// 128 h .. +127: Q6_K's ql/qh half, Q5_K's groups 4h .. 4h+3) for all 64
// tokens as two 32x32 tiles that share the weight operand.  One superblock
// per ring slot, two slots: the waves stage superblock b+1 by direct
// global->LDS loads while computing b (Q5_K's 176-byte records as 16-byte
// chunks when the rows are aligned).  A Q6_K record (210 bytes) is 2-byte
// aligned for odd b, so its row is staged from the dword holding its first
// byte (53 dwords as 16-byte chunks, 240 bytes per LDS row: 16 lanes' reads
// fall on all 64 banks) and the odd superblocks read with
// a 2-byte alignment; the even/odd slots are the two instantiations of the
// step.  Rows that are themselves only 2-byte aligned (an odd number of
// superblocks) take the third, which aligns by each lane's own row.  Both
// halves' partial sums meet in LDS at the end and every output
// is written once, even + odd, with 16-byte stores (tile_store.h).
#include <algorithm>
#include <type_traits>

#include "kernels.h"
#include "runtime.h"
#include "tile_store.h"
#include "weft_common.h"
#include "weft_hip.h"

namespace weft {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef short v2s __attribute__((ext_vector_type(2)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) void* lds_ptr;

constexpr int kMT = 64;        // tokens per workgroup tile
constexpr int kNT = 128;       // weight rows per workgroup tile
constexpr int kThreads = 512;  // 8 waves: 4 column groups x 2 half superblocks
constexpr int kAQ = kMT * 256;  // activation int8 of one superblock

enum class KQ { Q6_K, Q5_K };

template <KQ F>
struct KTile {
  static constexpr bool k6 = F == KQ::Q6_K;
  static constexpr int kRec = k6 ? kQ6_KBytes : kQ5_KBytes;  // 210 / 176
  static constexpr int kRowB = k6 ? 240 : 176;               // LDS bytes per weight row
  static constexpr int kLoadD = kRowB / 4;                   // in dwords
  static constexpr int kBS = k6 ? 0 : kMT * 32;              // Q5_K: the tokens' bsums
  static constexpr int kWT = kNT * kRowB;
  static constexpr int kSlot = kAQ + kBS + kWT;              // 47,104 / 40,960
  static constexpr int kWSlots = kNT * kLoadD / 64;          // wave-wide dword loads (Q5_K: 88)
  static_assert(kNT * kLoadD % 64 == 0, "weight tile is whole wave loads");
  static_assert(kTilePlaneBytes <= kSlot, "an output plane fits one ring slot");
};

struct GemmArgs {
  const uint8_t* W;
  const uint8_t* Xq;
  float* Y;
  int N, K, M;
  size_t ldw;      // bytes between weight rows
  long long ldy;   // floats between output rows
  GroupTiles grp;  // grouped (MUL_MAT_ID) mode
};

// Direct global->LDS loads; lane l writes [lds + size*l, +size).  Inline asm
// keeps the compiler from making unrelated LDS reads wait for them; the
// kernel waits (s_waitcnt) itself.  Nothing else in this kernel uses M0.
__device__ __forceinline__ void lds_dma16(const uint8_t* g, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
               :
               : "s"(lds), "v"(g)
               : "memory", "m0");
}
__device__ __forceinline__ void lds_dma4(const uint8_t* g, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off"
               :
               : "s"(lds), "v"(g)
               : "memory", "m0");
}
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return (uint32_t)(uintptr_t)(lds_ptr)p;
}
__device__ __forceinline__ void lds_store16(uint32_t lds, uint32_t v) {
  *reinterpret_cast<__attribute__((address_space(3))) uint16_t*>(lds) = (uint16_t)v;
}
__device__ __forceinline__ void pin(int& v) { asm volatile("" : "+v"(v)); }

// 16 bytes that start sh (0 or 2) bytes past the 16-byte aligned LDS address
// p: kSh = sh where it is known, else kRowShift
constexpr int kRowShift = -1;
template <int kSh>
__device__ __forceinline__ uint4 ld16(const uint8_t* p, uint32_t sh) {
  const uint4 a = *reinterpret_cast<const uint4*>(p);
  if constexpr (kSh == 0) {
    return a;
  } else {
    const uint32_t c = *reinterpret_cast<const uint32_t*>(p + 16);
    return make_uint4(__builtin_amdgcn_alignbyte(a.y, a.x, sh), __builtin_amdgcn_alignbyte(a.z, a.y, sh),
                      __builtin_amdgcn_alignbyte(a.w, a.z, sh), __builtin_amdgcn_alignbyte(c, a.w, sh));
  }
}

// kOdd (Q6_K): weight rows that are only 2-byte aligned
template <bool kGroup, KQ F, bool kOdd = false>
__global__ void __launch_bounds__(kThreads, 1) kq_mfma_gemm(GemmArgs a) {
  using TT = KTile<F>;
  constexpr bool k6 = TT::k6;
  constexpr int kRowB = TT::kRowB, kLoadD = TT::kLoadD, kWSlots = TT::kWSlots;
  __shared__ __align__(16) uint8_t ring0[TT::kSlot];
  __shared__ __align__(16) uint8_t ring1[TT::kSlot];
  // [slot][token]: the token's Q8_K d as the bf16 parts of the outer-product
  // factor MFMA ((h,h), (m,m), (l,l), 0)
  __shared__ __align__(16) uint4 dxq[2][kMT];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int h = wave >> 2, wcol = wave & 3;
  const int col = lane & 31, kg = lane >> 5;
  const int nsb = a.K >> 8;
  const size_t wrb = a.ldw;
  const size_t xrb = (size_t)nsb * kQ8_KBytes;

  // XCD-aware tile order (workgroups are dealt round-robin to 8 XCDs);
  // grouped: m0 indexes the pair list, mrows pairs, W the tile's expert
  int m0, n0, mrows;
  const uint8_t* W = a.W;
  {
    const int ntm = kGroup ? a.grp.tmax : (a.M + kMT - 1) / kMT;
    const int ntn = (a.N + kNT - 1) / kNT, Tn = ntm * ntn;
    const int L = blockIdx.x, x = L & 7, j = L >> 3;
    const int t = x * (Tn >> 3) + min(x, Tn & 7) + j;
    if constexpr (kGroup) {
      n0 = (t / ntm) * kNT;
      long long w_off;
      if (!group_tile(a.grp, t % ntm, m0, mrows, w_off)) return;  // no barrier yet
      W += w_off;
    } else {
      int tm, tn;
      banded_tile(t, ntm, ntn, tm, tn);
      m0 = tm * kMT;
      n0 = tn * kNT;
      mrows = min(kMT, a.M - m0);
    }
  }
  auto act_row = [&](int r) -> int {
    if constexpr (kGroup)
      return group_act_row(a.grp, m0, r);
    else
      return m0 + r;
  };

  // activation int8 of one superblock: 16 wave-wide 16-byte loads, 2 per
  // wave; token r's chunk c lands at 256 r + 16 (c ^ (r & 15))
  const uint8_t* asrc[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int q = 64 * (wave + 8 * i) + lane, r = q >> 4, c = (q & 15) ^ (r & 15);
    asrc[i] = a.Xq + (size_t)act_row(min(r, mrows - 1)) * xrb + 4 + 16 * c;
  }
  // Q5_K: the 32 bsum bytes of each token, 2 wave loads (waves 0, 1)
  const uint8_t* bsrc = a.Xq + (size_t)act_row(min((64 * (wave & 1) + lane) >> 1, mrows - 1)) * xrb + 260 +
                        16 * (lane & 1);
  const uint8_t* dsrc = a.Xq + (size_t)act_row(min(lane, mrows - 1)) * xrb;  // Q8_K d of token lane

  const bool w16 = ((reinterpret_cast<uintptr_t>(W) | wrb) & 15) == 0;  // Q5_K: 16-byte weight loads
  const uint32_t ring_lds[2] = {(uint32_t)__builtin_amdgcn_readfirstlane(lds_addr(ring0)),
                                (uint32_t)__builtin_amdgcn_readfirstlane(lds_addr(ring1))};
  // (kOdd) the weights of the row's last superblock b where the tile holds the
  // last row: of a record that begins with its dword, dword 52 ends two bytes
  // past it, and past the last row's last one nothing may be read.  That row's
  // d goes to its place (LDS bytes 220, 221) by itself.
  auto issue_last = [&](int b, uint32_t base) {
#pragma unroll 1
    for (int k = wave; k < kNT * 15 / 64; k += 8) {
      const int q = 64 * k + lane, row = q / 15, c = q - 15 * row, n = min(n0 + row, a.N - 1);
      const uint8_t* g = W + (size_t)n * wrb + (size_t)b * TT::kRec;
      const uint32_t gsh = (uint32_t)(uintptr_t)g & 2u;
      const uint32_t at = base + kAQ + TT::kBS + 1024 * k;
      if (n == a.N - 1 && gsh == 0 && c >= 13) {
        const uint32_t d = *reinterpret_cast<const uint16_t*>(g + 208);
        if (c == 13) lds_store16(at + 16 * lane + 12, d);
      } else {
        lds_dma16(g - gsh + min(16 * c, 196), at);
      }
    }
  };
  auto issue = [&](int b, int slot) {
    const uint32_t base = ring_lds[slot];
#pragma unroll
    for (int i = 0; i < 2; ++i)
      lds_dma16(asrc[i] + (size_t)b * kQ8_KBytes, base + 1024 * (wave + 8 * i));
    if constexpr (!k6) {
      if (wave < 2) lds_dma16(bsrc + (size_t)b * kQ8_KBytes, base + kAQ + 1024 * wave);
    }
    // weight rows: Q6_K from the dword holding the record's first byte (2
    // bytes before it for odd b), 53 dwords
    const size_t wb = (size_t)b * TT::kRec - (k6 && !kOdd ? 2 * (b & 1) : 0);
    if constexpr (k6) {
      // 15 chunks of 16 bytes a row (30 wave-wide loads, the row q / 15): 0 ..
      // 12 in place, 13 and 14 both the 16 bytes that end with dword 52, which
      // so lands at bytes 220 .. 223 and nothing past it is read (the weights'
      // last record: issue_last)
      if (kOdd && b + 1 == nsb && n0 + kNT >= a.N) return issue_last(b, base);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int k = wave + 8 * i;
        if (k < kNT * 15 / 64) {
          const int q = 64 * k + lane, row = q / 15, c = q - 15 * row;
          const uint8_t* g = W + (size_t)min(n0 + row, a.N - 1) * wrb + wb;
          if constexpr (kOdd) g -= (uint32_t)(uintptr_t)g & 2u;
          lds_dma16(g + min(16 * c, 196), base + kAQ + TT::kBS + 1024 * k);
        }
      }
      return;
    } else {
      // Q5_K records are 11 chunks of 16 bytes: 22 wave-wide 16-byte loads
      // when the rows are 16-byte aligned (row q / 11, chunk q % 11)
      if (w16) {
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          const int k = wave + 8 * i;
          if (k < kNT * 11 / 64) {
            const int q = 64 * k + lane, row = q / 11;
            const uint8_t* g = W + (size_t)min(n0 + row, a.N - 1) * wrb + wb + 16 * (q - 11 * row);
            lds_dma16(g, base + kAQ + TT::kBS + 1024 * k);
          }
        }
        return;
      }
    }
#pragma unroll
    for (int i = 0; i < (kWSlots + 7) / 8; ++i) {
      const int k = wave + 8 * i;
      if (k < kWSlots) {
        const int q = 64 * k + lane, row = q / kLoadD, part = q - kLoadD * row;
        const uint8_t* g = W + (size_t)min(n0 + row, a.N - 1) * wrb + wb + 4 * part;
        lds_dma4(g, base + kAQ + TT::kBS + 256 * k);
      }
    }
  };
  float dxr = 0.f;
  auto load_dx = [&](int b) { dxr = *reinterpret_cast<const float*>(dsrc + (size_t)b * kQ8_KBytes); };

  v16i acc[2], hi[2];
  v16f y[2];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) y[t][r] = 0.f;
  const v16i zero = {};
  const int sw = col & 15;
  // (kOdd) the low address bits of this lane's weight row
  const uint32_t row_addr = (uint32_t)(uintptr_t)(W + (size_t)min(n0 + 32 * wcol + col, a.N - 1) * wrb);

  auto step = [&](int b, const uint8_t* cur, int nxt, auto shift) {
    constexpr int kSh = decltype(shift)::value;  // byte offset of the Q6_K record in its LDS row
    const uint32_t sh = kSh == kRowShift ? (uint32_t)(row_addr + (uint32_t)b * TT::kRec) & 2u : (uint32_t)kSh;
    __builtin_amdgcn_s_waitcnt(0);  // this wave's loads of superblock b have landed
    __syncthreads();                // everyone's; superblock b - 1 is consumed
    const bool refill = b + 1 < nsb;
    if (refill && wave == 0) load_dx(b + 1);
    // this wave's share of superblock b + 1's direct loads goes out after
    // the half's second group (below): issued right after the barrier, every
    // wave's first group waited behind the workgroup's queued loads (the
    // MXFP4 GEMM measured 39.5 -> 37.8 us per call for the move)
    const uint8_t* AQ = cur;
    const uint8_t* row = cur + kAQ + TT::kBS + (32 * wcol + col) * kRowB;  // this lane's weight row
    const uint4* dxb = &dxq[b & 1][0];
    float dw, dmin = 0.f;
    v16f mn[2];
    if constexpr (k6) {
      // ql of groups s = 0, 2 (P0) and 1, 3 (P1), qh of all four, the 8 scales of the half
      const uint4 P0 = ld16<kSh>(row + 64 * h + 16 * kg, sh);
      const uint4 P1 = ld16<kSh>(row + 64 * h + 32 + 16 * kg, sh);
      const uint4 Q = ld16<kSh>(row + 128 + 32 * h + 16 * kg, sh);
      const uint2 s8 = *reinterpret_cast<const uint2*>(row + 192 + 8 * h);
      uint32_t sc0 = s8.x, sc1 = s8.y;
      if constexpr (kSh != 0) {
        const uint32_t s2 = *reinterpret_cast<const uint32_t*>(row + 200 + 20 * h);  // dword 50 or 52
        sc0 = __builtin_amdgcn_alignbyte(s8.y, s8.x, sh);
        sc1 = __builtin_amdgcn_alignbyte(s2, s8.y, sh);
      }
      const uint32_t dword = *reinterpret_cast<const uint32_t*>(row + 220);
      dw = fp16_to_fp32((dword >> (8 * sh)) & 0xffffu);
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const uint4 L = (s & 1) ? P1 : P0;
        const uint32_t lq[4] = {L.x, L.y, L.z, L.w}, hq[4] = {Q.x, Q.y, Q.z, Q.w};
        // this lane's 16 elements have one scale: 2 s + kg of the half
        const short sc = (short)(int8_t)((s < 2 ? sc0 : sc1) >> (16 * (s & 1) + 8 * kg));
        const v2s m = {sc, sc}, c = {(short)(128 - 32 * sc), (short)(128 - 32 * sc)};
        v4i lo_w, hi_w;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const uint32_t q = ((lq[i] >> (4 * (s >> 1))) & 0x0f0f0f0fu) |
                             ((s < 3 ? hq[i] << (4 - 2 * s) : hq[i] >> 2) & 0x30303030u);
          // p + 128 of values 0, 2 and of 1, 3 (p = sc (q - 32), 16 bits)
          const v2s te = __builtin_bit_cast(v2s, q & 0x00ff00ffu) * m + c;
          const v2s to = __builtin_bit_cast(v2s, __builtin_amdgcn_perm(0u, q, 0x0c030c01u)) * m + c;
          const uint32_t ue = __builtin_bit_cast(uint32_t, te), uo = __builtin_bit_cast(uint32_t, to);
          lo_w[i] = (int)(__builtin_amdgcn_perm(uo, ue, 0x06020400u) ^ 0x80808080u);
          hi_w[i] = (int)__builtin_amdgcn_perm(uo, ue, 0x07030501u);
        }
        const int chunk = (2 * (4 * h + s) + kg) ^ sw;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const v4i av = *reinterpret_cast<const v4i*>(AQ + (32 * t + col) * 256 + 16 * chunk);
          acc[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(av, lo_w, s == 0 ? zero : acc[t], 0, 0, 0);
          hi[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(av, hi_w, s == 0 ? zero : hi[t], 0, 0, 0);
        }
        if (s == 1 && refill) issue(b + 1, nxt);
      }
    } else {
      const uint4 hd = *reinterpret_cast<const uint4*>(row);  // d, dmin, 12 scale bytes
      dw = fp16_to_fp32(hd.x & 0xffffu);
      dmin = fp16_to_fp32(hd.x >> 16);
      const uint4 Q = *reinterpret_cast<const uint4*>(row + 16 + 16 * kg);  // qh bytes 16kg .. +15
      const uint4 L0 = *reinterpret_cast<const uint4*>(row + 48 + 64 * h + 16 * kg);       // qs of j = 2h
      const uint4 L1 = *reinterpret_cast<const uint4*>(row + 48 + 64 * h + 32 + 16 * kg);  // j = 2h + 1
      const uint32_t hq[4] = {Q.x, Q.y, Q.z, Q.w};
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int g = 4 * h + s;
        const uint4 L = (s >> 1) ? L1 : L0;
        const uint32_t lq[4] = {L.x, L.y, L.z, L.w};
        v4i bv;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          bv[i] = (int)(((lq[i] >> (4 * (s & 1))) & 0x0f0f0f0fu) | (((hq[i] >> g) & 0x01010101u) << 4));
        int sc, m;
        q4k_scale_min(g, hd.y, hd.z, hd.w, sc, m);
        const int chunk = (2 * g + kg) ^ sw;
        v16i I[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const v4i av = *reinterpret_cast<const v4i*>(AQ + (32 * t + col) * 256 + 16 * chunk);
          I[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(av, bv, zero, 0, 0, 0);
        }
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            int v = __mul24(I[t][r], sc) + (s == 0 ? 0 : acc[t][r]);
            pin(v);
            acc[t][r] = v;
          }
        if (s == 1 && refill) issue(b + 1, nxt);
      }
      // Mn of this half: bsums 8h + 4kg .. +3 of token 32t + col against the
      // mins of groups 4h + 2kg, 4h + 2kg + 1 (two bsums each) of row col
      int m_a, m_b, sdummy;
      q4k_scale_min(4 * h + 2 * kg, hd.y, hd.z, hd.w, sdummy, m_a);
      q4k_scale_min(4 * h + 2 * kg + 1, hd.y, hd.z, hd.w, sdummy, m_b);
      const v4h bm = {(_Float16)m_a, (_Float16)m_a, (_Float16)m_b, (_Float16)m_b};
      const v16f fz = {};
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const uint2 bs = *reinterpret_cast<const uint2*>(AQ + kAQ + (32 * t + col) * 32 + 16 * h + 8 * kg);
        const v4h am = {(_Float16)(short)(bs.x & 0xffffu), (_Float16)(short)(bs.x >> 16),
                        (_Float16)(short)(bs.y & 0xffffu), (_Float16)(short)(bs.y >> 16)};
        mn[t] = __builtin_amdgcn_mfma_f32_32x32x8f16(am, bm, fz, 0, 0, 0);
      }
    }
    // y += (dx dw) acc [- (dx dmin) Mn]: the factors of every output from a
    // bf16 outer-product MFMA per tile (token d = h + m + l against the
    // row's fp16 scale = f_h + f_l, K slots 0-5 of the kg = 0 lanes; the
    // kg = 1 lanes' slots are zero), then two VALU operations per output
    const uint32_t kz = kg ? 0u : 0xffffffffu;
    const uint32_t pw = bf16_split2(dw) & kz;
    const v4i bw = {(int)pw, (int)pw, (int)pw, 0};
    v4i bm = {};
    if constexpr (!k6) {
      const uint32_t pm = bf16_split2(dmin) & kz;
      bm = (v4i){(int)pm, (int)pm, (int)pm, 0};
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const uint4 d4 = dxb[32 * t + col];
      const v4i aq = {(int)(d4.x & kz), (int)(d4.y & kz), (int)(d4.z & kz), 0};
      const v16f fz = {};
      const v16f qw = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, aq),
                                                             __builtin_bit_cast(v8bf, bw), fz, 0, 0, 0);
      if constexpr (k6) {
#pragma unroll
        for (int r = 0; r < 16; ++r) y[t][r] = fmaf(qw[r], (float)(acc[t][r] + 256 * hi[t][r]), y[t][r]);
      } else {
        const v16f qm = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, aq),
                                                               __builtin_bit_cast(v8bf, bm), fz, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 16; ++r) y[t][r] = fmaf(-qm[r], mn[t][r], fmaf(qw[r], (float)acc[t][r], y[t][r]));
      }
    }
    if (refill && wave == 0) dxq[(b + 1) & 1][lane] = bf16_split3(dxr);  // slot last read a superblock ago
  };

  issue(0, 0);
  if (wave == 0) {
    load_dx(0);
    dxq[0][lane] = bf16_split3(dxr);
  }
  // Q6_K: the terms of four superblocks, then their sum into ysum with what
  // that addition rounds off kept in ylow (all of it where the running sum is the
  // larger one, which it is but for the first few or where it nearly cancels).  One chain over a row of 11008 values
  // had twice the error of the GEMV's short ones (against 64 bits, relative:
  // 1.3e-7, GEMV 0.70e-7; sums of eight without ylow 0.85e-7).
  v16f ysum[2] = {}, ylow[2] = {};
  auto fold = [&]() {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const v16f s = ysum[t] + y[t];
      ylow[t] += (ysum[t] - s) + y[t];
      ysum[t] = s;
      y[t] = v16f{};
    }
  };
  for (int b = 0; b < nsb; b += 2) {
    step(b, ring0, 1, std::integral_constant<int, kOdd ? kRowShift : 0>{});
    if (b + 1 < nsb) step(b + 1, ring1, 0, std::integral_constant<int, kOdd ? kRowShift : k6 ? 2 : 0>{});
    if (k6 && (b & 2)) fold();
  }
  if (k6) {
    fold();
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r)  // an infinite sum leaves NaN in ylow
        y[t][r] = ysum[t][r] + (fabsf(ysum[t][r]) < __builtin_huge_valf() ? ylow[t][r] : 0.f);
  }

  // both parities' partial sums -> two LDS planes (reusing the ring) -> Y
  __syncthreads();
  float* even_plane = reinterpret_cast<float*>(ring0);
  float* odd_plane = reinterpret_cast<float*>(ring1);
  tile_partials_to_lds(y, wcol, lane, h ? odd_plane : even_plane);
  __syncthreads();
  tile_store_from_lds(
      wave, lane, even_plane, odd_plane, mrows, min(kNT, a.N - n0),
      [&](int rr) {
        return a.Y + (kGroup ? group_dst_row(a.grp, m0, rr) : (long long)(m0 + rr) * a.ldy) + n0;
      },
      [](float e, float o) { return e + o; });
}

// MFMA path: prefill shapes with 4-byte aligned weight rows, Q6_K also with
// 2-byte aligned ones (kq_odd: a row of an odd number of 210-byte records
// leaves the next one there).  The weights themselves are 4-byte aligned: of
// ones that are not, the first row would be read from before its first byte.
// The small-batch kernel and the GEMVs take everything else.
template <KQ F>
bool kq_odd(size_t ldw, size_t w_es, size_t K) {
  return F == KQ::Q6_K && (K % 512 != 0 || ldw % 4 != 0 || w_es % 4 != 0);
}

template <KQ F>
bool gemm_kq_ok(const uint8_t* W, const void* Xq, const float* Y, size_t N, size_t K, size_t M,
                const RowStrides& st) {
  constexpr size_t kRec = KTile<F>::kRec;
  constexpr size_t kAlign = F == KQ::Q6_K ? 2 : 4;
  const size_t ldw = N > 1 ? st.ldw : K / 256 * kRec;
  // below 16 activation rows only when the GEMV's LDS cannot hold a row
  return (M >= 16 || !staged_gemv_fits(F == KQ::Q6_K ? 3 : 4, K)) && N > 0 && K > 0 && K % 256 == 0 &&
         W != nullptr && Xq != nullptr && Y != nullptr &&
         aligned(W, 4) && ldw % kAlign == 0 && aligned(Xq, 4) && aligned(Y, 4) && N <= (size_t)INT32_MAX &&
         K <= (size_t)INT32_MAX && M <= (size_t)INT32_MAX && strides_ok(st, K / 256 * kRec, 2, K, N, N, M) &&
         ((N + kNT - 1) / kNT) * ((M + kMT - 1) / kMT) <= (size_t)INT32_MAX;
}

template <KQ F>
void gemm_kq(const uint8_t* W, const uint8_t* Xq, float* Y, size_t N, size_t K, size_t M, const RowStrides& st) {
  const size_t ldw = N > 1 ? st.ldw : K / 256 * KTile<F>::kRec;
  GemmArgs ga{W, Xq, Y, (int)N, (int)K, (int)M, ldw, (long long)st.ldy, GroupTiles{}};
  const size_t tiles = ((N + kNT - 1) / kNT) * ((M + kMT - 1) / kMT);
  if (kq_odd<F>(ldw, 0, K))
    kq_mfma_gemm<false, F, F == KQ::Q6_K><<<dim3((unsigned)tiles), kThreads, 0, current_stream()>>>(ga);
  else
    kq_mfma_gemm<false, F><<<dim3((unsigned)tiles), kThreads, 0, current_stream()>>>(ga);
  check_launch(F == KQ::Q6_K ? "q6k_mfma_gemm" : "q5k_mfma_gemm");
}

}  // namespace

void mul_mat_q6k(const uint8_t* W, const float* X, uint8_t* Xq, float* Y, size_t N, size_t K, size_t M,
                 const RowStrides& st) {
  if (small_batch(3, W, X, Xq, nullptr, nullptr, Y, N, K, M, st)) return;
  if (X == nullptr || !aligned(X, 4) || !gemm_kq_ok<KQ::Q6_K>(W, Xq, Y, N, K, M, st)) {
    if (!small_batch(3, W, X, Xq, nullptr, nullptr, Y, N, K, M, st, false))
      decode_q6_k(W, X, Xq, Y, N, K, M, st);
    return;
  }
  quantize_q8_k_rows(X, st.ldx, Xq, M, K);
  gemm_kq<KQ::Q6_K>(W, Xq, Y, N, K, M, st);
}

bool gemm_kq_try(bool q6, const uint8_t* W, const float* X, uint8_t* Xq, float* Y, size_t N, size_t K,
                 size_t M, const RowStrides& st) {
  if (X == nullptr || !aligned(X, 4)) return false;
  if (q6) {
    if (!gemm_kq_ok<KQ::Q6_K>(W, Xq, Y, N, K, M, st)) return false;
    quantize_q8_k_rows(X, st.ldx, Xq, M, K);
    gemm_kq<KQ::Q6_K>(W, Xq, Y, N, K, M, st);
  } else {
    if (!gemm_kq_ok<KQ::Q5_K>(W, Xq, Y, N, K, M, st)) return false;
    quantize_q8_k_rows(X, st.ldx, Xq, M, K);
    gemm_kq<KQ::Q5_K>(W, Xq, Y, N, K, M, st);
  }
  return true;
}

void mul_mat_q5k(const uint8_t* W, const float* X, uint8_t* Xq, float* Y, size_t N, size_t K, size_t M,
                 const RowStrides& st) {
  if (small_batch(4, W, X, Xq, nullptr, nullptr, Y, N, K, M, st)) return;
  if (X == nullptr || !aligned(X, 4) || !gemm_kq_ok<KQ::Q5_K>(W, Xq, Y, N, K, M, st)) {
    if (!small_batch(4, W, X, Xq, nullptr, nullptr, Y, N, K, M, st, false))
      decode_q5_k(W, X, Xq, Y, N, K, M, st);
    return;
  }
  quantize_q8_k_rows(X, st.ldx, Xq, M, K);
  gemm_kq<KQ::Q5_K>(W, Xq, Y, N, K, M, st);
}

void mul_mat_q6k_quantized(const uint8_t* W, const uint8_t* Xq, float* Y, size_t N, size_t K, size_t M,
                           const RowStrides& st) {
  if (!gemm_kq_ok<KQ::Q6_K>(W, Xq, Y, N, K, M, st)) {
    if (!small_batch_quantized(3, W, Xq, nullptr, nullptr, Y, N, K, M, st, false))
      decode_quantized(3, W, Xq, nullptr, nullptr, Y, N, K, M, st);
    return;
  }
  gemm_kq<KQ::Q6_K>(W, Xq, Y, N, K, M, st);
}

void mul_mat_q5k_quantized(const uint8_t* W, const uint8_t* Xq, float* Y, size_t N, size_t K, size_t M,
                           const RowStrides& st) {
  if (!gemm_kq_ok<KQ::Q5_K>(W, Xq, Y, N, K, M, st)) {
    if (!small_batch_quantized(4, W, Xq, nullptr, nullptr, Y, N, K, M, st, false))
      decode_quantized(4, W, Xq, nullptr, nullptr, Y, N, K, M, st);
    return;
  }
  gemm_kq<KQ::Q5_K>(W, Xq, Y, N, K, M, st);
}

bool mul_mat_id_kq_grouped_ok(bool q6, const uint8_t* W, size_t xq_bytes, const float* Y, size_t N, size_t K,
                              const RowStrides& st, const PairArgs& pr, int n_pairs, const void* ws,
                              size_t ws_bytes) {
  const size_t rb = K / 256 * (q6 ? kQ6_KBytes : kQ5_KBytes);
  const size_t ldw = N > 1 ? st.ldw : rb;
  const size_t align = q6 ? 2 : 4;
  return N > 0 && n_pairs > 0 && K > 0 && K % 256 == 0 && W != nullptr && Y != nullptr &&
         aligned(W, 4) && ldw % align == 0 && aligned(Y, 4) && xq_bytes < ((size_t)1 << 32) && aligned(ws, 16) &&
         ws_bytes >= moe_group_bytes(n_pairs, pr.n_as) && pr.w_es % (long long)align == 0 && pr.n_as <= kMaxExperts &&
         N <= (size_t)INT32_MAX && K <= (size_t)INT32_MAX && strides_ok(st, rb, 2, K, N, N, 1) &&
         (size_t)moe_tile_bound(n_pairs, pr.n_as) * ((N + kNT - 1) / kNT) <= (size_t)INT32_MAX;
}

void mul_mat_id_kq_grouped(bool q6, const uint8_t* W, const uint8_t* Xq, float* Y, size_t N, size_t K,
                           const RowStrides& st, const PairArgs& pr, int n_pairs, void* ws) {
  const MoeGroups g = moe_group(pr, n_pairs, ws);
  const size_t ldw = N > 1 ? st.ldw : K / 256 * (q6 ? kQ6_KBytes : kQ5_KBytes);
  GemmArgs ga{W, Xq, Y, (int)N, (int)K, kMT, ldw, 0, group_tiles(g, pr)};
  const size_t wgs = (size_t)g.tmax * ((N + kNT - 1) / kNT);
  if (q6) {
    if (kq_odd<KQ::Q6_K>(ldw, (size_t)pr.w_es, K))
      kq_mfma_gemm<true, KQ::Q6_K, true><<<dim3((unsigned)wgs), kThreads, 0, current_stream()>>>(ga);
    else
      kq_mfma_gemm<true, KQ::Q6_K><<<dim3((unsigned)wgs), kThreads, 0, current_stream()>>>(ga);
    check_launch("q6k_mfma_gemm");
  } else {
    kq_mfma_gemm<true, KQ::Q5_K><<<dim3((unsigned)wgs), kThreads, 0, current_stream()>>>(ga);
    check_launch("q5k_mfma_gemm");
  }
}

}  // namespace weft
