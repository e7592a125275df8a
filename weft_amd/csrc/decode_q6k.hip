// Batch-1 decode GEMV for Q6_K x Q8_K: production_mul_mat_q6_k_decode /
// production_mul_mat_q6_k at M = 1 (examples/kernels/mul_mat/q6_k_decode.py,
// q6_k.py:9-37), rows of up to 4 * 4096 values.
//
// Semantics (ggml_vec_dot_q6_K_q8_K_generic, ggml-cpu/quants.c:800-853):
//   y = sum_b (dw_b dx_b) * sum_{j<16} sc_j * sum_{16} (q6 - 32) * x      (exact int32)
// computed as sum_j sc_j * (P_j - 32 X_j), P_j = sum q6 x with q6 in [0, 63]
// (an exact int8 operand) and X_j the 16 activation values' sum.
//
// gfx950 mapping, as the Q4_K / Q5_K batch-1 kernels: lane l of a row owns
// superblock l / 4 and its 64-element chunk g = l % 4 (half h = g / 2 of the
// record; the low nibbles of ql[64h .. 64h + 63] for even g, the high ones
// for odd g; qh[32h .. 32h + 31]; scales 4g .. 4g + 3).  A 210-byte record
// is 2-byte aligned for odd superblocks, so the lane's bytes come into VGPRs
// from the dword below them (16-byte loads at 4-byte aligned addresses) and
// are aligned with v_alignbyte.  The 64 activation values and their four
// 16-sums are held in VGPRs; values are formed four at a time and meet the
// activation in v_dot4_i32_i8.  One fp32 term per superblock and lane, a
// DPP wave sum per row, one row of lookahead.  The activation is quantized in
// every workgroup (bit-exact with quantize_row_q8_K_ref); workgroup 0 writes Xq.
#include <algorithm>

#include "activation.h"
#include "kernels.h"
#include "runtime.h"
#include "weft_common.h"
#include "weft_hip.h"

namespace weft {
namespace {

constexpr int kThreads = 1024;
constexpr int kWaves = kThreads / kWave;

struct Q6Args {
  const uint8_t* W;
  const float* X;
  uint8_t* xq_out;
  float* Y;
  int N, K;
  int rows_per_wg;
  size_t ldw;
};

// Rows longer than one step of 4096 values (KS > 1): the waves form groups of
// KS, wave w takes step w % KS (an even share of the superblocks, so its
// activation slice still fits the registers) of the rows of group w / KS, and
// the KS partial sums of a row are added in step order at the end.
// One call, against the staged GEMV, whose rows all pass through LDS (weights
// past the Infinity Cache): 4096 x 11008 (43 superblocks, 2-byte rows) 14.1 ->
// 11.8 us, 14336 x 4352 20.1 -> 16.3, 1024 x 14336 10.8 -> 7.1.
// kOdd: rows that are only 2-byte aligned, so a lane's shift depends on its row.
// kMany: a row's loads all go out before the row before it is computed, which
// pays where a wave has several rows (one call, weights past the Infinity Cache:
// 28672 x 4096 24.4 -> 23.0 us, 14336 x 12288 36 -> 33) and costs where it has one
// or two, or short ones (weights in it: 9856 x 1536 6.1 -> 6.5, 12288 x 2048 and
// 6144 x 6144 5 %); kOdd rows do not
// gain (4096 x 11008 11.6 -> 11.9).
template <int KS, bool kOdd, bool kMany>
__global__ void __launch_bounds__(kThreads) q6k_gemv_m1_kernel(Q6Args a) {
  constexpr int kGroups = kWaves / KS;
  extern __shared__ __align__(16) char lds[];  // Q8_K activation row, then the steps' partial sums
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int K = a.K;
  const int nsb = K >> 8;  // <= 16 KS
  const int st = wave % KS, grp = wave / KS;
  const int spb = (nsb + KS - 1) / KS;  // <= 16
  const bool live = (lane >> 2) < spb && st * spb + (lane >> 2) < nsb;
  const int sb = min(st * spb + (lane >> 2), nsb - 1), g = lane & 3, h = g >> 1;
  float* part = reinterpret_cast<float*>(lds + q8k_lds_row_bytes(K));  // [row - row_base][step]
  const uint32_t rec = (uint32_t)(kQ6_KBytes * sb);
  // A row is read from the dword that holds its first byte, rbit (0 or 2) bytes
  // before it: the row's address is then the wave's, and a lane's record lies
  // `shift` (0 or 2) past the dword at its own offset `base`.  (With the shift
  // taken from the lane's address instead, every row's loads need 64-bit
  // addresses computed per lane, and the rows a wave
  // has in flight fall behind: one call, weights past the Infinity Cache, 28672 x
  // 4096 25.7 us where this takes 23.0, 4096 x 11008 12.4 and 11.8, 14336 x
  // 16384 51.1 and 44.4.)
  auto row_bit = [&](int row) -> uint32_t {
    if constexpr (!kOdd) return 0u;
    return ((uint32_t)row * (uint32_t)a.ldw) & 2u;  // W itself is 4-byte aligned
  };
  auto shift = [&](uint32_t rbit) -> uint32_t { return (rec + rbit) & 2u; };
  const size_t rb = a.ldw;
  const int row_base = blockIdx.x * a.rows_per_wg, row_first = row_base + grp;
  const int row_end = min(a.N, row_base + a.rows_per_wg);
  const int nrows = grp < kGroups && row_first < row_end ? (row_end - row_first + kGroups - 1) / kGroups : 0;

  Q8KStager16<1> stager;
  stager.prefetch(a.X, (size_t)K, K, 0, 1);
  __builtin_amdgcn_sched_barrier(0);

  // 17 dwords of ql, 9 of qh, 2 of scales, and d.  A 17th / 9th / 2nd dword
  // only carries data at a shift of 2; at 0 the last dword before it is read
  // again (the region may end at the row's end).  kOdd reads d by itself: as a
  // dword at a shift of 0 it would reach two bytes past the record, and the last
  // row's last record is the end of the weights.  (Rows of whole pairs of records
  // end with one at a shift of 2, whose dword ends where the record does.)
  struct RowBuf {
    uint32_t ql[17], qh[9], sc[2], d;
  };
  auto issue = [&](RowBuf& buf, int k) {
    const int row = min(row_first + k * kGroups, a.N - 1);  // clamped: always a valid row
    const uint32_t rbit = row_bit(row), sh = shift(rbit), base = rec + rbit - sh;
    const uint8_t* rp = a.W + ((size_t)row * rb - rbit);
    // the dword at o, at a shift of 2 the one after it (the two forms schedule
    // differently: 14336 x 11008 32.6 us with the second one, 30.5 with the first;
    // 4096 x 4096 2 % faster with the second)
    auto last = [&](uint32_t o) {
      if constexpr (kOdd)
        return rp + (o + 2 * sh);
      else
        return rp + o + (sh ? 4 : 0);
    };
    const uint32_t o_ql = base + 64 * h, o_qh = base + 128 + 32 * h, o_sc = base + 192 + 4 * g;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint4 v = *reinterpret_cast<const uint4*>(rp + o_ql + 16 * i);
      buf.ql[4 * i] = v.x, buf.ql[4 * i + 1] = v.y, buf.ql[4 * i + 2] = v.z, buf.ql[4 * i + 3] = v.w;
    }
    buf.ql[16] = *reinterpret_cast<const uint32_t*>(last(o_ql + 60));
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint4 v = *reinterpret_cast<const uint4*>(rp + o_qh + 16 * i);
      buf.qh[4 * i] = v.x, buf.qh[4 * i + 1] = v.y, buf.qh[4 * i + 2] = v.z, buf.qh[4 * i + 3] = v.w;
    }
    buf.qh[8] = *reinterpret_cast<const uint32_t*>(last(o_qh + 28));
    buf.sc[0] = *reinterpret_cast<const uint32_t*>(rp + o_sc);
    buf.sc[1] = *reinterpret_cast<const uint32_t*>(last(o_sc));
    if constexpr (kOdd)
      buf.d = *reinterpret_cast<const uint16_t*>(rp + (rec + rbit + 208));
    else
      buf.d = *reinterpret_cast<const uint32_t*>(rp + base + 208);
  };
  RowBuf bufA, bufB;
  issue(bufA, 0);
  __builtin_amdgcn_sched_barrier(0);

  stager.finish(a.X, (size_t)K, blockIdx.x == 0 ? a.xq_out : nullptr, K, 0, 1, lds);
  __syncthreads();

  // this lane's 64 activation values (part a: elements 0-31 of the chunk,
  // part b: 32-63) and the sums of its four 16-value groups
  int xa[8], xb[8];
  int xs[4];
  float dx;
  {
    const Q8KView v = q8k_view(lds, K, 0);
    const int8_t* x = v.qs + 256 * sb + 64 * g;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int4 p = *reinterpret_cast<const int4*>(x + 16 * i);
      const int4 q = *reinterpret_cast<const int4*>(x + 32 + 16 * i);
      xa[4 * i] = p.x, xa[4 * i + 1] = p.y, xa[4 * i + 2] = p.z, xa[4 * i + 3] = p.w;
      xb[4 * i] = q.x, xb[4 * i + 1] = q.y, xb[4 * i + 2] = q.z, xb[4 * i + 3] = q.w;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int* src = j < 2 ? xa + 4 * j : xb + 4 * (j - 2);
      int s = dot4(0x01010101, src[0], 0);
      s = dot4(0x01010101, src[1], s);
      s = dot4(0x01010101, src[2], s);
      xs[j] = dot4(0x01010101, src[3], s);
    }
    dx = v.d[sb];
  }
  const uint32_t nsh = 4 * (g & 1);        // nibble: low for even g, high for odd
  const uint32_t hsh = 4 * (g & 1);        // qh bit pairs 2s: s = 2 (g & 1) and 2 (g & 1) + 1

  auto compute = [&](const RowBuf& buf, int k) {
    const uint32_t sh = shift(row_bit(row_first + k * kGroups));
    uint32_t ql[16], qh[8];
#pragma unroll
    for (int i = 0; i < 16; ++i) ql[i] = __builtin_amdgcn_alignbyte(buf.ql[i + 1], buf.ql[i], sh);  // sh 0 or 2
#pragma unroll
    for (int i = 0; i < 8; ++i) qh[i] = __builtin_amdgcn_alignbyte(buf.qh[i + 1], buf.qh[i], sh);
    const uint32_t sc4 = __builtin_amdgcn_alignbyte(buf.sc[1], buf.sc[0], sh);
    const float dw = fp16_to_fp32(kOdd ? buf.d : (buf.d >> (8 * sh)) & 0xffffu);
    // part a: ql[0 .. 31] with qh bits hsh .. hsh + 1; part b: ql[32 .. 63]
    // with bits hsh + 2 .. hsh + 3 (element l of both parts reads qh[l])
    int P[4] = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t hb = qh[i] >> hsh;
      const uint32_t va = ((ql[i] >> nsh) & 0x0f0f0f0fu) | ((hb & 0x03030303u) << 4);
      const uint32_t vb = ((ql[8 + i] >> nsh) & 0x0f0f0f0fu) | ((hb & 0x0c0c0c0cu) << 2);
      P[i >> 2] = dot4((int)va, xa[i], P[i >> 2]);
      P[2 + (i >> 2)] = dot4((int)vb, xb[i], P[2 + (i >> 2)]);
    }
    int tot = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int scj = (int)(int8_t)((sc4 >> (8 * j)) & 0xffu);
      tot += scj * (P[j] - 32 * xs[j]);  // |P - 32 X| <= 16 * 32 * 128: exact
    }
    const int bsum = sum4(live ? tot : 0);  // the superblock's four lanes
    const float p = dw * dx, b = (float)bsum;
    float t = (lane & 3) == 0 && live ? p * b : 0.f;
    if constexpr (KS > 1) {
      // with what the product of the scales rounds off: the steps' sums have
      // more additions than the staged kernel's (error against 64 bits at
      // 11008 values, relative: 0.76e-7 without it, staged 0.71e-7)
      const float e = fmaf(dw, dx, -p);
      if ((lane & 3) == 0 && live && fabsf(p) < __builtin_huge_valf()) t = fmaf(e, b, t);
    }
    const float y = wave_sum_f(t);
    if (lane == 0) {
      if constexpr (KS == 1)
        a.Y[row_first + k * kGroups] = y;
      else
        part[(row_first + k * kGroups - row_base) * KS + st] = y;
    }
  };

  int k = 0;
  for (; k + 2 < nrows; k += 2) {
    issue(bufB, k + 1);
    if constexpr (kMany) __builtin_amdgcn_sched_barrier(0);
    compute(bufA, k);
    issue(bufA, k + 2);
    if constexpr (kMany) __builtin_amdgcn_sched_barrier(0);
    compute(bufB, k + 1);
  }
  if (nrows - k == 2) {
    issue(bufB, k + 1);
    compute(bufA, k);
    compute(bufB, k + 1);
  } else if (nrows - k == 1) {
    compute(bufA, k);
  }
  if constexpr (KS > 1) gemv_add_steps<KS>(part, a.Y, row_base, row_end);
}

}  // namespace

namespace {
template <bool kOdd, bool kMany>
void launch_steps(int ks, int grid, size_t lds, const Q6Args& a) {
  switch (ks) {
    case 1: q6k_gemv_m1_kernel<1, kOdd, kMany><<<grid, kThreads, lds, current_stream()>>>(a); break;
    case 2: q6k_gemv_m1_kernel<2, kOdd, kMany><<<grid, kThreads, lds, current_stream()>>>(a); break;
    case 3: q6k_gemv_m1_kernel<3, kOdd, kMany><<<grid, kThreads, lds, current_stream()>>>(a); break;
    default: q6k_gemv_m1_kernel<4, kOdd, kMany><<<grid, kThreads, lds, current_stream()>>>(a); break;
  }
}
}  // namespace

// Launches the kernel above when the call suits it: one activation row of
// K <= 4 * 4096, 16-byte aligned X, W 4-byte aligned (of weights that begin in
// the middle of a dword the first row would be read from before its first byte)
// with rows a multiple of 2 bytes apart, Xq 4-byte aligned.
bool decode_q6k_m1(const uint8_t* W, const float* X, uint8_t* Xq, float* Y, size_t N, size_t K,
                   const RowStrides& st) {
  const size_t rb = K / 256 * kQ6_KBytes;
  const size_t ldw = N > 1 ? st.ldw : rb;
  if (N == 0 || K == 0 || K > 4 * 4096 || K % 256 != 0 || X == nullptr || Xq == nullptr || W == nullptr ||
      Y == nullptr || !aligned(X, 16) || !aligned(W, 4) || ldw % 2 != 0 || !aligned(Y, 4) ||
      !aligned(Xq, 4) || N > (size_t)INT32_MAX || (N > 1 && ldw < rb) || ldw >= ((size_t)1 << 40))
    return false;
  // The staged GEMV's 16-byte copies keep ahead of this kernel's per-lane reads
  // where three or four whole steps a row and many rows leave nothing else to
  // wait for: 14336 x 12288 32.7 us here, 32.0 there, 28672 x 16384 84.3 and
  // 80.5 (equal at 11008 rows; rows of an odd number of records 5 % faster here).
  if (K % 512 == 0 && K >= 3 * 4096 && N >= 14336) return false;
  const int cus = cu_count();
  const int ks = (int)((K + 4095) / 4096);
  const size_t groups = (size_t)(kWaves / ks);  // rows a workgroup works on at once
  const size_t wgs = std::max<size_t>(1, std::min<size_t>((size_t)cus, (N + groups - 1) / groups));
  Q6Args a;
  a.W = W;
  a.X = X;
  a.xq_out = Xq;
  a.Y = Y;
  a.N = (int)N;
  a.K = (int)K;
  // a CompileOptions NC binding sets the weight rows per workgroup
  const int nc = tile_bindings().nc;
  a.rows_per_wg = nc > 0 ? (int)std::min<size_t>(N, (size_t)nc) : (int)((N + wgs - 1) / wgs);
  a.ldw = ldw;
  const int grid = (int)((N + a.rows_per_wg - 1) / a.rows_per_wg);
  const size_t lds = q8k_lds_row_bytes((int)K) + (ks > 1 ? 4 * (size_t)ks * a.rows_per_wg : 0);
  if (lds > max_lds_per_block()) return false;
  if (K % 512 != 0 || ldw % 4 != 0)
    launch_steps<true, false>(ks, grid, lds, a);
  else if (K > 2048 && N >= (ks >= 3 ? 8192 : 12288))  // where the two cross, cold and warm
    launch_steps<false, true>(ks, grid, lds, a);
  else
    launch_steps<false, false>(ks, grid, lds, a);
  check_launch("q6k_gemv_m1_kernel");
  return true;
}

}  // namespace weft
