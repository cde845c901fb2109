// Draft-side sampling table of the serial last-write refinement for gfx950
// (kernels/dspine.py:505-613, serial_rs_table): for every block row n and sender lane j,
//   e      = sqrt(C) * codebook[sender]                            [C]
//   gate   = sigmoid(q[n] + e @ pg^T + gb),  value = e @ pv^T (+ res_emb[sender] @ res_proj^T)
//   msg    = gate * value                                          [R]
//   ref    = x[n] + scale[n] * (msg @ w_last^T)                    [H]
//   T[n, j, c] = (ref / sqrt(mean(ref^2) + eps) * norm_w) . head[n, c]
// in float32 accuracy on the bf16 matrix cores (v_mfma_f32_16x16x32_bf16, float32 accumulation): a
// float32 operand is three bf16 parts (split2), a bf16 operand one, and a product of two float32
// operands is the six part products that reach float32's last bit.  Three launches:
//   k_rs_message  sender rows x R: the gathered codebook rows times [pg; pv]^T, scaled, with the gate,
//                 the value and their product in the epilogue -> msg's parts [n*K, 3, R]; its last
//                 workgroups make w_last's parts [H, 3, R]
//   k_rs_table    (eight units of 16 senders, H slice): msg times w_last^T in 16 x 16 output blocks
//                 that are already the B operand of the second product against the 16 candidates'
//                 head rows, so ref never leaves registers; partial sums of ref^2 and of the dot
//                 products
//   k_rs_finish   the slices combined, divided by sqrt(mean + eps)
//
// What bounds it: matrix-core issue and the clock under it.  n 960, K 16, H 4096, R 512, C 1024 is 98.7
// GFLOP of float32 products, 489 GFLOP in bf16 parts: 445 us, 1.1 PFLOP/s (the library's bf16 product
// of 8192^3 runs at 1.17 on the same card).  Float32 MFMAs (16x16x4, 154 TFLOP/s at best) took 942 us.
// Relative error against float64: 3.5e-7 (float32 MFMAs: 5.5e-7; they round after every 4 k, these
// after every 32).
//
// MFMA operand layout (16x16x32, one wave): lane l holds A[l % 16][8g ..] and B[8g ..][l % 16] for the
// 8 k of its lane group g = l / 16, and receives D[4g + v][l % 16], v = 0..3.
#include <math.h>
#include <string.h>

#include "dsv_common.h"

namespace dsv {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef __bf16 bh2 __attribute__((ext_vector_type(2)));
typedef __bf16 bh8 __attribute__((ext_vector_type(8)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));
typedef f4 f4u __attribute__((aligned(4)));  // 16-byte vectors at the rows' own alignment
typedef u4 u4u __attribute__((aligned(8)));

constexpr int RS_RMAX = 512;
constexpr int RS_B = 128;   // tile: columns of the left operand (r or h) and senders of a workgroup
constexpr int RS_KS = 32;   // k depth of a stage: one v_mfma_f32_16x16x32_bf16
constexpr int RS_MKS = 64;  // of a stage of the message kernel
constexpr int RS_PLANE = RS_B * RS_KS * 2;  // bytes of one bf16 part of a staged tile

struct RsArgs {
  const uint16_t* raw;   // [m, H] bf16 bits (row stride raw_stride)
  const float* rms;      // [m]
  const uint16_t* query; // [m, >= R] bf16 bits (row stride query_stride)
  const int64_t* anchors;  // [bs]
  const int64_t* cand;     // [n, K]
  const uint16_t* codebook;  // [V, C] bf16 bits
  const float* pg;         // [R, C]
  const float* pv;         // [R, C]
  const float* gb;         // [R]
  const float* w_last;     // [H, R]
  const float* norm_w;     // [H]
  const uint16_t* head;    // lm_head [V, H] bf16 bits, or the candidate head [n, K, H]
  const uint16_t* res_emb; // [V, RR] bf16 bits or NULL
  const float* res_proj;   // [R, RR]
  int64_t raw_stride, query_stride;
  int32_t T, K, H, R, C, RR;
  int32_t n, head_is_cand;
  float eps, sqrt_c;
  uint16_t* msg;    // [n * K, 3, R] workspace: the message's bf16 parts
  uint16_t* wsplit; // [H, 3, R] workspace: w_last's bf16 parts
  float* part;      // [parts, units, 16 + 16 * KB * 16] workspace
  float* out;       // [n, K, K]
  int32_t KB;       // ceil(K / 16): candidate blocks
  int32_t units;    // n * KB: (row, 16-sender block) pairs
  int32_t hs, parts;  // columns of an H slice (a multiple of the tile's); partial sums a unit leaves
  int32_t sblocks;  // 128-sender blocks of the message
};

__device__ __forceinline__ float bf(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }
__device__ __forceinline__ f4 mfma(u4 a, u4 b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bh8, a), __builtin_bit_cast(bh8, b), c, 0, 0, 0);
}

// x = hi + mid + lo, each bf16 (8 significant bits, round to nearest even): exact for finite float32 of
// 2^-110 and above.  Below, lo and then mid end under the smallest bf16 (16 bits are left at 2^-118, 8 at
// 2^-126): what is lost is under 2^-133 an operand, so it shows in a table entry only where a code or a write
// scale of 2^100 and more multiplies it.  hi is held to the largest bf16, so that a finite x above it stays
// finite against a zero; an infinite x is (largest, inf, finite): its product with a bf16 operand is the
// infinity or, against zero, the NaN that it is.  (Against a second split operand it may be NaN for inf, in
// ref alone: an infinite ref makes its dot products over its norm NaN either way.)  Two values a call, packed.
__device__ __forceinline__ void split2(float a, float b, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
  const float top = __uint_as_float(0x7F7F0000u);  // the largest bf16
  hi = __builtin_bit_cast(uint32_t, __builtin_convertvector((f2{__builtin_amdgcn_fmed3f(a, -top, top),
                                                                __builtin_amdgcn_fmed3f(b, -top, top)}), bh2));
  const float ra = a - __uint_as_float(hi << 16), rb = b - __uint_as_float(hi & 0xFFFF0000u);
  mid = __builtin_bit_cast(uint32_t, __builtin_convertvector((f2{ra, rb}), bh2));
  // (inf - inf is NaN: the bound, below every finite x's lo)
  const float la = fmaxf(ra - __uint_as_float(mid << 16), -1e34f);
  const float lb = fmaxf(rb - __uint_as_float(mid & 0xFFFF0000u), -1e34f);
  lo = __builtin_bit_cast(uint32_t, __builtin_convertvector((f2{la, lb}), bh2));
}
__device__ __forceinline__ void split8(const f4& x, const f4& y, u4& hi, u4& mid, u4& lo) {
  uint32_t h, m, l;
  split2(x[0], x[1], h, m, l);
  hi[0] = h, mid[0] = m, lo[0] = l;
  split2(x[2], x[3], h, m, l);
  hi[1] = h, mid[1] = m, lo[1] = l;
  split2(y[0], y[1], h, m, l);
  hi[2] = h, mid[2] = m, lo[2] = l;
  split2(y[2], y[3], h, m, l);
  hi[3] = h, mid[3] = m, lo[3] = l;
}

// A staged tile's part: bf16 rows of 32 k, 64 bytes a row, its four 16-byte chunks (8 k each) placed
// at chunk ^ (row / 2 % 4): eight lanes of a fragment read (eight rows, one chunk) cover the banks
// once (placed at chunk ^ (row / 4 % 4), half of the reads' cycles were bank conflicts).
__device__ __forceinline__ int tile_at(int row, int kc) { return row * 64 + ((kc ^ (row >> 1)) & 3) * 16; }
// the same for stages of 64 k: 128 bytes a row, eight chunks
__device__ __forceinline__ int tile_at64(int row, int kc) { return row * 128 + ((kc ^ (row >> 1)) & 7) * 16; }
// 16 bytes a lane from memory to LDS (the wave's 64 chunks in lane order from `dst`)
__device__ __forceinline__ void to_lds(const uint16_t* src, char* dst) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                   (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}
// this wave's copies to LDS have landed, and every wave's; every wave is done reading the other buffer
__device__ __forceinline__ void stage_wait() {
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
  __syncthreads();
}
__device__ __forceinline__ u4 lds16(const char* p) { return *reinterpret_cast<const u4*>(p); }
__device__ __forceinline__ void put16(char* p, u4 v) { *reinterpret_cast<u4*>(p) = v; }

// The sender token of sender row i = n * K + j: the anchor on a request's first block row, else
// candidate j of the previous row.
__device__ __forceinline__ int64_t sender_of(const RsArgs& A, int64_t i) {
  const int64_t n = i / A.K, j = i - n * A.K;
  const int tm = (int)(n % (A.T - 1));
  return tm == 0 ? A.anchors[n / (A.T - 1)] : A.cand[(n - 1) * A.K + j];
}
// The state row (of the [bs*T] rows) block row n refines.
__device__ __forceinline__ int64_t state_row(const RsArgs& A, int64_t n) {
  return n / (A.T - 1) * A.T + 1 + n % (A.T - 1);
}

// ---------------------------------------------------------------------------------------
// k_rs_message: 128 sender rows x 64 R columns of both the gate and the value (the tile's 128 left
// rows: pg rows r0.., then pv rows r0..).  Wave (w & 1, w >> 1) has 64 senders and 32 columns of
// each; D[4g + v][li] is column 4g + v of sender li.  A stage is 64 k deep (at the sizes above
// 128 us where 32 deep, with half the products between barriers, took 139; 148 now in the median under the
// profiler); the weights' parts are made while
// staging, the next stage's loads in flight in registers.
// ---------------------------------------------------------------------------------------
// w_last's parts, [H, 3, R]: eight values a thread.
__device__ __forceinline__ void split_w_last(const RsArgs& A, int64_t q) {
  const int rc = A.R / 8;
  if (q >= (int64_t)A.H * rc) return;
  const int64_t h = q / rc, c = q - h * rc;
  const float* p = A.w_last + h * A.R + 8 * c;
  u4 hi, mid, lo;
  const f4 x = *reinterpret_cast<const f4u*>(p), y = *reinterpret_cast<const f4u*>(p + 4);
  split8(x, y, hi, mid, lo);
  uint16_t* o = A.wsplit + h * 3 * A.R + 8 * c;
  *reinterpret_cast<u4*>(o) = hi;
  *reinterpret_cast<u4*>(o + A.R) = mid;
  *reinterpret_cast<u4*>(o + 2 * A.R) = lo;
}

template <int RC>
__global__ __launch_bounds__(256, 2) void k_rs_message(RsArgs A) {
  constexpr int NS = RC == 64 ? 4 : 2, NR = RC == 64 ? 2 : 1;  // a wave's 16-sender and 16-column blocks
  constexpr int NW = RC / 16, PLANE = 2 * RC * RS_MKS * 2;     // weight chunks a thread copies; bytes of a part
  __shared__ __align__(16) char wt[3 * PLANE];
  __shared__ __align__(16) char et[RS_B * RS_MKS * 2];
  const int mblocks = A.sblocks * (A.R / RC);
  if ((int)blockIdx.x >= mblocks) {
    split_w_last(A, (int64_t)(blockIdx.x - mblocks) * 256 + threadIdx.x);
    return;
  }
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, g = lane >> 4, li = lane & 15;
  const int ws = RC == 64 ? (w & 1) * 64 : w * 32, wr = RC == 64 ? (w >> 1) * 32 : 0;
  const int64_t Ns = (int64_t)A.n * A.K;
  const int64_t i0 = (int64_t)(blockIdx.x % A.sblocks) * RS_B;
  const int r0 = (int)(blockIdx.x / A.sblocks) * RC;
  // this thread copies chunk tid % 8 of tile rows tid / 8 + 32 c (senders; pg, then pv rows)
  const int crow = tid >> 3, kc = tid & 7;
  // (a row past the last sender repeats it: its column of D is dropped)
  int64_t sid[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int64_t i = i0 + crow + 32 * c;
    sid[c] = sender_of(A, i < Ns ? i : Ns - 1);
  }
  f4 acc[2][NR][NS];  // [gate, value][16 columns][16 senders]
#pragma unroll
  for (int i = 0; i < 2 * NR * NS; ++i) acc[i / (NR * NS)][i / NS % NR][i % NS] = f4{0.f, 0.f, 0.f, 0.f};

  // one product over `depth` (a multiple of 16): rows of `src` (bf16) times gate / value weight rows
  auto product = [&](const uint16_t* src, const float* wg, const float* wv, int depth) {
    u4 pe[4];
    f4 pw[NW][2];
    auto fetch = [&](int k0) {
      // (chunks past the depth repeat the stage's first two against zero weights)
      const bool in = k0 + 8 * kc < depth;
      const int k = in ? k0 + 8 * kc : k0 + 8 * (kc & 1);
#pragma unroll
      for (int c = 0; c < 4; ++c) pe[c] = *reinterpret_cast<const u4u*>(src + sid[c] * depth + k);
#pragma unroll
      for (int c = 0; c < NW; ++c) {
        const int row = crow + 32 * c;  // (of gate rows, then value rows)
        const float* m = row >= RC || !wg ? wv : wg;
        const float* p = m + (int64_t)(r0 + row % RC) * depth + k;
        pw[c][0] = *reinterpret_cast<const f4u*>(p);
        pw[c][1] = *reinterpret_cast<const f4u*>(p + 4);
      }
    };
    fetch(0);
    for (int k0 = 0; k0 < depth; k0 += RS_MKS) {
      __syncthreads();  // (the previous stage's readers are done)
#pragma unroll
      for (int c = 0; c < 4; ++c) put16(et + tile_at64(crow + 32 * c, kc), pe[c]);
#pragma unroll
      for (int c = 0; c < NW; ++c) {
        u4 hi, mid, lo;
        split8(pw[c][0], pw[c][1], hi, mid, lo);
        if (k0 + 8 * kc >= depth) hi = mid = lo = u4{0, 0, 0, 0};
        char* at = wt + tile_at64(crow + 32 * c, kc);
        put16(at, hi);
        put16(at + PLANE, mid);
        put16(at + 2 * PLANE, lo);
      }
      __syncthreads();
      if (k0 + RS_MKS < depth) fetch(k0 + RS_MKS);  // in flight under this stage's products
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        u4 e[NS];
#pragma unroll
        for (int sb = 0; sb < NS; ++sb) e[sb] = lds16(et + tile_at64(ws + 16 * sb + li, 4 * ks + g));
#pragma unroll
        for (int m = 0; m < 2; ++m) {
          if (m == 0 && !wg) continue;
#pragma unroll
          for (int rb = 0; rb < NR; ++rb) {
            const char* wp = wt + tile_at64(RC * m + wr + 16 * rb + li, 4 * ks + g);
            const u4 hi = lds16(wp), mid = lds16(wp + PLANE), lo = lds16(wp + 2 * PLANE);
#pragma unroll
            for (int sb = 0; sb < NS; ++sb) acc[m][rb][sb] = mfma(lo, e[sb], acc[m][rb][sb]);
#pragma unroll
            for (int sb = 0; sb < NS; ++sb) acc[m][rb][sb] = mfma(mid, e[sb], acc[m][rb][sb]);
#pragma unroll
            for (int sb = 0; sb < NS; ++sb) acc[m][rb][sb] = mfma(hi, e[sb], acc[m][rb][sb]);
          }
        }
      }
    }
  };
  product(A.codebook, A.pg, A.pv, A.C);
#pragma unroll
  for (int i = 0; i < 2 * NR * NS; ++i) acc[i / (NR * NS)][i / NS % NR][i % NS] *= A.sqrt_c;
  if (A.res_emb) product(A.res_emb, nullptr, A.res_proj, A.RR);  // value += res_emb[sender] @ res_proj^T

#pragma unroll
  for (int sb = 0; sb < NS; ++sb) {
    const int64_t io = i0 + ws + 16 * sb + li;
    if (io >= Ns) continue;
    const uint16_t* qrow = A.query + state_row(A, io / A.K) * A.query_stride;
#pragma unroll
    for (int rb = 0; rb < NR; ++rb) {
      const int r = r0 + wr + 16 * rb + 4 * g;
      float msg[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float pre = (bf(qrow[r + v]) + acc[0][rb][sb][v]) + A.gb[r + v];
        msg[v] = 1.f / (1.f + expf(-pre)) * acc[1][rb][sb][v];
      }
      uint2 part[3];
      split2(msg[0], msg[1], part[0].x, part[1].x, part[2].x);
      split2(msg[2], msg[3], part[0].y, part[1].y, part[2].y);
#pragma unroll
      for (int q = 0; q < 3; ++q) *reinterpret_cast<uint2*>(A.msg + (io * 3 + q) * A.R + r) = part[q];
    }
  }
}

// ---------------------------------------------------------------------------------------
// k_rs_table: eight units (a row's 16 senders each) a workgroup, one H slice a grid column.  Wave
// (w & 1, w >> 1) has 4 units and 64 h of a TH-h tile (256 or 64: rs_plan); D[4g + v][li] is h 4g + v of
// sender li, which two 16-h blocks at a time is the B operand of the product with the head rows.
// A stage (32 k of the tile's w_last and message parts, 72 KB) goes from memory straight to LDS, the
// next one into the other buffer while this one is multiplied: 333 us at the sizes above at the least,
// 372 in the median under the profiler.  128-h tiles of four waves with the parts of w_last made while
// staging through registers (two workgroups a CU) took 446 (this then 320 at the least): the splitting, 13 spilled registers, and 1.4 times the operand traffic.
// ---------------------------------------------------------------------------------------
template <int KB, int TH>
__global__ __launch_bounds__(2 * TH, TH == 256 && KB <= 2 ? 2 : 1) void k_rs_table(RsArgs A) {
  constexpr int NWAVE = TH / 32;           // waves: two of 64 senders each for every 64 h
  constexpr int WPLANE = TH * RS_KS * 2;   // bytes of one part of a stage's w_last rows
  constexpr int STAGE = 3 * (WPLANE + RS_PLANE);
  __shared__ __align__(16) char buf0[STAGE];
  __shared__ __align__(16) char buf1[STAGE];
  __shared__ const uint16_t* hrows[8 * KB * 16];
  __shared__ const uint16_t* xrows[8];
  __shared__ float scales[8];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4, li = lane & 15;
  const int ws = (w & 1) * 64, wh = (w >> 1) * 64;
  const int unit0 = blockIdx.x * (RS_B / 16);
  const int slice = blockIdx.y;
  const int h_lo = slice * A.hs, h_hi = h_lo + A.hs < A.H ? h_lo + A.hs : A.H;
  // copies: 16 rows of 64 bytes a wave at a time, w_last's parts (rows 16 (w + NWAVE c)) and then the
  // messages'; LDS chunk (row, slot) holds the row's chunk slot ^ (row / 2 % 4) -- see tile_at
  constexpr int NC = TH / 16 / NWAVE, NM = RS_B / 16 / NWAVE;  // row blocks of each a wave copies
  const int cch = 8 * ((lane ^ (lane >> 3)) & 3);
  const uint16_t* msrc[NM];
#pragma unroll
  for (int c = 0; c < NM; ++c) {
    const int u = unit0 + w + NWAVE * c, unit = u < A.units ? u : A.units - 1, j = (unit % KB) * 16 + (lane >> 2);
    msrc[c] = A.msg + ((int64_t)(unit / KB) * A.K + (j < A.K ? j : A.K - 1)) * 3 * A.R + cch;
  }
  auto fetch = [&](char* buf, int h0, int k0) {
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int row = 16 * (w + NWAVE * c), h = h0 + row + (lane >> 2);
      const uint16_t* src = A.wsplit + (int64_t)(h < h_hi ? h : h_hi - 1) * 3 * A.R + cch + k0;
#pragma unroll
      for (int q = 0; q < 3; ++q) to_lds(src + q * A.R, buf + q * WPLANE + row * 64);
    }
#pragma unroll
    for (int c = 0; c < NM; ++c)
#pragma unroll
      for (int q = 0; q < 3; ++q)
        to_lds(msrc[c] + q * A.R + k0, buf + 3 * WPLANE + q * RS_PLANE + 16 * (w + NWAVE * c) * 64);
  };
  fetch(buf0, h_lo, 0);
  // where each unit's state row and each sender column's head rows are (a unit past the last, and a
  // lane past K, repeats one: what it computes is dropped)
  for (int q = tid; q < 8 * KB * 16; q += 64 * NWAVE) {
    const int unit = unit0 + q / (KB * 16) < A.units ? unit0 + q / (KB * 16) : A.units - 1, c = q % (KB * 16);
    const int64_t at = (int64_t)(unit / KB) * A.K + (c < A.K ? c : A.K - 1);
    hrows[q] = A.head + (A.head_is_cand ? at : A.cand[at]) * A.H;
  }
  if (tid < 8) {
    const int unit = unit0 + tid < A.units ? unit0 + tid : A.units - 1;
    const int64_t mrow = state_row(A, unit / KB);
    xrows[tid] = A.raw + mrow * A.raw_stride;
    scales[tid] = A.rms[mrow];
  }
  f4 dot[4][KB];
  float ss[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    ss[u] = 0.f;
#pragma unroll
    for (int cb = 0; cb < KB; ++cb) dot[u][cb] = f4{0.f, 0.f, 0.f, 0.f};
  }
  f4 acc[4][4];  // [16 h][unit]
  const int wb = tile_at(wh + li, g), mb = 3 * WPLANE + tile_at(ws + li, g);  // (16 rows on: 1024 bytes)
  auto multiply = [&](const char* buf) {
    u4 b[4][3];
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int q = 0; q < 3; ++q) b[u][q] = lds16(buf + mb + q * RS_PLANE + 1024 * u);
#pragma unroll
    for (int hb = 0; hb < 4; ++hb) {
      const char* wp = buf + wb + 1024 * hb;
      const u4 hi = lds16(wp), mid = lds16(wp + WPLANE), lo = lds16(wp + 2 * WPLANE);
      // the products down to 2^-18 of the first, smallest first (what is left out is under 2^-25)
#pragma unroll
      for (int u = 0; u < 4; ++u) acc[hb][u] = mfma(lo, b[u][0], acc[hb][u]);
#pragma unroll
      for (int u = 0; u < 4; ++u) acc[hb][u] = mfma(hi, b[u][2], acc[hb][u]);
#pragma unroll
      for (int u = 0; u < 4; ++u) acc[hb][u] = mfma(mid, b[u][1], acc[hb][u]);
#pragma unroll
      for (int u = 0; u < 4; ++u) acc[hb][u] = mfma(mid, b[u][0], acc[hb][u]);
#pragma unroll
      for (int u = 0; u < 4; ++u) acc[hb][u] = mfma(hi, b[u][1], acc[hb][u]);
#pragma unroll
      for (int u = 0; u < 4; ++u) acc[hb][u] = mfma(hi, b[u][0], acc[hb][u]);
    }
  };
  for (int h0 = h_lo; h0 < h_hi; h0 += TH) {
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i >> 2][i & 3] = f4{0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < A.R; k0 += 2 * RS_KS) {  // (R is a multiple of 64)
      // (the copies are issued before the products: the compiler may not move them down)
      stage_wait();
      fetch(buf1, h0, k0 + RS_KS);
      __builtin_amdgcn_sched_barrier(0);
      multiply(buf0);
      stage_wait();
      const bool last = k0 + 2 * RS_KS >= A.R;
      const int nh = last ? h0 + TH : h0;
      if (nh < h_hi) fetch(buf0, nh, last ? 0 : k0 + 2 * RS_KS);
      __builtin_amdgcn_sched_barrier(0);
      multiply(buf1);
    }
    // ref, its square, and (ref * norm_w) . head.  A 16-h block past the slice repeats its last one
    // (H is a multiple of 16) with ref 0; its operands are loaded four units at a time, before use
    const bool whole = h0 + wh + 64 <= h_hi;
    int hx[4];
    f4 nw[4];
#pragma unroll
    for (int hb = 0; hb < 4; ++hb) {
      const int h = h0 + wh + 16 * hb;
      hx[hb] = (h < h_hi ? h : h_hi - 16) + 4 * g;
      nw[hb] = *reinterpret_cast<const f4u*>(A.norm_w + hx[hb]);
    }
    uint2 xb[4][4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const uint16_t* xrow = xrows[(ws >> 4) + u];
#pragma unroll
      for (int hb = 0; hb < 4; ++hb) xb[u][hb] = *reinterpret_cast<const uint2*>(xrow + hx[hb]);
    }
#pragma unroll
    for (int cb = 0; cb < KB; ++cb) {
      uint2 hd[4][4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const uint16_t* hrow = hrows[((ws >> 4) + u) * KB * 16 + cb * 16 + li];
#pragma unroll
        for (int hb = 0; hb < 4; ++hb) hd[u][hb] = *reinterpret_cast<const uint2*>(hrow + hx[hb]);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (cb == 0) {
          const float scale = scales[(ws >> 4) + u];
#pragma unroll
          for (int hb = 0; hb < 4; ++hb) {
            const bool in = whole || h0 + wh + 16 * hb < h_hi;
            const f4 xv = {__uint_as_float(xb[u][hb].x << 16), __uint_as_float(xb[u][hb].x & 0xFFFF0000u),
                           __uint_as_float(xb[u][hb].y << 16), __uint_as_float(xb[u][hb].y & 0xFFFF0000u)};
#pragma unroll
            for (int v = 0; v < 4; ++v) {
              const float ref = in ? xv[v] + scale * acc[hb][u][v] : 0.f;
              ss[u] += ref * ref;
              acc[hb][u][v] = ref * nw[hb][v];
            }
          }
        }
#pragma unroll
        for (int hp = 0; hp < 4; hp += 2) {
          u4 hi, mid, lo;
          split8(acc[hp][u], acc[hp + 1][u], hi, mid, lo);
          const u4 a = {hd[u][hp].x, hd[u][hp].y, hd[u][hp + 1].x, hd[u][hp + 1].y};
          dot[u][cb] = mfma(a, lo, dot[u][cb]);
          dot[u][cb] = mfma(a, mid, dot[u][cb]);
          dot[u][cb] = mfma(a, hi, dot[u][cb]);
        }
      }
    }
  }
  // the wave's partial sums: ss over the lane groups' h (lanes li, li+16, li+32, li+48 share a sender),
  // dot[u][cb][v] = sum_h head[c = cb*16 + 4g + v][h] * ref[j][h] * norm_w[h]
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int unit = unit0 + (ws >> 4) + u;
    if (unit >= A.units) continue;
    float s = ss[u];
    s += __shfl_xor(s, 16);
    s += __shfl_xor(s, 32);
    float* pp = A.part + ((int64_t)(slice * (TH / 64) + (w >> 1)) * A.units + unit) * (16 + 16 * KB * 16);
    if (g == 0) pp[li] = s;
#pragma unroll
    for (int cb = 0; cb < KB; ++cb)
#pragma unroll
      for (int v = 0; v < 4; ++v) pp[16 + (cb * 16 + 4 * g + v) * 16 + li] = dot[u][cb][v];
  }
}

// out[n, j, c] = (sum over slices of the dot products) / sqrt(sum of ref^2 / H + eps)
__global__ void k_rs_finish(RsArgs A) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;  // n * K * K + j * K + c
  const int64_t total = (int64_t)A.n * A.K * A.K;
  if (e >= total) return;
  const int64_t n = e / ((int64_t)A.K * A.K);
  const int j = (int)(e / A.K % A.K), c = (int)(e % A.K);
  const int unit = (int)n * A.KB + j / 16, jl = j % 16;
  const int stride = 16 + 16 * A.KB * 16;
  float ss = 0.f, d = 0.f;
  const float* pp = A.part + (int64_t)unit * stride;
  const int64_t step = (int64_t)A.units * stride;
  for (int s = 0; s < A.parts; s += 8) {  // eight parts' loads in flight (one by one: 24 us for 64 parts)
    float a[8], b[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const float* p = pp + (s + q < A.parts ? s + q : A.parts - 1) * step;
      a[q] = p[jl];
      b[q] = p[16 + c * 16 + jl];
    }
#pragma unroll
    for (int q = 0; q < 8; ++q)
      if (s + q < A.parts) ss += a[q], d += b[q];
  }
  A.out[e] = d / sqrtf(ss / (float)A.H + A.eps);
}

}  // namespace dsv

using namespace dsv;

// The table's tile and H slices.  256-h tiles of eight waves (one workgroup a CU) from where they keep more
// than half of the card busy; below that 64-h tiles of two waves, two workgroups a CU, which spread a small
// batch over more of it.  The call at 16 lanes, narrow against wide in us, by wide tiles: H 4096, R 512 64
// tiles (30 rows) 58, 70; 128: 68, 72; 192: 87, 79; 240: 90, 84; 480: 156, 132.  H 2048, R 256 120: 42, 46;
// 136: 54, 48.  H 1024 120: 42, 46; 136: 55, 51.  32 lanes 128: 67, 75; 240: 96, 88.  64 lanes 240: 111, 112.
struct RsPlan {
  int tile, slices, hs;
};
static RsPlan rs_plan(int64_t units, int32_t H) {
  const int64_t blocks = (units + RS_B / 16 - 1) / (RS_B / 16);
  RsPlan p;
  p.tile = blocks * ((H + 255) / 256) > 128 ? 256 : 64;
  const int64_t slots = p.tile == 256 ? 256 : 512, tiles = (H + p.tile - 1) / p.tile;
  const int64_t want = blocks >= slots ? 1 : slots / blocks;
  p.slices = (int)(want < tiles ? want : tiles);
  p.hs = (int)((tiles + p.slices - 1) / p.slices) * p.tile;
  p.slices = (H + p.hs - 1) / p.hs;  // (none of them empty)
  return p;
}
static int64_t rs_round(int64_t bytes) { return (bytes + 255) / 256 * 256; }

// (a bound that grows with n: a workspace sized for n serves every smaller n.  A unit leaves a partial
// sum for every 64 h of a slice's tile: units * parts is at most units * H / 64, and at most 8 * 256 * 4
// while there is more than one slice)
extern "C" int64_t dsv_rs_table_workspace_bytes(int64_t n, int32_t K, int32_t H, int32_t R) {
  const int64_t KB = (K + 15) / 16, units = n * KB, tiles = (H + 255) / 256;
  int64_t us = units * tiles < 2048 ? units * tiles : 2048;
  if (us < units) us = units;
  return rs_round(n * K * R * 6) + rs_round((int64_t)H * R * 6) + 4 * us * (16 + 16 * KB * 16) * 4 + 256;
}

extern "C" int dsv_rs_table(const void* raw, int64_t raw_stride, const float* rms, const void* query,
                            int64_t query_stride, const int64_t* anchors, const int64_t* cand, int64_t n, int32_t K,
                            int32_t T, const void* codebook, int32_t C, const float* pred_gate_w, const float* prev_w,
                            const float* gate_b, const float* write_w, int32_t H, int32_t R, const float* norm_w,
                            const void* head, int32_t head_is_candidates, const void* res_emb, const float* res_proj,
                            int32_t RR, float eps, float* out, void* workspace, int64_t workspace_bytes,
                            dsv_stream_t stream_) {
  hipStream_t stream = reinterpret_cast<hipStream_t>(stream_);
  if (n < 0 || K < 1 || K > 64 || T < 2 || n % (T - 1))
    DSV_FAIL(DSV_ERR_INVALID, "dsv_rs_table: layout mismatch (n %lld, K %d, T %d)", (long long)n, K, T);
  if (n == 0) return DSV_OK;
  if (!raw || !rms || !query || !anchors || !cand || !codebook || !pred_gate_w || !prev_w || !gate_b || !write_w ||
      !norm_w || !head || !out || !workspace || (res_emb && !res_proj))
    DSV_FAIL(DSV_ERR_INVALID, "dsv_rs_table: required pointer is null");
  if (C < 16 || C % 16 || H < 16 || H % 16 || R < 64 || R % 64 || R > RS_RMAX || (res_emb && (RR < 16 || RR % 16)))
    DSV_FAIL(DSV_ERR_UNSUPPORTED,
             "dsv_rs_table: needs C, H (and the residual width) multiples of 16 and R a multiple of 64 up to %d "
             "(C %d, H %d, R %d)", RS_RMAX, C, H, R);
  if (raw_stride < H || query_stride < R || (uintptr_t)raw % 8 || (uintptr_t)query % 8 || (uintptr_t)codebook % 8 ||
      (uintptr_t)head % 8 || raw_stride % 4 || (res_emb && (uintptr_t)res_emb % 8))
    DSV_FAIL(DSV_ERR_INVALID, "dsv_rs_table: bf16 operands need 8-byte aligned rows");
  if (workspace_bytes < dsv_rs_table_workspace_bytes(n, K, H, R))
    DSV_FAIL(DSV_ERR_WORKSPACE, "dsv_rs_table: workspace too small");
  RsArgs A;
  memset(&A, 0, sizeof(A));
  A.raw = reinterpret_cast<const uint16_t*>(raw);
  A.rms = rms;
  A.query = reinterpret_cast<const uint16_t*>(query);
  A.anchors = anchors;
  A.cand = cand;
  A.codebook = reinterpret_cast<const uint16_t*>(codebook);
  A.pg = pred_gate_w;
  A.pv = prev_w;
  A.gb = gate_b;
  A.w_last = write_w;
  A.norm_w = norm_w;
  A.head = reinterpret_cast<const uint16_t*>(head);
  A.res_emb = reinterpret_cast<const uint16_t*>(res_emb);
  A.res_proj = res_proj;
  A.raw_stride = raw_stride;
  A.query_stride = query_stride;
  A.T = T;
  A.K = K;
  A.H = H;
  A.R = R;
  A.C = C;
  A.RR = res_emb ? RR : 0;
  A.n = (int32_t)n;
  A.head_is_cand = head_is_candidates ? 1 : 0;
  A.eps = eps;
  A.sqrt_c = (float)sqrt((double)C);
  A.KB = (K + 15) / 16;
  A.units = (int32_t)n * A.KB;
  const RsPlan plan = rs_plan(A.units, H);
  A.hs = plan.hs;
  A.parts = plan.slices * (plan.tile / 64);
  char* ws = reinterpret_cast<char*>(rs_round((int64_t)workspace));  // (16-byte copies; the size has 256 spare)
  A.msg = reinterpret_cast<uint16_t*>(ws);
  A.wsplit = reinterpret_cast<uint16_t*>(ws + rs_round(n * K * R * 6));
  A.part = reinterpret_cast<float*>(ws + rs_round(n * K * R * 6) + rs_round((int64_t)H * R * 6));
  A.out = out;
  // 64 message columns a workgroup where that fills the card, 16 below (15 rows: 21 us against 44)
  A.sblocks = (int32_t)((n * K + RS_B - 1) / RS_B);
  const int rc = A.sblocks * (R / 64) >= 256 ? 64 : 16;
  const dim3 mg((unsigned)(A.sblocks * (R / rc) + ((int64_t)H * R / 8 + 255) / 256));
  if (rc == 64) hipLaunchKernelGGL(k_rs_message<64>, mg, dim3(256), 0, stream, A);
  else hipLaunchKernelGGL(k_rs_message<16>, mg, dim3(256), 0, stream, A);
  DSV_CHECK_LAUNCH("k_rs_message");
  const dim3 tg((unsigned)((A.units + RS_B / 16 - 1) / (RS_B / 16)), (unsigned)plan.slices);
  auto table = [&](auto wide, auto narrow) {
    if (plan.tile == 256) hipLaunchKernelGGL(wide, tg, dim3(512), 0, stream, A);
    else hipLaunchKernelGGL(narrow, tg, dim3(128), 0, stream, A);
  };
  switch (A.KB) {
    case 1: table(k_rs_table<1, 256>, k_rs_table<1, 64>); break;
    case 2: table(k_rs_table<2, 256>, k_rs_table<2, 64>); break;
    case 3: table(k_rs_table<3, 256>, k_rs_table<3, 64>); break;
    default: table(k_rs_table<4, 256>, k_rs_table<4, 64>); break;
  }
  DSV_CHECK_LAUNCH("k_rs_table");
  const int64_t total = n * K * K;
  hipLaunchKernelGGL(k_rs_finish, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, stream, A);
  DSV_CHECK_LAUNCH("k_rs_finish");
  return DSV_OK;
}
