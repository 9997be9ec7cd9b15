// Modulation projection: mods[r][n] = sum_k silu(c[r][k]) W[n][k] + bias[n] for the rows r = (sample, Euler
// step) of one expert call — every AdaRMS scale, shift and gate of every layer and step in one product
// (MODW = 9 L H + 2 H columns; the reference's kernel reads these rows, src/mk_expert.py:336-340, and
// REKI's _step_modulations makes them, mk_expert.py:529).
//
// HBM-bound on W (bf16 [MODW, H]: 108.5 MB for L10 H768), so each weight byte is read once and the weights are
// what streams: a workgroup keeps silu(c) of up to five 16-row tiles on the chip for the whole launch (each of its 8
// waves an eighth of K, split into three bf16 parts, an MFMA per part and fragment) and walks a contiguous range of
// 16-column tiles, every wave loading its own K / 8 of a tile's weights a few tiles ahead. The arithmetic of a row, and
// the order of its sums, are the same whatever the number of rows: its bits do not depend on its company.
#pragma once

#include "mkx.h"
#include "mkx_device.h"

namespace mkx {

constexpr int MODP_WAVES = 8;     // waves of a projection workgroup, each over 1 / 8 of K
constexpr int MODP_GRID = 256;    // workgroups at once: one per CU of an MI355X (two with one row tile)
constexpr int MODP_XCDS = 8;      // XCDs the dispatcher deals consecutive workgroups to
constexpr int MODP_PARTS = 3;     // bf16 parts of silu(c): as exact as fp32, and the same for every number of rows

typedef float modp_f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 modp_bf16x2 __attribute__((ext_vector_type(2)));

// two floats rounded to nearest-even bf16 by the packed hardware conversion, low element in the low half
__device__ __forceinline__ uint32_t modp_cvt2(float x, float y) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((modp_f32x2){x, y}, modp_bf16x2));
}

// a pair of fp32 values as NS packed bf16 parts, each the rounded rest of the ones before (NS = 2: exact to about
// 2^-17 relative, NS = 3: as exact as fp32)
template <int NS>
__device__ __forceinline__ void modp_split2(float x, float y, uint32_t (&p)[NS]) {
#pragma unroll
  for (int i = 0; i < NS; ++i) {
    p[i] = modp_cvt2(x, y);
    x -= __uint_as_float(p[i] << 16);
    y -= __uint_as_float(p[i] & 0xffff0000u);
  }
}
// silu of 8 values (hardware exp and reciprocal) as NS bf16 fragments
template <int NS>
__device__ __forceinline__ void modp_silu_split(f32x4 x0, f32x4 x1, bf16x8 (&f)[NS]) {
  const float g[8] = {x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
  u32x4 o[NS];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float v0 = g[2 * e] * __builtin_amdgcn_rcpf(1.f + __expf(-g[2 * e]));
    const float v1 = g[2 * e + 1] * __builtin_amdgcn_rcpf(1.f + __expf(-g[2 * e + 1]));
    uint32_t p[NS];
    modp_split2<NS>(v0, v1, p);
#pragma unroll
    for (int i = 0; i < NS; ++i) o[i][e] = p[i];
  }
#pragma unroll
  for (int i = 0; i < NS; ++i) f[i] = __builtin_bit_cast(bf16x8, o[i]);
}

// column tiles of weights a wave has in flight ahead of the one it multiplies, KW KB each. With one row tile two
// workgroups share a CU, and more in flight is better while 128 registers hold it; with more rows the time goes to the
// products as well, and two tiles ahead are enough (K 768, 40 rows 25.1 us with four ahead, 23.3 with two; 80 rows 33.9
// with three, 31.3 with two, 33.5 with one).
template <int KT, int NRT>
constexpr int modp_ahead() { return NRT > 1 ? 2 : KT <= 8 ? 8 : KT <= 24 ? 4 : 3; }

// row tiles of 16 that a workgroup holds at most, and the number of them whose third part lies in LDS: what the registers
// do not hold of the KW * 3 KB per row tile and wave (K 768, 80 rows: 32.3 us with none in LDS, 31.4 with one tile)
template <int KT>
constexpr int modp_max_nrt() { return KT <= 24 ? 5 : 4; }
template <int KT, int NRT>
constexpr int modp_lds_tiles() { return KT * NRT > 120 ? 2 : KT * NRT > 100 ? 1 : 0; }

// grid: x = MODP_XCDS ranges of 16-column tiles x the groups of NRT row tiles, y = the further ranges; the workgroups of
// one range lie MODP_XCDS apart, so that one XCD runs them side by side and the weights come from beyond its L2 once. Wave w
// holds k-blocks [KW w, KW (w + 1)), KW = KT / 8, of silu(c) of every row of the group (NRT KW fragments in three parts)
// and multiplies them with its KW weight fragments of one column tile after the other; the 8 waves' partial tiles
// are summed in wave order through one of two LDS buffers (one barrier per column tile: a buffer is written
// again two tiles later, after the barrier that follows its readers), and wave r stores row tile r.
// Measured (L10 H768, 70656 columns): 10 rows 21.3 -> 19.1 us (5.8 TB/s of weights and results; a large copy reaches 5.1), 80
// rows 59.4 -> 31.3 us (4.2 TB/s), 160 rows 104 -> 51 us, against one workgroup per 64 columns that held the weights and
// staged silu(c) of every row tile anew, in two parts (error against 64 bits 2.5e-6; three parts: 9e-8). With the third part
// only where the registers hold it 80 rows take 29.5 us, and a row's bits depend on how many rows there are.
template <int KT, int NRT>
__global__ __launch_bounds__(64 * MODP_WAVES, NRT == 1 ? 4 : 2) void modproj_kernel(mkx_modproj_args a) {
  constexpr int KW = KT / MODP_WAVES, PF = modp_ahead<KT, NRT>(), NS = MODP_PARTS;
  static_assert(KT % MODP_WAVES == 0 && NRT <= MODP_WAVES, "K splits over the waves; one wave stores a row tile");
  constexpr int NL = modp_lds_tiles<KT, NRT>(), N3 = NRT - NL;  // row tiles from N3 on: third part in LDS
  __shared__ f32x4 part[2][MODP_WAVES][NRT][64];
  __shared__ bf16x8 xl[NL ? MODP_WAVES : 1][NL ? NL : 1][KW][64];  // (each wave reads what it wrote)
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int K = a.K, r0 = (int)(blockIdx.x / MODP_XCDS) * (16 * NRT), nct = a.N / 16;
  const int nr = gridDim.y * MODP_XCDS, range = blockIdx.y * MODP_XCDS + blockIdx.x % MODP_XCDS;
  const int ct0 = (int)((int64_t)nct * range / nr), ct1 = (int)((int64_t)nct * (range + 1) / nr);
  // weight fragments of column tile ct: row 16 ct + (lane & 15), k = 32 t + 8 (lane >> 4) (fragment order: one
  // contiguous KW KB block per wave and tile; row-major: 16 rows x 64 KW B)
  const bool fo = a.w_fragment_order != 0;
  const bf16_t* wp = (const bf16_t*)a.w + (fo ? ((int64_t)wave * KW * 64 + lane) * 8
                                              : (int64_t)(lane & 15) * K + 32 * KW * wave + 8 * (lane >> 4));
  const int wstep = fo ? 64 * 8 : 32;
  // (the bias, wave 0's starting sum, travels with the weights: loads return in order, so one issued at its use
  // would wait for all of the tiles ahead)
  const float* bp = a.bias + 4 * (lane >> 4);
  u32x4 wf[PF][KW];
  f32x4 bias[PF];
  auto load = [&](int slot, int ct) {
    const int c = min(ct, ct1 - 1);  // past the range: its last tile again, unused
    const bf16_t* q = wp + (int64_t)c * 16 * K;
#pragma unroll
    for (int t = 0; t < KW; ++t) wf[slot][t] = ld16(q + t * wstep);
    bias[slot] = *reinterpret_cast<const f32x4*>(bp + c * 16);
  };
  if (ct0 < ct1) {
#pragma unroll
    for (int s = 0; s < PF; ++s) load(s, ct0 + s);
  }
  bf16x8 x[NRT][KW][2], x3[N3][KW];
#pragma unroll
  for (int r = 0; r < NRT; ++r) {
    const int row = min(r0 + 16 * r + (lane & 15), a.R - 1);  // rows past R repeat a valid row, never stored
    const float* cp = a.c + (int64_t)row * a.c_stride + 32 * KW * wave + 8 * (lane >> 4);
#pragma unroll
    for (int t = 0; t < KW; ++t) {
      bf16x8 f[NS];
      modp_silu_split<NS>(*reinterpret_cast<const f32x4*>(cp + 32 * t), *reinterpret_cast<const f32x4*>(cp + 32 * t + 4), f);
      x[r][t][0] = f[0];
      x[r][t][1] = f[1];
      if (r < N3) x3[r < N3 ? r : 0][t] = f[2];
      else xl[wave][r - N3][t][lane] = f[2];
    }
  }
  const int row = r0 + 16 * wave + (lane & 15);  // the row this lane stores (waves below NRT)
  const bool stores = wave < NRT && row < a.R;
  float* op = a.out + (int64_t)(stores ? row : 0) * a.out_stride + 4 * (lane >> 4);
  auto tile = [&](int s, int ct) {
    f32x4 acc[NRT];
#pragma unroll
    for (int r = 0; r < NRT; ++r) acc[r] = wave == 0 ? bias[s] : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = NS - 1; i >= 0; --i)  // the small parts first
#pragma unroll
      for (int t = 0; t < KW; ++t)
#pragma unroll
        for (int r = 0; r < NRT; ++r)
          acc[r] = mfma16(__builtin_bit_cast(bf16x8, wf[s][t]),
                          i < 2 ? x[r][t][i & 1] : r < N3 ? x3[r < N3 ? r : 0][t] : xl[wave][r - N3][t][lane], acc[r]);
    load(s, ct + PF);
    const int buf = (ct - ct0) & 1;
#pragma unroll
    for (int r = 0; r < NRT; ++r) part[buf][wave][r][lane] = acc[r];
    __syncthreads();
    if (stores) {
      f32x4 o = part[buf][0][wave][lane];
#pragma unroll
      for (int w = 1; w < MODP_WAVES; ++w) o += part[buf][w][wave][lane];
      *reinterpret_cast<f32x4*>(op + ct * 16) = o;
    }
  };
  int ct = ct0;
  for (; ct + PF <= ct1; ct += PF) {
#pragma unroll
    for (int s = 0; s < PF; ++s) tile(s, ct + s);
  }
#pragma unroll
  for (int s = 0; s < PF - 1; ++s)
    if (ct + s < ct1) tile(s, ct + s);
}

}  // namespace mkx

namespace mkx {

// The input of the modulation projection for an N-step Euler schedule (t_k = 1 - k / N):
// c[b][k] = silu(temb(t_k) W1^T + b1) W2^T + b2 + state_cond[b], temb(t) = [cos(1000 t f_i) | sin(1000 t f_i)]
// with f_i = 10000^(-i / (tdim / 2)) (the small MLP ahead of the projection in REKI's _step_modulations,
// mk_expert.py:529, as the synthetic expert defines it). One workgroup per 64 output columns of c and 16 steps, 16
// waves: each workgroup computes the whole hidden layer h1 = silu(temb W1^T + b1) for its steps on MFMAs
// (the embedding and h1 staged in LDS as fragments of three bf16 parts, weights bf16, fp32 accumulation), then its
// 64 columns of c for every sample. The embedding's arguments and cos / sin are computed in fp64 and rounded to fp32, as
// the fp32 eager expert computes them.
// Bound by the reads of W1: every workgroup needs it whole, no L2 holds it after the projection of the call before, and
// one CU draws about 12 bytes per cycle from beyond its L2 (393 KB: 14 us). A wave's first weights are loaded before
// the embedding, its part of W2 before the hidden layer's activation and each k-block's weights of the hidden layer
// while the ones before are multiplied. Measured (H 768, 10 steps): 45.6 -> 20.3 us against 4 waves per workgroup,
// the library's sincos for each of cosine and sine, and one k-block's loads at a time.
constexpr int MODIN_BLOCK = 1024;
constexpr int MODIN_WAVES = MODIN_BLOCK / 64;
constexpr int MODIN_KS = MODIN_WAVES / 4;  // waves sharing one 16-column tile of c, each over 1 / 4 of K
constexpr int MODIN_MAX_TKB = 16;  // tdim <= 512
constexpr int MODIN_CK = 2;        // k-blocks of W1 loaded together
constexpr int MODIN_NS = 3;        // bf16 parts of the embedding and of h1: as exact as fp32
// dynamic LDS: the fragments of temb (later the K parts of c) and of h1
__host__ __device__ constexpr int modin_es_bytes(int tdim) {
  return tdim / 32 * MODIN_NS * 1024 > MODIN_WAVES * 1024 ? tdim / 32 * MODIN_NS * 1024 : MODIN_WAVES * 1024;
}
__host__ __device__ constexpr int modin_lds_bytes(int tdim, int H) { return modin_es_bytes(tdim) + H / 32 * MODIN_NS * 1024; }

// Sine and cosine of 0 <= x <= 1000 to about 1e-13 in fp64: x reduced by the nearest multiple of pi / 2 (pi / 2 in
// two parts, so that the difference is exact to that), then both Taylor series on [-pi / 4, pi / 4] and the
// quadrant's swap and signs. The library's sincos, which serves every argument, took most of the kernel's time.
__device__ __forceinline__ void modin_sincos(double x, double& sn, double& cs) {
  const double n = rint(x * 0.63661977236758134308);  // 2 / pi
  const double r = fma(-n, 6.123233995736766036e-17, fma(-n, 1.5707963267948965580, x)), q = r * r;
  double s = -1.0 / 1307674368000.0, c = 1.0 / 20922789888000.0;  // r^15 / 15!, r^16 / 16!
  s = fma(s, q, 1.0 / 6227020800.0);
  s = fma(s, q, -1.0 / 39916800.0);
  s = fma(s, q, 1.0 / 362880.0);
  s = fma(s, q, -1.0 / 5040.0);
  s = fma(s, q, 1.0 / 120.0);
  s = fma(s, q, -1.0 / 6.0);
  s = fma(s * q, r, r);
  c = fma(c, q, -1.0 / 87178291200.0);
  c = fma(c, q, 1.0 / 479001600.0);
  c = fma(c, q, -1.0 / 3628800.0);
  c = fma(c, q, 1.0 / 40320.0);
  c = fma(c, q, -1.0 / 720.0);
  c = fma(c, q, 1.0 / 24.0);
  c = fma(c, q, -0.5);
  c = fma(c, q, 1.0);
  const int k = (int)n & 3;
  sn = (k & 1) ? c : s;
  cs = (k & 1) ? s : c;
  if (k & 2) sn = -sn;
  if (k == 1 || k == 2) cs = -cs;
}

// TPW: hidden tiles per wave, H / 256
template <int TPW>
__global__ __launch_bounds__(MODIN_BLOCK) void modin_kernel(mkx_modin_args a) {
  constexpr int NS = MODIN_NS;
  extern __shared__ __align__(16) char es[];                     // temb, split fragments: [kb][part][64 lanes] x 16 B
  char* const hs = es + modin_es_bytes(a.tdim);                  // h1, split fragments
  f32x4(*part)[4][64] = reinterpret_cast<f32x4(*)[4][64]>(es);  // K parts of c: [MODIN_KS][4][64], after temb
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  constexpr int H = TPW * MODIN_WAVES * 16, KH = H / 32 / MODIN_KS;
  const int TKB = a.tdim / 32, half = a.tdim / 2, k0 = blockIdx.y * 16;
  const int ct = wave & 3, ks = wave >> 2;
  const int n0 = (blockIdx.x * 4 + ct) * 16;  // this wave's 16 columns of c
  // this wave's hidden tiles wave, wave + 16, ...: MODIN_CK k-blocks of each loaded together
  const int nck = (TKB + MODIN_CK - 1) / MODIN_CK;
  // weight rows as MFMA fragments: row n + (lane & 15), k = 32 kb + 8 (lane >> 4)
  const bf16_t* w1 = (const bf16_t*)a.t1_w + (int64_t)(wave * 16 + (lane & 15)) * a.tdim + 8 * (lane >> 4);
  u32x4 wf1[MODIN_CK][TPW];
  auto load1 = [&](int ck) {  // (past the last k-block: that one again, unused)
#pragma unroll
    for (int i = 0; i < MODIN_CK; ++i)
#pragma unroll
      for (int j = 0; j < TPW; ++j)
        wf1[i][j] = ld16(w1 + j * MODIN_WAVES * 16 * a.tdim + 32 * min(ck * MODIN_CK + i, TKB - 1));
  };
  load1(0);
  // temb of steps k0 .. k0 + 15 (the rows of steps past N hold what LDS held: rows are independent, and these are
  // never stored): column fi holds the cosine and half + fi the sine of one angle
  const int nr = min(16, a.N - k0);
  const double lf = log(10000.0) / (double)half;
  for (int it = threadIdx.x; it < nr * half; it += MODIN_BLOCK) {
    const int fi = it / nr, r = it - fi * nr;
    double sn, cs;
    modin_sincos((1.0 - (double)(k0 + r) / (double)a.N) * 1000.0 * exp(-lf * (double)fi), sn, cs);
    uint32_t p[NS];
    modp_split2<NS>((float)cs, (float)sn, p);
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int i = fi + e * half;
      char* q = es + ((i >> 5) * NS * 64 + r + 16 * ((i & 31) >> 3)) * 16 + (i & 7) * 2;
#pragma unroll
      for (int n = 0; n < NS; ++n) *reinterpret_cast<bf16_t*>(q + n * 1024) = (bf16_t)(e ? p[n] >> 16 : p[n]);
    }
  }
  __syncthreads();
  // h1 = silu(temb W1^T + b1), all H columns (D^T = W X^T: lane l holds columns 4 (l / 16) + i of row l % 16; a
  // wave's tiles share the reads of the embedding), into LDS as split fragments: the lane's 4 columns c0 .. c0 + 3 of
  // row l % 16 are elements 4 (j % 2) .. of 8-column group j / 2 of k-block c0 / 32 (fragment lane l % 16 + 16
  // ((c0 % 32) / 8))
  f32x4 hacc[TPW];
#pragma unroll
  for (int j = 0; j < TPW; ++j) hacc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int ck = 0; ck < nck; ++ck) {
    u32x4 w[MODIN_CK][TPW];
#pragma unroll
    for (int i = 0; i < MODIN_CK; ++i)
#pragma unroll
      for (int j = 0; j < TPW; ++j) w[i][j] = wf1[i][j];
    load1(ck + 1);
#pragma unroll
    for (int i = 0; i < MODIN_CK; ++i) {
      const int kb = ck * MODIN_CK + i;
      if (kb >= TKB) break;
      bf16x8 x[NS];
#pragma unroll
      for (int n = 0; n < NS; ++n) x[n] = *reinterpret_cast<const bf16x8*>(es + ((kb * NS + n) * 64 + lane) * 16);
#pragma unroll
      for (int n = NS - 1; n >= 0; --n)  // the small parts first
#pragma unroll
        for (int j = 0; j < TPW; ++j)
          hacc[j] = mfma16(__builtin_bit_cast(bf16x8, w[i][j]), x[n], hacc[j]);
    }
  }
  const bf16_t* w2 = (const bf16_t*)a.t2_w + (int64_t)(n0 + (lane & 15)) * H + 8 * (lane >> 4);
  u32x4 wf2[KH];
#pragma unroll
  for (int i = 0; i < KH; ++i) wf2[i] = ld16(w2 + 32 * (ks * KH + i));
#pragma unroll
  for (int j = 0; j < TPW; ++j) {
    const int c0 = (wave + j * MODIN_WAVES) * 16 + 4 * (lane >> 4);
    const f32x4 b1 = *reinterpret_cast<const f32x4*>(a.t1_b + c0);
    float v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float x = hacc[j][i] + b1[i];
      v[i] = x / (1.f + __expf(-x));
    }
    uint32_t p0[NS], p1[NS];
    modp_split2<NS>(v[0], v[1], p0);
    modp_split2<NS>(v[2], v[3], p1);
    char* q = hs + ((c0 >> 5) * NS * 64 + (lane & 15) + 16 * ((c0 & 31) >> 3)) * 16 + ((c0 >> 2) & 1) * 8;
#pragma unroll
    for (int n = 0; n < NS; ++n) *reinterpret_cast<u32x2*>(q + n * 1024) = u32x2{p0[n], p1[n]};
  }
  __syncthreads();
  // this wave's quarter of K of its 16 columns of c
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < KH; ++i) {
    const char* x = hs + ((ks * KH + i) * NS * 64 + lane) * 16;
#pragma unroll
    for (int n = NS - 1; n >= 0; --n)
      acc = mfma16(__builtin_bit_cast(bf16x8, wf2[i]), *reinterpret_cast<const bf16x8*>(x + n * 1024), acc);
  }
  part[ks][ct][lane] = acc;
  const int k = k0 + (lane & 15), c0 = n0 + 4 * (lane >> 4);
  const f32x4 b2 = *reinterpret_cast<const f32x4*>(a.t2_b + c0);
  __syncthreads();
  f32x4 z = part[0][ct][lane];
#pragma unroll
  for (int j = 1; j < MODIN_KS; ++j) z += part[j][ct][lane];
  z += b2;
  if (k < a.N) {
    for (int b = ks; b < a.B; b += MODIN_KS) {
      const f32x4 sc = *reinterpret_cast<const f32x4*>(a.state_cond + (int64_t)b * a.sc_stride + c0);
      *reinterpret_cast<f32x4*>(a.out + (int64_t)b * a.out_stride_b + (int64_t)k * a.out_stride_k + c0) = z + sc;
    }
  }
}

// The same input in two launches through a workspace of N x H floats (h1), each over H / 16 workgroups: no workgroup
// needs more than 16 rows of a weight matrix (H 768, 10 steps: 5.1 + 4.3 us against the 20.3 us of the single launch,
// which serves callers without a workspace). One workgroup = 16 columns and 16 steps, 8 waves over K, summed through
// LDS in wave order; the fragments are computed in the registers that multiply them.
constexpr int MODIN2_WAVES = 8;

// this wave's K part of a 16 x 16 tile, summed over the waves (every wave returns the sum)
__device__ __forceinline__ f32x4 modin2_sum(f32x4 acc, int wave, int lane) {
  __shared__ f32x4 part[MODIN2_WAVES][64];
  part[wave][lane] = acc;
  __syncthreads();
  f32x4 z = part[0][lane];
#pragma unroll
  for (int w = 1; w < MODIN2_WAVES; ++w) z += part[w][lane];
  return z;
}

// h1[k][n] = silu(temb(t_k) W1^T + b1). K is taken in blocks of 16 cosines and the 16 sines of the same angles: lane
// group g = lane / 16 of block q holds columns 16 q + 8 g + e (g < 2) or half + 16 q + 8 (g - 2) + e of step
// lane % 16, so that every embedding width (a multiple of 32) has whole blocks.
__global__ __launch_bounds__(64 * MODIN2_WAVES) void modin_hidden_kernel(mkx_modin_args a, float* __restrict__ h1) {
  constexpr int NS = MODIN_NS;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4;
  const int half = a.tdim / 2, k = min((int)blockIdx.y * 16 + (lane & 15), a.N - 1), n0 = blockIdx.x * 16;
  const int col = (g < 2 ? 8 * g : half + 8 * (g - 2));
  const bf16_t* w1 = (const bf16_t*)a.t1_w + (int64_t)(n0 + (lane & 15)) * a.tdim + col;
  const double t = (1.0 - (double)k / (double)a.N) * 1000.0, lf = log(10000.0) / (double)half, step = exp(-lf);
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int q = wave; q < a.tdim / 32; q += MODIN2_WAVES) {
    const bf16x8 w = __builtin_bit_cast(bf16x8, ld16(w1 + 16 * q));
    double arg = t * exp(-lf * (double)(16 * q + 8 * (g & 1)));
    u32x4 x[NS];
#pragma unroll 1
    for (int e = 0; e < 4; ++e) {
      float v[2];
#pragma unroll 1
      for (int i = 0; i < 2; ++i) {
        double sn, cs;
        modin_sincos(arg, sn, cs);
        arg *= step;
        const float r = (float)(g < 2 ? cs : sn);
        if (i) v[1] = r;
        else v[0] = r;
      }
      uint32_t p[NS];
      modp_split2<NS>(v[0], v[1], p);
#pragma unroll
      for (int n = 0; n < NS; ++n) {  // element pair e, by selects: the loop stays rolled
        x[n][0] = e == 0 ? p[n] : x[n][0];
        x[n][1] = e == 1 ? p[n] : x[n][1];
        x[n][2] = e == 2 ? p[n] : x[n][2];
        x[n][3] = e == 3 ? p[n] : x[n][3];
      }
    }
#pragma unroll
    for (int n = NS - 1; n >= 0; --n) acc = mfma16(w, __builtin_bit_cast(bf16x8, x[n]), acc);  // the small parts first
  }
  const f32x4 z = modin2_sum(acc, wave, lane);
  const int row = blockIdx.y * 16 + (lane & 15), c0 = n0 + 4 * g;
  if (wave == 0 && row < a.N) {
    f32x4 o = z + *reinterpret_cast<const f32x4*>(a.t1_b + c0);
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = o[i] / (1.f + __expf(-o[i]));
    *reinterpret_cast<f32x4*>(h1 + (int64_t)row * a.H + c0) = o;
  }
}

// c[b][k][n] = h1[k] W2^T + b2 + state_cond[b]
__global__ __launch_bounds__(64 * MODIN2_WAVES) void modin_out_kernel(mkx_modin_args a, const float* __restrict__ h1) {
  constexpr int NS = MODIN_NS;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4;
  const int row = blockIdx.y * 16 + (lane & 15), n0 = blockIdx.x * 16, c0 = n0 + 4 * g;
  const float* hp = h1 + (int64_t)min(row, a.N - 1) * a.H + 8 * g;
  const bf16_t* w2 = (const bf16_t*)a.t2_w + (int64_t)(n0 + (lane & 15)) * a.H + 8 * g;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int kb = wave; kb < a.H / 32; kb += MODIN2_WAVES) {
    const bf16x8 w = __builtin_bit_cast(bf16x8, ld16(w2 + 32 * kb));
    const f32x4 v0 = *reinterpret_cast<const f32x4*>(hp + 32 * kb), v1 = *reinterpret_cast<const f32x4*>(hp + 32 * kb + 4);
    u32x4 x[NS];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      uint32_t p[NS];
      modp_split2<NS>(e < 2 ? v0[2 * e] : v1[2 * e - 4], e < 2 ? v0[2 * e + 1] : v1[2 * e - 3], p);
#pragma unroll
      for (int n = 0; n < NS; ++n) x[n][e] = p[n];
    }
#pragma unroll
    for (int n = NS - 1; n >= 0; --n) acc = mfma16(w, __builtin_bit_cast(bf16x8, x[n]), acc);
  }
  const f32x4 z = modin2_sum(acc, wave, lane) + *reinterpret_cast<const f32x4*>(a.t2_b + c0);
  if (row >= a.N) return;
  for (int b = wave; b < a.B; b += MODIN2_WAVES)
    *reinterpret_cast<f32x4*>(a.out + (int64_t)b * a.out_stride_b + (int64_t)row * a.out_stride_k + c0) =
        z + *reinterpret_cast<const f32x4*>(a.state_cond + (int64_t)b * a.sc_stride + c0);
}

}  // namespace mkx
