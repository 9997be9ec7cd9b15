// Cross-attention source K/V preparation: per layer, the VLM context projected onto the expert's
// cross-attention K and V, K normed per head (weight 1 + w) and rotated (rotate-half RoPE at the source
// positions), bf16 [B, SP, NH, 64] with rows >= ca_len zero — the caches the megakernel reads as
// past.cross_attn_kv (src/mk_expert.py:491-492), produced by REKI's register_prepare (README.md:279-281:
// "the cross-attention K/V projections of the VLM source (31 M weights)").
//
// The product runs on v_mfma_f32_16x16x32_bf16 with the weight rows as the first operand, so a lane ends
// with 4 consecutive columns of each 16-column group for one source row: the RMS of a row is a sum over the
// lane's 16 values and two cross-lane swaps, and each column's RoPE partner (d +- 32) sits in the same
// lane. Both operands are read in fragment order, one contiguous 1 KB block per fragment: the weights are
// packed so once at creation and the context at each call (pack_ctx_kernel, which also numbers the valid rows).
#pragma once

#include "mkx.h"
#include "mkx_device.h"
#include "mkx_kernel.h"  // cvt_pk (two fp32 -> bf16 pair)

namespace mkx {

constexpr int PREP_BLOCK = 256;

// Fragment-order packing of a row-major bf16 matrix [rows, C]: out[g][t][j][lane][8] = in[row][k .. k + 8)
// with row = (g * S + j) * 16 + (lane & 15), k = 32 t + 8 (lane >> 4); rows >= nrows are zero. One thread
// per 16-byte output piece (n_out pieces).
__global__ __launch_bounds__(256) void pack_rows_kernel(const bf16_t* __restrict__ in, bf16_t* __restrict__ out,
                                                        int nrows, int C, int S, long long n_out) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n_out) return;
  const int lane = (int)(i & 63);
  const long long q = i >> 6;
  const int T = C / 32;
  const int j = (int)(q % S);
  const long long gt = q / S;
  const int t = (int)(gt % T);
  const long long g = gt / T;
  const long long row = (g * S + j) * 16 + (lane & 15);
  u32x4 v = {0u, 0u, 0u, 0u};
  if (row < nrows) v = ld16(in + row * C + 32 * t + 8 * (lane >> 4));
  *reinterpret_cast<u32x4*>(out + i * 8) = v;
}

// Valid source rows: sample b's rows [0, len_b), len_b = ca_len[b] clamped to [0, SP]. Calls of at most
// PREP_MAP_B samples number them densely over the samples (row v of the packed context), so that no product is
// computed for rows past a sample's length (eight prompts of 300 down to 41 rows: 1364 of 2400 rows); calls of
// more samples number every row, v = b SP + s.
constexpr int PREP_MAP_B = 64;
struct PrepRows {
  const int* ends;  // LDS, two samples and more: valid rows of samples 0 .. b
  int nv;           // rows numbered
};
// The first of n ascending keys that is above v (the last at the latest), by halves. The search runs per lane on LDS: a
// scan of the samples by lane reads of the prefix sums took as many steps as there are samples (64 samples of 37 rows
// 244 us a call against 196 with the rows numbered by division) and read lanes that the caller's branch had switched off.
template <class F>
__host__ __device__ constexpr int prep_first_above(int v, int n, F key) {
  int b = 0, d = 1;
  while (2 * d < n) d *= 2;
  for (; d > 0; d /= 2)
    if (b + d < n && v >= key(b + d - 1)) b += d;
  return b;
}
// (every thread of the workgroup calls this once, ahead of any return; `ends` is LDS of the caller's)
__device__ __forceinline__ PrepRows prep_rows(const int32_t* ca_len, int B, int SP, int (&ends)[PREP_MAP_B]) {
  if (B > PREP_MAP_B) return PrepRows{ends, B * SP};
  if (B == 1) return PrepRows{ends, min(max(ca_len[0], 0), SP)};
  if (threadIdx.x < 64) {
    const int lane = threadIdx.x;
    int n = lane < B ? min(max(ca_len[lane], 0), SP) : 0;
    for (int d = 1; d < B; d *= 2) {
      const int o = __shfl_up(n, d);
      if (lane >= d) n += o;
    }
    ends[lane] = n;
  }
  __syncthreads();
  return PrepRows{ends, __builtin_amdgcn_readfirstlane(ends[B - 1])};
}
// (sample, source row) of row v < nv
__device__ __forceinline__ void prep_row_at(int v, int B, int SP, const PrepRows& rows, int& b, int& s) {
  if (B > PREP_MAP_B) {
    b = v / SP;
    s = v - b * SP;
    return;
  }
  b = prep_first_above(v, B, [&](int i) { return rows.ends[i]; });
  s = v - (b ? rows.ends[b - 1] : 0);
}

// The call's context [B, SP, C] into fragment order by row number v: out[g][t][j][lane][8] as pack_rows_kernel,
// S row tiles per group; the rows that pad the last group are zero, groups past it are not written (no
// workgroup reads them).
__global__ __launch_bounds__(256) void pack_ctx_kernel(const bf16_t* __restrict__ in, bf16_t* __restrict__ out,
                                                       const int32_t* __restrict__ ca_len, int B, int SP, int C, int S,
                                                       long long n_out) {
  __shared__ int ends[PREP_MAP_B];
  const PrepRows rows = prep_rows(ca_len, B, SP, ends);
  const int nv = rows.nv;
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n_out) return;
  const int lane = (int)(i & 63);
  const long long q = i >> 6;
  const int T = C / 32;
  const int j = (int)(q % S);
  const long long gt = q / S;
  const int t = (int)(gt % T);
  const long long g = gt / T;
  if (g * S * 16 >= nv) return;
  const long long v = (g * S + j) * 16 + (lane & 15);
  u32x4 x = {0u, 0u, 0u, 0u};
  if (v < nv) {
    int b, s;
    prep_row_at((int)v, B, SP, rows, b, s);
    x = ld16(in + ((long long)b * SP + s) * C + 32 * t + 8 * (lane >> 4));
  }
  *reinterpret_cast<u32x4*>(out + i * 8) = x;
}

struct SourceParams {
  int L, NH, C, B, SP;
  int sbw;              // row groups per block of the workgroup order
  const bf16_t* ctxp;   // context in fragment order, S = NRT (one group per workgroup), rows padded to whole groups
  const bf16_t* wkp;    // K weights in fragment order, S = 4 (16-row groups of one head)
  const bf16_t* wvp;
  const bf16_t* k_norm; // [L, 64]
  const int32_t* ca_len;
  const float* cos; const float* sin;
  void* kca[MKX_MAX_LAYERS]; void* vca[MKX_MAX_LAYERS];
  long long src_sb;
  float eps;
};

// The packed context is padded to PREP_ROW_PAD more rows than the largest workgroup covers.
constexpr int PREP_ROW_PAD = 16 * 5;
constexpr int PREP_L2_CTX = 2 << 20;  // context bytes per block of the workgroup order: half an XCD's L2
constexpr int PREP_XCDS = 8;  // XCDs the dispatcher deals consecutive workgroups to
constexpr int PREP_UPP = 4;   // (row tile, head) units of the result summed over the waves and stored per phase

// k-blocks of weight fragments a wave has in flight or in use (the accumulators leave the registers for that)
template <int NRT>
constexpr int prep_wbufs() { return NRT <= 3 ? 4 : NRT <= 4 ? 3 : 2; }

// One unit of the result: 16 rows (numbered row tile) x head h of K or V of layer l. prep_unit_load finds the lane's row and
// issues its RoPE loads, ahead of the sum over the waves; prep_unit sums the waves' parts ([wave][column
// tile][lane]) in wave order, rounds, norms and rotates (K) and stores.
struct PrepUnit {
  int b, s;
  bool stored, live;
  f32x4 csv[4], snv[4];
};
__device__ __forceinline__ void prep_unit_load(PrepUnit& q, const SourceParams& a, const PrepRows& rows, int tile, int is_v, int lane) {
  const int row = tile * 16 + (lane & 15);
  q.stored = row < rows.nv;
  // rows past the end (zero in the packed context) are not stored
  prep_row_at(min(row, rows.nv - 1), a.B, a.SP, rows, q.b, q.s);
  // (with every row numbered, those past their sample's length are stored as zero here)
  q.live = a.B <= PREP_MAP_B || q.s < a.ca_len[q.b];
  if (!is_v) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      q.csv[j] = *reinterpret_cast<const f32x4*>(a.cos + (int64_t)q.s * 64 + 16 * j + 4 * (lane >> 4));
      q.snv[j] = *reinterpret_cast<const f32x4*>(a.sin + (int64_t)q.s * 64 + 16 * j + 4 * (lane >> 4));
    }
  }
}
__device__ __forceinline__ void prep_unit(const PrepUnit& q, const SourceParams& a, const f32x4* pt, int h, int is_v, bf16_t* outl,
                                          const uint2 (&wnv)[4], int lane) {
  f32x4 v4[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    f32x4 p[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) p[w] = pt[(w * 4 + j) * 64 + lane];
    v4[j] = ((p[0] + p[1]) + p[2]) + p[3];
  }
  // columns in pairs (2 e, 2 e + 1) of each group, rounded to bf16 by the packed hardware conversion
  uint32_t yp[4][2];
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int e = 0; e < 2; ++e) yp[j][e] = cvt_pk(v4[j][2 * e], v4[j][2 * e + 1]);
  if (!is_v) {
    float y[4][4];
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        y[j][2 * e] = __uint_as_float(yp[j][e] << 16);
        y[j][2 * e + 1] = __uint_as_float(yp[j][e] & 0xffff0000u);
        ss += y[j][2 * e] * y[j][2 * e];
        ss += y[j][2 * e + 1] * y[j][2 * e + 1];
      }
    ss = xor32_sum(xor16_sum(ss));
    const float r = rsqrtf(ss / 64.f + a.eps);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float wv[4] = {__uint_as_float(wnv[j].x << 16), __uint_as_float(wnv[j].x & 0xffff0000u),
                           __uint_as_float(wnv[j].y << 16), __uint_as_float(wnv[j].y & 0xffff0000u)};
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const uint32_t n = cvt_pk(y[j][2 * e] * r * (1.f + wv[2 * e]), y[j][2 * e + 1] * r * (1.f + wv[2 * e + 1]));
        y[j][2 * e] = __uint_as_float(n << 16);
        y[j][2 * e + 1] = __uint_as_float(n & 0xffff0000u);
      }
    }
    {
#pragma clang fp contract(off)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float z[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float rot = j < 2 ? -y[j + 2][i] : y[j - 2][i];
          z[i] = y[j][i] * q.csv[j][i] + rot * q.snv[j][i];
        }
        yp[j][0] = cvt_pk(z[0], z[1]);
        yp[j][1] = cvt_pk(z[2], z[3]);
      }
    }
  }
  if (!q.stored || h >= a.NH) return;
  bf16_t* out = outl + (int64_t)q.b * a.src_sb + ((int64_t)q.s * a.NH + h) * 64;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    u32x2 v;
    v[0] = q.live ? yp[j][0] : 0u;
    v[1] = q.live ? yp[j][1] : 0u;
    *reinterpret_cast<u32x2*>(out + 16 * j + 4 * (lane >> 4)) = v;
  }
}

// grid: x = row groups of NRT 16-row tiles, y = (layer * 2 + (0: K, 1: V)) * ceil(NH / 2) + head pair.
// Workgroup = 16 NRT numbered source rows x two heads (128 columns) of K or V of one layer. Each of the 4 waves computes
// the whole tile over a quarter of the k-blocks (wave, wave + 4, ...) and the quarters are summed through LDS in wave
// order: no wave needs another's operands, so the k-loop has no LDS, no barrier and no wave in step with another,
// and a wave's NRT + 8 fragments (1 KB each, straight into registers) feed 8 NRT MFMAs. Shared through LDS by
// waves that split the tile instead (80 x 64 each, fragments written once and read by two waves per k-block, one
// barrier per k-block), the k-loop took 1180 cycles per k-block and 160 x 128 tile against 320 of MFMA: the LDS
// traffic, the issue of its instructions and the barrier follow one another with one wave per SIMD.
// A row tile's fragment is loaded again right behind its last MFMA (one k-block ahead), the weights, which come
// from memory where the context comes from L2, prep_wbufs() - 1 k-blocks ahead; loads and MFMAs alternate, so that the
// wave does not stand at a full load queue. Rows past a sample's valid length are zero in the result: the row
// groups' workgroups share the stores of them. At most 5 row tiles, so that two workgroups share a CU (256 registers a
// wave) and one's first loads and epilogue run beside the other's MFMAs.
// Measured (10 layers, 12 heads, C 2048): one call of 300 rows 44.4 -> 31 us (609 TFLOP/s; a large matrix product
// reaches 1115), eight of 300 down to 41 rows 183.6 -> 120 us, of which the numbering of the valid rows gives the
// larger part. No unit is full there: the matrix cores are busy 29 % of the time, operands come at 25 bytes per cycle and CU
// (an L2-resident stream alone reaches 46 to 56), and the waves spend 39 % of theirs waiting for operands and 32 %
// waiting to issue: 2160 workgroups in 4.2 rounds of two per CU, each with a start and an epilogue of its own.
template <int NRT>
__global__ __launch_bounds__(PREP_BLOCK, 2) void prepare_source_kernel(SourceParams a) {
  constexpr int WB = prep_wbufs<NRT>();
  __shared__ __attribute__((aligned(1024))) char sm[4 * PREP_UPP * 4096];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int NH = a.NH, T = a.C / 32, NP = (NH + 1) / 2;
  // Order: blocks of a.sbw row groups whose context stays in an L2 (PREP_L2_CTX bytes), within a block every column
  // group. Consecutive workgroups run on different XCDs (round-robin dispatch), so a block's linear index is regrouped to
  // give each XCD a contiguous run of (column group, row group) tiles, row group fastest: the row groups of one
  // column group then share its weight fragments, and the block's column groups its context, in their XCD's L2 (with
  // every row group in one block the 5.6 MB of 1364 rows came from beyond the L2 for each column group anew: 138 us
  // instead of 127).
  const int ngr = gridDim.x, ncg = gridDim.y, lin = blockIdx.y * ngr + blockIdx.x;
  const int sb = lin / (a.sbw * ncg), rs = lin - sb * a.sbw * ncg, sw = min(a.sbw, ngr - sb * a.sbw);
  const int nwg = sw * ncg, nfull = nwg - nwg % PREP_XCDS, per = nfull / PREP_XCDS;
  const int tix = rs < nfull ? (rs % PREP_XCDS) * per + rs / PREP_XCDS : rs;
  const int rg = sb * a.sbw + tix % sw, cgp = tix / sw;
  const int pair = cgp % NP, lk = cgp / NP, l = lk >> 1, is_v = lk & 1;
  bf16_t* const outl = (bf16_t*)(is_v ? a.vca[l] : a.kca[l]);
  __shared__ int ends[PREP_MAP_B];
  const PrepRows rows = prep_rows(a.ca_len, a.B, a.SP, ends);
  const int nv = rows.nv;
  if (a.B <= PREP_MAP_B && nv < a.B * a.SP) {
    // this row group's share of the rows past their sample's length (numbered over the samples), zeroed: 16 bytes
    // per thread, 8 or 16 threads per row (this workgroup's columns)
    const int nd = a.B * a.SP - nv, d1 = (int)((long long)nd * (rg + 1) / ngr);
    const int tpr = 2 * pair + 1 < NH ? 16 : 8, piece = threadIdx.x % tpr;
    for (int d = (int)((long long)nd * rg / ngr) + (int)threadIdx.x / tpr; d < d1; d += PREP_BLOCK / tpr) {
      const int b = prep_first_above(d, a.B, [&](int i) { return (i + 1) * a.SP - rows.ends[i]; });
      const int past = b ? rows.ends[b - 1] : 0, len = (a.B > 1 ? rows.ends[b] : nv) - past;
      const int s = d - (b * a.SP - past) + len;  // (the sample's valid rows come first)
      bf16_t* o = outl + (int64_t)b * a.src_sb + ((int64_t)s * NH + 2 * pair) * 64 + piece * 8;
      const u32x2 z = {0u, 0u};
      *reinterpret_cast<u32x2*>(o) = z;
      *reinterpret_cast<u32x2*>(o + 4) = z;
    }
  }
  const int g0 = rg * NRT;  // first 16-row tile of the workgroup
  if (g0 * 16 >= nv) return;
  // fragments of k-block kb: context row tile r at (kb NRT + r) KB of the row group, weight column tile j at
  // (kb 4 + j % 4) KB of head j / 4 (an odd head count's last pair repeats its head, never stored)
  // (64-bit k-block offsets: a context of 2^25 columns has 4 GB of weights per head)
  const uint32_t vl = (uint32_t)lane * 16;
  const char* const xsrc = (const char*)(a.ctxp + (int64_t)rg * T * NRT * 512);
  const char* const wsrc0 = (const char*)((is_v ? a.wvp : a.wkp) + (int64_t)(l * NH + 2 * pair) * T * 2048);
  const char* const wsrc1 = 2 * pair + 1 < NH ? wsrc0 + (int64_t)T * 4096 : wsrc0;
  const int nk = (T - wave + 3) / 4;  // this wave's k-blocks (0 where T < 4 leaves it none)
  auto ldw = [&](int i, int j) {  // (past the last k-block: that one again, unused)
    const int kb = min(wave + 4 * max(min(i, nk - 1), 0), T - 1);
    return bload(rsrc((j < 4 ? wsrc0 : wsrc1) + (int64_t)kb * 4096), vl + (j & 3) * 1024, 0);
  };
  auto ldx = [&](int i, int r) {
    const int kb = min(wave + 4 * max(min(i, nk - 1), 0), T - 1);
    return bload(rsrc(xsrc + (int64_t)kb * NRT * 1024), vl, r * 1024);
  };
  u32x4 xf[NRT], wf[WB][8];
#pragma unroll
  for (int j = 0; j < 8; ++j) wf[0][j] = ldw(0, j);
#pragma unroll
  for (int r = 0; r < NRT; ++r) xf[r] = ldx(0, r);
#pragma unroll
  for (int s = 1; s < WB - 1; ++s)
#pragma unroll
    for (int j = 0; j < 8; ++j) wf[s][j] = ldw(s, j);
  f32x4 acc[NRT][8];
#pragma unroll
  for (int r = 0; r < NRT; ++r)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[r][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  // k-block i of the wave, weights in slot s = i % WB: per row tile its 8 MFMAs, its next fragment and its share of
  // the weights of k-block i + WB - 1 (into the slot of k-block i - 1)
  auto step = [&](int s, int i) {
    const int ws = (s + WB - 1) % WB;
#pragma unroll
    for (int r = 0; r < NRT; ++r) {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        acc[r][j] = mfma16(__builtin_bit_cast(bf16x8, wf[s][j]), __builtin_bit_cast(bf16x8, xf[r]), acc[r][j]);
      xf[r] = ldx(i + 1, r);
#pragma unroll
      for (int j = r * 8 / NRT; j < (r + 1) * 8 / NRT; ++j) wf[ws][j] = ldw(i + WB - 1, j);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  int i0 = 0;
  for (; i0 + WB <= nk; i0 += WB) {
#pragma unroll
    for (int s = 0; s < WB; ++s) step(s, i0 + s);
  }
#pragma unroll
  for (int s = 0; s < WB - 1; ++s)
    if (i0 + s < nk) step(s, i0 + s);
  // the lane's number anew: kept over the k-loop, the thread index it came from was the one register too many there
  const int el = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
  // the K norm weights of this lane's 16 columns d = 16 j + 4 (lane >> 4) + i (4 bf16 per j)
  uint2 wnv[4];
  if (!is_v) {
#pragma unroll
    for (int j = 0; j < 4; ++j) wnv[j] = *reinterpret_cast<const uint2*>(a.k_norm + l * 64 + 16 * j + 4 * (el >> 4));
  }
  // Units u = (row tile u / 2, head u % 2), PREP_UPP per phase: every wave leaves its part of each in LDS
  // ([unit][wave][column tile][lane]), then each wave sums and stores one of them. Lane: columns d = 16 j + 4 (lane >> 4)
  // + i of source row `row`.
  f32x4* const pt = reinterpret_cast<f32x4*>(sm);
#pragma unroll
  for (int u0 = 0; u0 < 2 * NRT; u0 += PREP_UPP) {
    static_assert(PREP_UPP == 4, "one unit per wave and phase");
    const int u = min(u0 + wave, 2 * NRT - 1);  // (a last phase of fewer units repeats one, unstored)
    PrepUnit q;
    prep_unit_load(q, a, rows, g0 + (u >> 1), is_v, el);
    if (u0) __syncthreads();  // the phase before has been read
#pragma unroll
    for (int v = u0; v < min(u0 + PREP_UPP, 2 * NRT); ++v)
#pragma unroll
      for (int j = 0; j < 4; ++j) pt[(((v - u0) * 4 + wave) * 4 + j) * 64 + el] = acc[v >> 1][(v & 1) * 4 + j];
    __syncthreads();
    if (u0 + wave < 2 * NRT) prep_unit(q, a, pt + (u - u0) * 1024, 2 * pair + (u & 1), is_v, outl, wnv, el);
  }
}

}  // namespace mkx
