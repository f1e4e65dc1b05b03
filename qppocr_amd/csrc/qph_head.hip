// The fused rec head over a split weight: logits x[M][256] . w[256][N] + bias,
// softmax and argmax, of which only the (value, index) pair per row is stored.
//
// Each float32 operand is held as two float16 terms, v * s = h + l (+ e), with
// s a power of two per row of x and per column of w that puts the row's /
// column's largest magnitude in [2^14, 2^15): h the nearest float16, l the
// nearest float16 to the exact remainder.  |e| is at most one float32 ulp of v
// (and 0 for three values in four) for the elements within 2^-15 of the largest,
// and 2^-39 of the largest for the smaller ones.  A product keeps h.h, h.l and l.h;
// each is exact in float32, and v_mfma_f32_32x32x16_f16 adds them into a float32
// accumulator: 48 accumulator roundings per logit where the float32 chain has
// 256.  l.l, left out, is at most 2^-22 of a product (2^-24.6 in the mean square).
//
// So a logit of many terms is closer to float64 than the chain's, one of few
// terms is not, nor one whose terms are all far below the row's largest element
// (against a weight of 0).  Mean square error of the logits, split / chain, K =
// 256 terms of normal values: 4.1e-7 / 8.1e-7; operands spread over 2^20: half the
// chain's as well; 128 nonzero terms 1.0 / 1.3 of a value, 64: 2.1 / 2.05e-7, 16:
// 8.8 / 5.2e-8, 1: 14.8 / 4.9e-9; a channel of weight 0 at 2^16 times the others
// 4.3 / 8.1e-7, at 2^20 2.2e-6 / 8.1e-7.  Rows of fewer than HS_TERMS terms, or with
// a product past HS_PRODUCT (whose small elements could be off by 2^-18 of a logit's
// unit, in the worst case), are therefore computed in float32 (flagged_tile), and a
// weight with a column of so few terms keeps the session on the unsplit kernels.
// The pair values of the rec net are 2.5e-6 off (mean square, relative), the
// chain's 3.6e-6.
//
// What it measured (N = 18709; split rows + product + pairs, traced, against
// gemm_wave_kernel + head_pairs_kernel): 1280 rows 47.6 us against 128, 6800 rows
// 182 against 615, 24 rows 19 against 26.  What bounds it: the matrix cores are
// busy 78% of the cycles of head_split_kernel's loop, and at that load the clock
// falls from 2.1 to 1.7 GHz (3930 cycles a block of 32 columns, 2.3 us; the bare
// products 3445 cycles at 1.72 GHz); below some 64 rows the 19 MB of weight.
//
// Rows that hold an infinity, a NaN or a magnitude past 2^60 are flagged and
// computed in float32 too; a weight or bias that holds one keeps the session on
// the unsplit kernels (gemm_wave_kernel, head_pairs_kernel) altogether.
#include <cmath>
#include <algorithm>
#include <vector>

#include "qph_internal.h"

namespace qph {

typedef _Float16 h16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

#define HS_K 256                       // row length
#define HS_KS (HS_K / 16)              // MFMA steps
#define HS_BLOCK (HS_KS * 2 * 1024)    // bytes of a packed 32-column block
#define HS_STAGES 3
#define HS_ROWS 256                    // rows of a workgroup (64 a wave)
#define HS_MAX_LEN 224                 // most column blocks of a slice (their scales sit in LDS)
#define HS_SMALL 64                    // rows up to which each wave streams its own block
#define HS_LIMIT 1.152921504606847e18f // 2^60
#define HS_PRODUCT 4096.0f             // the largest |x| |w| a split row may have
#define HS_TERMS 96                    // and the fewest terms of a split row or column:
#define HS_TERM 9.5367431640625e-7f    // elements past 2^-20 of its largest (or none at all)
#define HS_L2E 1.44269504f

// 2^(14 - exponent of mx), so that mx times it lies in [2^14, 2^15); the
// exponent is held to 2^100 (a row of tiny or zero values).
__device__ __forceinline__ float pow2_scale(float mx) {
  const int e = (int)((__float_as_uint(mx) >> 23) & 0xff) - 127;
  const int se = min(14 - e, 100);
  return __uint_as_float((unsigned)(se + 127) << 23);
}

// Packs the weight: block cb holds columns 32 cb .. + 31 as, per MFMA step ks
// and term (h, l), the 64 lanes' eight float16 (lane L: column L % 32, k = 16
// ks + 8 (L / 32) ..), so a lane's operand is one 16-byte read and a wave's
// 1024 contiguous bytes.  ci: per column (2^-s log2 e, bias log2 e), past N (0, -3e38):
// such a column's exponential is 0 beside any other.  top[cb]: the block's
// largest magnitude, -1 where the block cannot be split (infinity, NaN, past
// 2^60, a column of few terms).
__global__ __launch_bounds__(256) void head_pack_kernel(const float* __restrict__ w, int n,
                                                        const float* __restrict__ bias,
                                                        _Float16* __restrict__ wp,
                                                        float2* __restrict__ ci,
                                                        float* __restrict__ top) {
  __shared__ float t[HS_K * 33];
  __shared__ float mxs[8 * 32];
  __shared__ float scs[32];
  __shared__ int bad;
  const int tid = threadIdx.x, c = tid & 31, part = tid >> 5;
  const int cb = blockIdx.x, j = cb * 32 + c;
  if (tid == 0) bad = 0;
  float mx = 0.0f;
  bool odd = false;
  for (int q = 0; q < HS_K / 8; q++) {
    const int k = part * (HS_K / 8) + q;
    const float v = j < n ? w[(int64_t)k * n + j] : 0.0f;
    t[k * 33 + c] = v;
    const float a = __builtin_fabsf(v);
    odd = odd || !(a <= HS_LIMIT);
    mx = fmaxf(mx, a);
  }
  mxs[part * 32 + c] = mx;
  __syncthreads();
  if (odd) bad = 1;
  if (tid < 32) {
    for (int q = 1; q < 8; q++) mx = fmaxf(mx, mxs[q * 32 + c]);
    int terms = 0;
    for (int k = 0; k < HS_K; k++) terms += __builtin_fabsf(t[k * 33 + c]) > mx * HS_TERM;
    if (terms > 0 && terms < HS_TERMS) bad = 1;
    const float s = pow2_scale(mx);
    scs[c] = s;
    const float b = j < n && bias ? bias[j] : 0.0f;
    if (!(__builtin_fabsf(b) <= HS_LIMIT)) bad = 1;
    float2 o;
    o.x = j < n ? (1.0f / s) * HS_L2E : 0.0f;
    o.y = j < n ? b * HS_L2E : -3.0e38f;
    ci[j] = o;
    mxs[c] = mx;
  }
  __syncthreads();
  for (int q = tid; q < HS_KS * 64; q += 256) {
    const int ks = q >> 6, lane = q & 63;
    const int col = lane & 31, k0 = 16 * ks + 8 * (lane >> 5);
    h16x8 h, l;
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const float v = t[(k0 + i) * 33 + col] * scs[col];
      h[i] = (_Float16)v;
      l[i] = (_Float16)(v - (float)h[i]);
    }
    h16x8* o = (h16x8*)wp + (int64_t)cb * (HS_BLOCK / 16) + ks * 128 + lane;
    o[0] = h;
    o[64] = l;
  }
  if (tid == 0) {
    for (int q = 1; q < 32; q++) mx = fmaxf(mx, mxs[q]);
    top[cb] = bad ? -1.0f : mx;
  }
}

// The rows of x as split MFMA operands, one workgroup per 32 rows: xs holds per
// row tile and step ks the h and the l terms of the 64 lanes (lane L: row
// L % 32, k = 16 ks + 8 (L / 32) ..), so that a wave reads 1 KB at a time; rs
// holds each row's 2^-s, -1 for a flagged row (whose terms are 0); wmax is the
// weight's largest magnitude.  Rows past m repeat the last one.  Made once per
// run in a launch of its own (4.8 us at 1280 rows): splitting its own rows cost
// every workgroup of the product about 10 us (strided reads, some 1300
// conversions a lane).
__global__ __launch_bounds__(256) void head_rows_kernel(const float* __restrict__ x, int m,
                                                        float wmax, _Float16* __restrict__ xs,
                                                        float* __restrict__ rs) {
  typedef _Float16 h16x4 __attribute__((ext_vector_type(4)));
  const int tid = threadIdx.x, r = tid >> 3, c = tid & 7;
  const float* xr = x + (int64_t)min((int)blockIdx.x * 32 + r, m - 1) * HS_K + 4 * c;
  f32x4 raw[HS_K / 32];
#pragma unroll
  for (int i = 0; i < HS_K / 32; i++) raw[i] = *(const f32x4*)(xr + 32 * i);
  float mx = 0.0f;
  int odd = 0;
#pragma unroll
  for (int i = 0; i < HS_K / 32; i++)
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const float a = __builtin_fabsf(raw[i][u]);
      odd |= !(a <= HS_LIMIT);
      mx = fmaxf(mx, a);
    }
#pragma unroll
  for (int off = 4; off >= 1; off >>= 1) {
    mx = fmaxf(mx, __shfl_xor(mx, off, 64));
    odd |= __shfl_xor(odd, off, 64);
  }
  int terms = 0;
#pragma unroll
  for (int i = 0; i < HS_K / 32; i++)
#pragma unroll
    for (int u = 0; u < 4; u++) terms += __builtin_fabsf(raw[i][u]) > mx * HS_TERM;
#pragma unroll
  for (int off = 4; off >= 1; off >>= 1) terms += __shfl_xor(terms, off, 64);
  odd |= !(mx * wmax <= HS_PRODUCT) || (terms > 0 && terms < HS_TERMS);
  const float s = pow2_scale(mx);
#pragma unroll
  for (int i = 0; i < HS_K / 32; i++) {
    h16x4 h, l;
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const float v = odd ? 0.0f : raw[i][u] * s;
      h[u] = (_Float16)v;
      l[u] = (_Float16)(v - (float)h[u]);
    }
    const int k = 32 * i + 4 * c;
    _Float16* o = xs + ((int64_t)blockIdx.x * HS_KS + (k >> 4)) * 1024 +
                  (((k >> 3) & 1) * 32 + r) * 8 + (k & 7);
    *(h16x4*)o = h;
    *(h16x4*)(o + 512) = l;
  }
  if (c == 0) rs[blockIdx.x * 32 + r] = odd ? -1.0f : 1.0f / s;
}

// A wave's operands of one step of a row tile, from xs.
__device__ __forceinline__ void load_rows(const _Float16* __restrict__ xs, int tile, int ks,
                                          h16x8& ah, h16x8& al) {
  const h16x8* p = (const h16x8*)xs + (int64_t)(tile * HS_KS + ks) * 128 + (threadIdx.x & 63);
  ah = p[0];
  al = p[64];
}

// Running (max, block of the first max, sum of exponentials against that max)
// of one row's columns lane % 32, 32 + lane % 32, ..., all in powers of two.  A
// sum is taken against its own running max, so it lies between 1 and the
// column count whatever the row's logits are.  (Columns past N alone leave a max
// of -3e38, whose sum the first real column's exponential, 0, clears.)
struct RowState {
  float m[16], s[16];
  int b[16];
};

__device__ __forceinline__ void state_init(RowState& st) {
#pragma unroll
  for (int v = 0; v < 16; v++) {
    st.m[v] = -3.0e38f;
    st.s[v] = 0.0f;
    st.b[v] = 0;
  }
}

// Value v of a block's 32x32 accumulators (lane: column L % 32, rows 8 (v / 4) +
// 4 (L / 32) + v % 4).  F32: of a flagged tile, in natural units (c.y the bias).
template <bool F32>
__device__ __forceinline__ float exp_less(float d) {
  return __builtin_amdgcn_exp2f(F32 ? d * HS_L2E : d);
}

template <bool F32>
__device__ __forceinline__ void state_add(RowState& st, int v, float acc, float sr, float2 c,
                                          int blk) {
  const float t = F32 ? acc + c.y : __builtin_fmaf(acc * sr, c.x, c.y);
  // the lesser of the two against the larger: one exponential either way
  const float e = exp_less<F32>(-__builtin_fabsf(t - st.m[v]));
  const bool up = t > st.m[v];
  st.s[v] = __builtin_fmaf(st.s[v], up ? e : 1.0f, up ? 1.0f : e);
  st.b[v] = up ? blk : st.b[v];
  st.m[v] = up ? t : st.m[v];
}

// The 32 lanes of each half meet, each step halving the rows a lane still
// holds; then lane 2 v of a half stores row v's (max, first column of the max,
// sum, flag) if the row is flagged (F32) or is not.
template <bool F32>
__device__ __forceinline__ void state_store(RowState& st, const float* rw, int m, int row,
                                            int slices, int slice, float* __restrict__ part) {
  const int lane = threadIdx.x & 63, lr = lane & 31, lh = lane >> 5;
#pragma unroll
  for (int v = 0; v < 16; v++) st.b[v] = st.b[v] * 32 + lr;
  auto meet = [&](int v, float mo, float so, int io) {
    const float mm = fmaxf(st.m[v], mo);
    st.s[v] = st.s[v] * exp_less<F32>(st.m[v] - mm) + so * exp_less<F32>(mo - mm);
    const int first = min(io, st.b[v]);
    st.b[v] = mo > st.m[v] ? io : mo == st.m[v] ? first : st.b[v];
    st.m[v] = mm;
  };
#pragma unroll
  for (int step = 3; step >= 0; step--) {
    const int half = 1 << step;
    const bool hi = (lr & (2 * half)) != 0;
#pragma unroll
    for (int v = 0; v < 8; v++) {
      if (v >= half) break;
      const float mo = __shfl_xor(hi ? st.m[v] : st.m[v + half], 2 * half, 64);
      const float so = __shfl_xor(hi ? st.s[v] : st.s[v + half], 2 * half, 64);
      const int io = __shfl_xor(hi ? st.b[v] : st.b[v + half], 2 * half, 64);
      st.m[v] = hi ? st.m[v + half] : st.m[v];
      st.s[v] = hi ? st.s[v + half] : st.s[v];
      st.b[v] = hi ? st.b[v + half] : st.b[v];
      meet(v, mo, so, io);
    }
  }
  meet(0, __shfl_xor(st.m[0], 1, 64), __shfl_xor(st.s[0], 1, 64), __shfl_xor(st.b[0], 1, 64));
  const int v = lr >> 1;
  const int r = 8 * (v >> 2) + 4 * lh + (v & 3);
  if (!(lr & 1) && row + r < m && (rw[r] < 0.0f) == F32) {
    f32x4 o;
    o[0] = st.m[0];
    o[1] = __int_as_float(st.b[0]);
    o[2] = st.s[0];
    o[3] = F32 ? 1.0f : 0.0f;   // (in every slice alike)
    *(f32x4*)(part + ((int64_t)(row + r) * slices + slice) * 4) = o;
  }
}

// The partials of a tile's flagged rows over column blocks b0 .. b0 + len - 1, in
// float32: the whole tile's logits on v_mfma_f32_32x32x2f32, whose two k terms are
// added in order (the fma chain of the unsplit kernels), an infinity or a NaN
// staying in its own row.  Every slice does its share: one such row among 1280
// costs a call 70 us and 1280 of them 170 (as much as the unsplit kernels take for
// the whole head, and half as much again); a wave a row in the pairs kernel took
// 7.6 ms for the first.
__device__ __forceinline__ void flagged_tile(const float* __restrict__ x, int m,
                                             const float* __restrict__ w, int n,
                                             const float* __restrict__ bias, int row, int b0,
                                             int len, const float* rw, int slices, int slice,
                                             float* __restrict__ part) {
  const int lane = threadIdx.x & 63, lr = lane & 31, lh = lane >> 5;
  // operands: lane (row or column L % 32, half L / 32), k = 2 s + half of step s
  const float* xr = x + (int64_t)min(row + lr, m - 1) * HS_K + lh;
  float a[HS_K / 2];
#pragma unroll
  for (int s = 0; s < HS_K / 2; s++) a[s] = xr[2 * s];
  RowState st;
  state_init(st);
#pragma unroll 1
  for (int b = b0; b < b0 + len; b++) {
    const int j = b * 32 + lr, jc = min(j, n - 1);
    const float* wc = w + (int64_t)lh * n + jc;
    // the block's loads all in flight (left alone, the scheduler puts most of
    // them one by one between the products)
    float q[HS_K / 2];
#pragma unroll
    for (int s = 0; s < HS_K / 2; s++) q[s] = wc[(int64_t)(2 * s) * n];
    __builtin_amdgcn_sched_barrier(0);
    f32x16 acc = {};
#pragma unroll
    for (int s = 0; s < HS_K / 2; s++)
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[s], q[s], acc, 0, 0, 0);
    const float2 c = {0.0f, bias ? bias[jc] : -0.0f};
#pragma unroll
    for (int v = 0; v < 16; v++)
      state_add<true>(st, v, j < n ? acc[v] : -3.0e38f, 0.0f, j < n ? c : float2{0.0f, 0.0f}, b);
  }
  state_store<true>(st, rw, m, row, slices, slice, part);
}

// Workgroup (row tile of 256, slice of the column blocks): each of the four
// waves keeps its 64 rows' split operands in registers (256 of the 512 that one
// wave a SIMD has) for the whole slice; the blocks stream through a ring of
// three 32 KB LDS stages that all waves read, two in flight.  A block is two
// chains of 48 MFMAs a wave; the softmax state takes the block before it in
// between, two values a step, in the shadow of the products.  With 32 rows a
// wave and eight waves the same LDS reads fed half as many products, and the two
// waves of a SIMD fell into step with each other: 3.0 us a block.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void
head_split_kernel(const _Float16* __restrict__ xs, const float* __restrict__ rsc, int m,
                  const _Float16* __restrict__ wp, const float2* __restrict__ ci, int nb,
                  int tiles, int slices, int share, int extra, int per_xcd,
                  float* __restrict__ part, const float* __restrict__ x,
                  const float* __restrict__ w, int n, const float* __restrict__ bias) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  // slice-major over the XCDs: the row tiles of one slice share an XCD's L2;
  // a slice is share blocks, the first `extra` ones one more
  const int u = (int)(blockIdx.x % 8) * per_xcd + (int)(blockIdx.x / 8);
  if (u >= tiles * slices) return;
  const int slice = u / tiles, tile = u - slice * tiles;
  const int b0 = slice * share + min(slice, extra);
  const int len = share + (slice < extra ? 1 : 0);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, lr = lane & 31;
  float* srl = (float*)(lds + HS_STAGES * HS_BLOCK);   // the rows' scales
  float2* cil = (float2*)(srl + HS_ROWS);
  const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
      (void*)wp, 0, nb * HS_BLOCK, 0x00020000);
  // eight 1 KB loads a wave and stage (the asm keeps the compiler from waiting
  // for them before the reads of another stage)
  const unsigned voff = (unsigned)(wave * 8192 + lane * 16);
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
  auto issue = [&](int b, int st) {
#pragma unroll
    for (int q = 0; q < 8; q++) {
      const unsigned dst = lds0 + (unsigned)(st * HS_BLOCK + wave * 8192 + q * 1024);
      const unsigned soff = (unsigned)((b0 + b) * HS_BLOCK + q * 1024);
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"   // m0 is reserved; nothing else uses it here
      __asm__ volatile(QPH_M0 "buffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(dst),
                       "v"(voff), "s"(wr), "s"(soff)
                       : "m0", "memory");
#pragma clang diagnostic pop
    }
  };
  const int row = tile * HS_ROWS + wave * 64;
  const bool rows = row < m;
  // a wave's second 32 rows past the last row tile repeat its first
  const int rt0 = rows ? row / 32 : 0, rt1 = row + 32 < m ? rt0 + 1 : rt0;
  h16x8 ah[2][HS_KS], al[2][HS_KS];
#pragma unroll
  for (int ks = 0; ks < HS_KS; ks++) {
    load_rows(xs, rt0, ks, ah[0][ks], al[0][ks]);
    load_rows(xs, rt1, ks, ah[1][ks], al[1][ks]);
  }
  srl[wave * 64 + lane] = rsc[(lane < 32 ? rt0 : rt1) * 32 + lr];
  for (int i = threadIdx.x; i < len * 32; i += 256) cil[i] = ci[b0 * 32 + i];
  // (spelled out, so that the loop below has no waits for these loads: they
  // would wait for the stages in flight as well)
  wait_vmcnt<0>();
  __syncthreads();
  // 224 of the 256 operand registers and the products' 32 are the accumulation
  // ones, the rest the others: without the hint the allocator mixes them and
  // copies operands in every step (4270 cycles a block with 256, 5590 without)
#pragma unroll
  for (int ks = 0; ks < HS_KS; ks++) {
    __asm__ volatile("" : "+a"(ah[0][ks]), "+a"(ah[1][ks]), "+a"(al[0][ks]));
    if (ks < HS_KS / 2) __asm__ volatile("" : "+a"(al[1][ks]));
    else __asm__ volatile("" : "+v"(al[1][ks]));
  }
  issue(0, 0);
  if (len > 1) issue(1, 1);
  const float* rw = srl + wave * 64;
  const float* rh = rw + 4 * (lane >> 5);
  RowState rs[2];
  state_init(rs[0]);
  state_init(rs[1]);
  // before the first block: a column like those past N
  f32x16 prev[2] = {};
  float2 pc = {0.0f, -3.0e38f};
  int st = 0;
  for (int b = 0; b < len; b++) {
    // this wave's share of block b is in; after the barrier everyone's is,
    // and nobody reads block b - 1's stage any more
    if (b + 1 < len) wait_vmcnt<8>();
    else wait_vmcnt<0>();
    __asm__ volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    __asm__ volatile("" ::: "memory");
    if (b + 2 < len) issue(b + 2, st == 0 ? 2 : st - 1);
    const h16x8* bs = (const h16x8*)(lds + st * HS_BLOCK) + lane;
    f32x16 acc[2] = {};
    // operands and scales one step ahead
    h16x8 bh = bs[0], bl = bs[64];
    float rq[2] = {rh[0], rh[32]};
#pragma unroll
    for (int ks = 0; ks < HS_KS; ks++) {
      h16x8 nh = bh, nl = bl;
      float nq[2] = {rq[0], rq[1]};
      if (ks + 1 < HS_KS) {
        const int r = 8 * ((ks + 1) >> 2) + ((ks + 1) & 3);
        nh = bs[(ks + 1) * 128];
        nl = bs[(ks + 1) * 128 + 64];
        nq[0] = rh[r];
        nq[1] = rh[32 + r];
      }
      // the reads stay in front: left alone, the scheduler puts them after
      // the step's MFMAs, into the registers these have just read
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < 2; t++)
        acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al[t][ks], bh, acc[t], 0, 0, 0);
#pragma unroll
      for (int t = 0; t < 2; t++)
        acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[t][ks], bl, acc[t], 0, 0, 0);
#pragma unroll
      for (int t = 0; t < 2; t++)
        acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[t][ks], bh, acc[t], 0, 0, 0);
#pragma unroll
      for (int t = 0; t < 2; t++)
        state_add<false>(rs[t], ks, prev[t][ks], rq[t], pc, b0 + b - 1);
#pragma unroll
      for (int q = 0; q < 6; q++) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      bh = nh;
      bl = nl;
      rq[0] = nq[0];
      rq[1] = nq[1];
    }
    prev[0] = acc[0];
    prev[1] = acc[1];
    pc = cil[b * 32 + lr];
    st = st == 2 ? 0 : st + 1;
  }
  if (!rows) return;
#pragma unroll
  for (int t = 0; t < 2; t++) {
#pragma unroll
    for (int v = 0; v < 16; v++)
      state_add<false>(rs[t], v, prev[t][v], rh[32 * t + 8 * (v >> 2) + (v & 3)], pc,
                       b0 + len - 1);
    state_store<false>(rs[t], rw + 32 * t, m, row + 32 * t, slices, slice, part);
  }
  const uint64_t odd = __ballot(rw[lane] < 0.0f);
#pragma unroll 1
  for (int t = 0; t < 2 && row + 32 * t < m; t++)
    if ((unsigned)(odd >> (32 * t)) != 0)
      flagged_tile(x, m, w, n, bias, row + 32 * t, b0, len, rw + 32 * t, slices, slice, part);
}

// Up to HS_SMALL rows: a wave per (32 rows, column block), the block's operands
// straight into registers, all 32 loads of a lane in flight at once (24 rows:
// 7.5 us, for 19 MB of weight; the row tile form would keep one wave in eight).
__global__ __launch_bounds__(64) void head_split_small_kernel(const _Float16* __restrict__ xs,
                                                              const float* __restrict__ rsc, int m,
                                                              const _Float16* __restrict__ wp,
                                                              const float2* __restrict__ ci,
                                                              int nb, int tiles, int per_xcd,
                                                              float* __restrict__ part,
                                                              const float* __restrict__ x,
                                                              const float* __restrict__ w, int n,
                                                              const float* __restrict__ bias) {
  __shared__ float srl[32];
  const int u = (int)(blockIdx.x % 8) * per_xcd + (int)(blockIdx.x / 8);
  if (u >= tiles * nb) return;
  const int cb = u / tiles, row = (u - cb * tiles) * 32;
  const int lane = threadIdx.x;
  const h16x8* bs = (const h16x8*)wp + (int64_t)cb * (HS_BLOCK / 16) + lane;
  h16x8 bh[HS_KS], bl[HS_KS];
#pragma unroll
  for (int ks = 0; ks < HS_KS; ks++) {
    bh[ks] = bs[ks * 128];
    bl[ks] = bs[ks * 128 + 64];
  }
  const float2 c = ci[cb * 32 + (lane & 31)];
  h16x8 ah[HS_KS], al[HS_KS];
#pragma unroll
  for (int ks = 0; ks < HS_KS; ks++) load_rows(xs, row / 32, ks, ah[ks], al[ks]);
  if (lane < 32) srl[lane] = rsc[row + lane];
  __syncthreads();
  f32x16 acc = {};
#pragma unroll
  for (int ks = 0; ks < HS_KS; ks++) {
    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(al[ks], bh[ks], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[ks], bl[ks], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[ks], bh[ks], acc, 0, 0, 0);
  }
  RowState rs;
  state_init(rs);
#pragma unroll
  for (int v = 0; v < 16; v++)
    state_add<false>(rs, v, acc[v], srl[8 * (v >> 2) + 4 * (lane >> 5) + (v & 3)], c, cb);
  state_store<false>(rs, srl, m, row, nb, cb, part);
  if (__ballot(srl[lane & 31] < 0.0f) != 0)
    flagged_tile(x, m, w, n, bias, row, cb, 1, srl, nb, cb, part);
}

// Per row: the slices' partials to the (value, index) pair, one wave a row.  A
// flagged row's are in natural units, and its logits may have no maximum (nothing
// but -infinity and NaN: the id is 0x7fffffff) or an infinite one: its value is
// then 1 / 0, as the unsplit kernels give it.
__global__ __launch_bounds__(256) void head_split_pairs_kernel(const float* __restrict__ part,
                                                               int64_t rows, int slices,
                                                               float* __restrict__ pairs) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const f32x4* pr = (const f32x4*)part + row * slices;
  float m = -3.0e38f, sum = 0.0f, l2e = 1.0f;
  int idx = 0x7fffffff;
  for (int t = lane; t < slices; t += 64) {
    const f32x4 q = pr[t];
    l2e = q[3] != 0.0f ? HS_L2E : 1.0f;
    if (q[0] > m) {
      sum = sum * __builtin_amdgcn_exp2f((m - q[0]) * l2e) + q[2];
      m = q[0];
      idx = __float_as_int(q[1]);
    } else {
      sum += q[2] * __builtin_amdgcn_exp2f((q[0] - m) * l2e);
    }
  }
  l2e = __shfl(l2e, 0, 64);   // (a lane past the slices has not seen the flag)
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const float mo = __shfl_xor(m, off, 64);
    const int io = __shfl_xor(idx, off, 64);
    const float so = __shfl_xor(sum, off, 64);
    const float mm = fmaxf(m, mo);
    sum = sum * __builtin_amdgcn_exp2f((m - mm) * l2e) + so * __builtin_amdgcn_exp2f((mo - mm) * l2e);
    if (mo > m || (mo == m && io < idx)) idx = io;
    m = mm;
  }
  if (lane == 0) {
    // the max's exponential is exp2(0) = 1
    pairs[2 * row] = 1.0f / (m > -3.0e38f && m - m == 0.0f ? sum : 0.0f);
    pairs[2 * row + 1] = __int_as_float(idx);
  }
}

// Slices of the column blocks per row tile: the count with the least rounds of
// 256 workgroups (one a CU) times (blocks of a slice + 2: loading a tile's 256 KB
// of rows and closing its state take about two blocks' time), its scales
// within LDS.
static int split_slices(int tiles, int nb) {
  const int lo = (nb + HS_MAX_LEN - 1) / HS_MAX_LEN;
  int best = lo;
  int64_t cost = INT64_MAX;
  for (int s = lo; s <= nb && (s == lo || (int64_t)s * tiles <= 512); s++) {
    const int64_t c = (((int64_t)s * tiles + 255) / 256) * ((nb + s - 1) / s + 2);
    if (c < cost) {
      cost = c;
      best = s;
    }
  }
  return best;
}

bool head_split_eligible(int64_t k, int64_t n) { return k == HS_K && n > 0 && n <= (1 << 20); }

// Partials, at any row count up to m: few rows have a partial per column block,
// otherwise at most 512 workgroups (or the least slices there can be).
static int64_t part_floats(int64_t m, int64_t n) {
  const int64_t nb = ceil_div(n, 32);
  return 4 * std::max({std::min<int64_t>(m, HS_SMALL) * nb, (int64_t)512 * HS_ROWS,
                       (m + HS_ROWS - 1) * ceil_div(nb, HS_MAX_LEN)});
}

int64_t head_split_scratch_floats(int64_t m, int64_t n) {
  return part_floats(m, n) + ceil_div(m, 32) * 32 * (HS_K + 1);
}

// Packs w[256][n] (rows n apart); *out stays NULL for a weight or bias that
// cannot be split.  Waits for the stream.
int head_split_pack(const float* w, int64_t n, const float* bias, HeadSplit* out, hipStream_t s) {
  const int nb = (int)ceil_div(n, 32);
  char* d = nullptr;
  const size_t wb = (size_t)nb * HS_BLOCK, cb = (size_t)nb * 32 * sizeof(float2);
  QPH_TRY_HIP(hipMalloc((void**)&d, wb + cb + (size_t)nb * 4));
  float* top = (float*)(d + wb + cb);
  hipLaunchKernelGGL(head_pack_kernel, dim3((unsigned)nb), dim3(256), 0, s, w, (int)n, bias,
                     (_Float16*)d, (float2*)(d + wb), top);
  int rc = launch_check("head_pack_kernel");
  std::vector<float> f((size_t)nb, 0.0f);
  if (rc == QPH_OK)
    rc = hip_check(hipMemcpyAsync(f.data(), top, (size_t)nb * 4, hipMemcpyDeviceToHost, s),
                   "hipMemcpyAsync(head maxima)");
  if (rc == QPH_OK) rc = hip_check(hipStreamSynchronize(s), "hipStreamSynchronize");
  bool odd = false;
  for (float v : f) odd = odd || v < 0.0f, out->wmax = std::max(out->wmax, v);
  if (rc != QPH_OK || odd) {
    (void)hipFree(d);
    return rc;
  }
  out->wp = d;
  out->ci = (const float*)(d + wb);
  return QPH_OK;
}

int launch_head_split(const float* x, int64_t m, const HeadSplit& hs, const float* w, int64_t n,
                      const float* bias, float* scratch, float* pairs, hipStream_t s) {
  if ((uintptr_t)x % 16 != 0) return fail(QPH_EUNSUPPORTED, "fused head: A not 16-byte aligned");
  if (m <= 0 || m * HS_K >= (1ll << 31)) return fail(QPH_EUNSUPPORTED, "fused head: row count");
  const int nb = (int)ceil_div(n, 32), rt = (int)ceil_div(m, 32);
  const _Float16* wp = (const _Float16*)hs.wp;
  const float2* ci = (const float2*)hs.ci;
  // scratch: the split rows, their scales, the partials
  _Float16* xs = (_Float16*)scratch;
  float* rs = scratch + (int64_t)rt * 32 * HS_K;
  float* part = rs + (int64_t)rt * 32;
  hipLaunchKernelGGL(head_rows_kernel, dim3((unsigned)rt), dim3(256), 0, s, x, (int)m, hs.wmax, xs,
                     rs);
  QPH_TRY(launch_check("head_rows_kernel"));
  int slices = nb;
  if (m <= HS_SMALL) {
    const int per = (int)ceil_div((int64_t)rt * nb, 8);
    hipLaunchKernelGGL(head_split_small_kernel, dim3((unsigned)per * 8), dim3(64), 0, s, xs, rs,
                       (int)m, wp, ci, nb, rt, per, part, x, w, (int)n, bias);
    QPH_TRY(launch_check("head_split_small_kernel"));
  } else {
    const int tiles = (int)ceil_div(m, HS_ROWS);
    slices = split_slices(tiles, nb);
    const int len = (nb + slices - 1) / slices;
    const int per = (int)ceil_div((int64_t)tiles * slices, 8);
    const size_t shm = HS_STAGES * HS_BLOCK + HS_ROWS * sizeof(float) + (size_t)len * 32 * sizeof(float2);
    QPH_TRY(allow_full_lds((const void*)head_split_kernel));
    hipLaunchKernelGGL(head_split_kernel, dim3((unsigned)per * 8), dim3(256), shm, s, xs, rs,
                       (int)m, wp, ci, nb, tiles, slices, nb / slices, nb % slices, per, part, x, w,
                       (int)n, bias);
    QPH_TRY(launch_check("head_split_kernel"));
  }
  hipLaunchKernelGGL(head_split_pairs_kernel, dim3(ceil_div(m, 4)), dim3(256), 0, s, part, m,
                     slices, pairs);
  return launch_check("head_split_pairs_kernel");
}

}  // namespace qph
