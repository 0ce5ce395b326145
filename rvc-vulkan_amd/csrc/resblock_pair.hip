// One dilation group of a decoder ResBlock in one launch, on the split
// products of conv_split.hip:
//   out = x + conv2(lrelu(conv1(lrelu(x)) + b1)) + b2
// with K taps, conv1 at dilation d and conv2 at 1.  Up to three groups (the
// ResBlocks of a stage, K = 3, 7, 11) share a grid, heaviest first.
//
// Bound by the matrix cores where channels are many: at 128 they are busy 0.67 of
// the cycles at the 1.63 GHz the clock falls to (SQ counters), at 64 0.54, the
// rest being waits for operands, barriers and the two epilogues (2.5 and 4.3 VALU
// instructions an MFMA).  At 32 channels (0.41) HBM bounds it: 538 MB in 140 us,
// 0.8 of the card's copy rate.  Run as two launches the intermediate crosses HBM
// twice, and at 32 channels the second
// launch moved 444 MB in 104 us, the card's copy rate.  Here a workgroup owns
// all C channels of BN intermediate columns.  It forms them (the staging and
// main loop of conv1d_split_kernel), applies bias and leaky ReLU in registers,
// splits the result into LDS over the dead staging buffers,
//   ys[part][channel / 8][column],
// and forms conv2 from there without another barrier.  The BN columns serve
// BN - (K - 1) outputs: both convs compute (K - 1) / BN more than two launches
// would (4 % at K = 11, BN = 256).  Columns outside the signal are zero, as
// conv2's padding wants them.
//
// The input's scale is that of conv_split.hip, and so is the intermediate's,
// which is still in registers when its columns' largest values are known.  What
// the scales do not hold takes the fp32 matrix cores (fp32_sums): columns of
// the intermediate from x, and outputs whose intermediate columns do not fit
// from an fp32 intermediate, which has just the two parts' room in LDS.
//
// 40k, 1000 frames, ms of a stage's six convs, two launches -> fused: C = 128
// 1.20 -> 1.19 (half the launches), C = 64 0.78 -> 0.69, C = 32 0.60 -> 0.45
// (343 / 299 / 229 TFLOP/s of fp32 products).
//
// BF: the same on bf16 operands (x and the intermediate rounded to bf16 as
// they go to LDS, weights in bf16, chunks of 32 channels, one product); the
// matrix work is a third and LDS and HBM bound it.
//
// out and x must be different tensors: neighbouring tiles read x's halo.
#include <algorithm>
#include <type_traits>

#include "split.h"

namespace rvc {

namespace {

template <bool BF, int C, int BN, int WM, int WN>
__global__ __launch_bounds__((C / WM) * (BN / WN) * 64)
__attribute__((amdgpu_waves_per_eu(2)))
void resblock_pair_kernel(PairLaunch a) {
  constexpr int NWM = C / WM, NW = NWM * (BN / WN), NT = NW * 64;
  constexpr int TM = WM / 32, TN = WN / 32, NRB = C / 32;
  constexpr int CH = BF ? 32 : 16, XU = CH / 8;  // channels per chunk
  constexpr int XPT = (XU * (BN + kConvHaloMax) + NT - 1) / NT;
  constexpr int nchunk = C / CH, PARTS = BF ? 1 : 2;
  constexpr unsigned wpart = 1024u * NRB;
  constexpr int YS = BN + kConvTapsMax - 1;  // row length of an fp32 intermediate in LDS
  int gi = 0, lin = blockIdx.x;
  while (gi + 1 < a.n && lin >= a.g[gi].tiles * a.B) {
    lin -= a.g[gi].tiles * a.B;
    ++gi;
  }
  const PairGroup& G = a.g[gi];
  const int b = lin / G.tiles;
  const int K = G.K, dil = G.dil, L = a.L;
  const int BO = BN - (K - 1);
  const int o0 = (lin - b * G.tiles) * BO;  // first output column
  const int y0 = o0 - (K - 1) / 2;          // first intermediate column
  const int x0 = y0 - dil * ((K - 1) / 2);  // first input column
  const int XW = BN + (K - 1) * dil, YW = BN + (K - 1);

  extern __shared__ uint4 sm[];  // [2 buffers][2 parts][2][XW], then [2 parts][C / 8][YW]
  __shared__ float wmax[NW];
  __shared__ unsigned vote[3][NW];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave % NWM, wn = wave / NWM;
  const int half = lane >> 5, l32 = lane & 31;
  const int co_l = wm * WM + 4 * half;  // the lane's first row; row r: + m 32 + (r & 3) + 8 (r / 4)
  const float* xb = G.x + (long long)b * C * L;

  // ---- staging of x, as in conv1d_split_kernel
  unsigned xo[XPT];
  int xu[XPT];
#pragma unroll
  for (int e = 0; e < XPT; ++e) {
    const int u = tid + e * NT;
    int c8 = u >= XW;
    if constexpr (BF) c8 += (u >= 2 * XW) + (u >= 3 * XW);
    const int t = x0 + u - c8 * XW;
    xu[e] = u < XU * XW ? u : -1;
    xo[e] = u < XU * XW && t >= 0 && t < L ? 4u * (unsigned)(c8 * 8 * L + t) : kBufOut;
  }
  float xv[XPT][8];
  auto gload = [&](int c) {
    const __amdgpu_buffer_rsrc_t rs = uniform_rsrc(xb + (long long)c * CH * L, 4u * CH * (unsigned)L);
#pragma unroll
    for (int e = 0; e < XPT; ++e)
#pragma unroll
      for (int j = 0; j < 8; ++j) xv[e][j] = buf_load4(rs, xo[e], 4u * (unsigned)(j * L));
  };
  float sx = kScaleX, xm[XPT];  // each unit's largest magnitude, scaled
  auto lstore = [&](int buf) __attribute__((always_inline)) {
    uint4* xs = sm + buf * 4 * XW;
#pragma unroll
    for (int e = 0; e < XPT; ++e) {
      if (xu[e] < 0) continue;
      float v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = leaky(xv[e][j], a.slope);
      stage_unit<BF>(v, sx, xm[e], xs + xu[e], 2 * XW);
    }
  };
  const unsigned wvo = 16u * (unsigned)lane + 1024u * (unsigned)(wm * TM);
  const unsigned wbytes = (unsigned)(nchunk * K) * 2u * wpart;
  uint4 Ah[2][TM], Al[2][TM], Bh[TN], Bl[TN];  // the weights of the current step and of the next one
  auto lda = [&](uint4(&A)[TM], __amdgpu_buffer_rsrc_t rs, unsigned so) {
#pragma unroll
    for (int m = 0; m < TM; ++m) A[m] = buf_load16(rs, wvo + 1024u * m, so);
  };
  auto ldb = [&](uint4(&B)[TN], const uint4* p) {
#pragma unroll
    for (int n = 0; n < TN; ++n) B[n] = p[n * 32];
  };
  floatx16 acc[TM][TN];
  auto zero = [&] {
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
      for (int n = 0; n < TN; ++n)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[m][n][r] = 0.f;
  };
  auto prod = [&](const uint4(&A)[TM], const uint4(&B)[TN]) {
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
      for (int n = 0; n < TN; ++n)
        acc[m][n] = mma16<BF>(A[m], B[n], acc[m][n]);
  };
  // the first two steps' weights
  const unsigned last = wbytes - 2u * wpart;  // the last step's
  unsigned next = 0;
  auto first = [&](__amdgpu_buffer_rsrc_t rs) {
    next = min(2u * wpart, last);
    lda(Al[0], rs, wpart);
    lda(Ah[0], rs, 0);
    lda(Al[1], rs, next + wpart);
    lda(Ah[1], rs, next);
    next = min(next + 2 * wpart, last);
  };
  // one chunk's taps (an odd number): column operands at xh (part h) and xh + pl
  // (part l), tap k at column k * step.  Each tap loads the weights two steps on.
  auto taps = [&](__amdgpu_buffer_rsrc_t rs, const uint4* xh, int pl, int step) {
    ldb(Bh, xh);
    ldb(Bl, xh + pl);
    auto tap = [&](int k, uint4(&H)[TM], uint4(&Lo)[TM]) __attribute__((always_inline)) {
      xh += k + 1 < K ? step : 0;
      if constexpr (BF) {
        prod(H, Bh);
        lda(H, rs, next);
        ldb(Bh, xh);
        prod(Lo, Bl);
        lda(Lo, rs, next + wpart);
        ldb(Bl, xh + pl);
      } else {
        prod(Lo, Bh);
        lda(Lo, rs, next + wpart);
        prod(H, Bh);
        ldb(Bh, xh);
        prod(H, Bl);
        lda(H, rs, next);
        ldb(Bl, xh + pl);
      }
      next = min(next + 2 * wpart, last);
      sched_tap<BF, TM, TN>();
    };
    for (int k = 0; k + 1 < K; k += 2) {
      tap(k, Ah[0], Al[0]);
      tap(k + 1, Ah[1], Al[1]);
    }
    tap(K - 1, Ah[0], Al[0]);
    swap_sets(Ah, Al);
  };
  // sum * scale of its row * inv + bias (the scales are powers of two)
  auto finish = [&](const float* sc, float inv, const float* bias) {
    const __amdgpu_buffer_rsrc_t rs = uniform_rsrc(sc, BF ? 0u : 4u * C), rb = uniform_rsrc(bias, 4u * C);
#pragma unroll
    for (int m = 0; m < TM; ++m) {
      float s[16], t[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = 4 * (m * 32 + (r & 3) + 8 * (r >> 2));
        s[r] = BF ? 1.f : buf_load4(rs, 4u * (unsigned)co_l, row) * inv;
        t[r] = buf_load4(rb, 4u * (unsigned)co_l, row);
      }
#pragma unroll
      for (int n = 0; n < TN; ++n)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[m][n][r] = fmaf(acc[m][n][r], s[r], t[r]);
    }
  };
  // bit n: the lane's sums of column block n hold a NaN
  auto nan_bits = [&] {
    unsigned bits = 0;
#pragma unroll
    for (int n = 0; n < TN; ++n) {
      float nan = 0.f;
#pragma unroll
      for (int m = 0; m < TM; ++m)
#pragma unroll
        for (int r = 0; r < 16; ++r) nan = fmaf(acc[m][n][r], 0.f, nan);
      if (nan != nan) bits |= 1u << n;
    }
    return bits;
  };
  // bit n: the lane's column block n has a column among the K from p on, `step`
  // apart, whose largest magnitude (bits) the split does not hold at `scale`
  auto unfit_bits = [&](const unsigned* cm, int step, float scale) {
    unsigned bits = 0;
#pragma unroll
    for (int n = 0; n < TN; ++n) {
      const unsigned* p = cm + wn * WN + n * 32 + l32;
      unsigned t = 0;
      for (int k = 0; k < K; ++k) t = max(t, p[k * step]);
      if (!split_holds(__builtin_bit_cast(float, t) * scale)) bits |= 1u << n;
    }
    return bits;
  };
  // the lane's column blocks of `bits` again in fp32, from weights [K][C][C] and
  // x(B, k, c) (fp32_sums), and their bias; every lane of the wave calls it
  auto form_again = [&](unsigned bits, const float* w, const float* bias, auto x) {
    floatx16 f[TM][TN];
    const __amdgpu_buffer_rsrc_t rs = uniform_rsrc(w, 4u * (unsigned)(K * C * C)), rb = uniform_rsrc(bias, 4u * C);
    const unsigned fo = 4u * (unsigned)(half * C + wm * WM + l32);
    fp32_sums(
        f, C, K,
        [&](float(&A)[TM], int k, int c) {
#pragma unroll
          for (int m = 0; m < TM; ++m) A[m] = buf_load4(rs, fo + 128u * m, 4u * (unsigned)((k * C + c) * C));
        },
        x);
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float t = buf_load4(rb, 4u * (unsigned)co_l, 4 * (m * 32 + (r & 3) + 8 * (r >> 2)));
#pragma unroll
        for (int n = 0; n < TN; ++n) acc[m][n][r] = bits >> n & 1u ? f[m][n][r] + t : acc[m][n][r];
      }
  };
  // outputs of the lane's column blocks of `bits`, with the residual
  const int cols = min(BO, L - o0);
  auto store = [&](unsigned bits) {
    const __amdgpu_buffer_rsrc_t rrs = uniform_rsrc(xb, 4u * (unsigned)(C * L));
    const __amdgpu_buffer_rsrc_t ors = uniform_rsrc(G.out + (long long)b * C * L, 4u * (unsigned)(C * L));
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
      for (int n = 0; n < TN; ++n) {
        const int col = wn * WN + n * 32 + l32;
        const unsigned oo = col < cols && (bits >> n & 1u) ? 4u * (unsigned)(co_l * L + o0 + col) : kBufOut;
        float pre[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) pre[r] = buf_load4(rrs, oo, 4 * (m * 32 + (r & 3) + 8 * (r >> 2)) * L);
#pragma unroll
        for (int r = 0; r < 16; ++r)
          __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, acc[m][n][r] + pre[r]), ors, oo,
                                                4 * (m * 32 + (r & 3) + 8 * (r >> 2)) * L, 0);
      }
  };

  // ---- conv1 over the BN intermediate columns
  const __amdgpu_buffer_rsrc_t w1 = uniform_rsrc(G.w1.w, wbytes);
  bool mixed = false;  // some units lie outside the split's range
  for (bool again = false;; again = true) {
    zero();
#pragma unroll
    for (int e = 0; e < XPT; ++e) xm[e] = 0.f;
    gload(0);
    first(w1);
    lstore(0);
    __syncthreads();
    for (int c = 0; c < nchunk; ++c) {
      const bool more = c + 1 < nchunk;
      if (more) gload(c + 1);
      taps(w1, sm + (c & 1) * 4 * XW + half * XW + wn * WN + l32, 2 * XW, dil);
      if (more) lstore((c & 1) ^ 1);
      __syncthreads();
    }
    if (BF) break;
    float top;
    const unsigned f = block_or<NW>(range_bits(xm, 1.f, top), vote[0]);
    mixed = f & 1u;
    if (!mixed || again || (f & 2u)) break;
    top = block_max<NW>(top, wmax);
    if (top == 0.f) break;  // infinities and zeros
    sx = pow2_scale(top * (1.f / kScaleX));
  }
  unsigned bad = 0;  // the lane's intermediate columns that the split does not hold
  if constexpr (!BF) {
    if (mixed) {
      unsigned* cm = reinterpret_cast<unsigned*>(sm);  // a column's largest magnitude; every wave is past its operands
      for (int u = tid; u < XW; u += NT) cm[u] = 0u;
      __syncthreads();
#pragma unroll
      for (int e = 0; e < XPT; ++e)
        if (xu[e] >= 0) atomicMax(cm + (xu[e] < XW ? xu[e] : xu[e] - XW), __builtin_bit_cast(unsigned, xm[e]));
      __syncthreads();
      bad = unfit_bits(cm, dil, 1.f);
      __syncthreads();  // the room is free again
    }
    bad |= nan_bits();
  }
  finish(G.w1.sc, 1.f / sx, G.b1);
  const bool again1 = __any(bad != 0u);
  if (again1)
    form_again(bad, G.f1, G.b1, [&](float(&B)[TN], int k, int c) {
      const __amdgpu_buffer_rsrc_t rs = uniform_rsrc(xb + (long long)c * L, 8u * (unsigned)L);
#pragma unroll
      for (int n = 0; n < TN; ++n) {
        const int t = x0 + wn * WN + n * 32 + l32 + k * dil;
        B[n] = leaky_mma(buf_load4(rs, t >= 0 && t < L ? 4u * (unsigned)(half * L + t) : kBufOut, 0), a.slope);
      }
    });

  // ---- leaky ReLU, zero outside the signal, scale, split to LDS
  float ym[TN];
#pragma unroll
  for (int n = 0; n < TN; ++n) {
    const int t = y0 + wn * WN + n * 32 + l32;
    const bool in = t >= 0 && t < L;
    ym[n] = 0.f;
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
      for (int r = 0; r < 16; r += 2) {
        const float u = in ? leaky(acc[m][n][r], a.slope) : 0.f;
        const float v = in ? leaky(acc[m][n][r + 1], a.slope) : 0.f;
        if constexpr (!BF) ym[n] = max3_abs(ym[n], u, v);
        acc[m][n][r] = u;
        acc[m][n][r + 1] = v;
      }
  }
  float sy = kScaleX;
  unsigned done = 0;  // the lane's column blocks whose outputs are stored already
  if constexpr (!BF) {
    float top;
    const unsigned has_nan = again1 && nan_bits() ? 1u : 0u;
    unsigned f = block_or<NW>(range_bits(ym, sy, top) | has_nan, vote[1]);
    if ((f & 3u) == 1u) {
      top = block_max<NW>(top, wmax);
      if (top > 0.f) {
        sy = pow2_scale(top);
        f = block_or<NW>(range_bits(ym, sy, top) | has_nan, vote[2]);
      }
    }
    if (f & 1u) {
      // the outputs whose own columns of the intermediate do not fit
      unsigned* cm = reinterpret_cast<unsigned*>(sm);
      for (int u = tid; u < YW; u += NT) cm[u] = 0u;
      __syncthreads();
#pragma unroll
      for (int n = 0; n < TN; ++n) {
        unsigned t = 0;
#pragma unroll
        for (int m = 0; m < TM; ++m)
#pragma unroll
          for (int r = 0; r < 16; ++r) t = max(t, __builtin_bit_cast(unsigned, acc[m][n][r]) & 0x7fffffffu);
        atomicMax(cm + wn * WN + n * 32 + l32, t);
      }
      __syncthreads();
      done = unfit_bits(cm, 1, sy);
#pragma unroll
      for (int n = 0; n < TN; ++n)
        if (wn * WN + n * 32 + l32 >= cols) done &= ~(1u << n);
      if (block_or<NW>(done ? 1u : 0u, vote[0])) {
        float* yf = reinterpret_cast<float*>(sm);  // [C][YS]
#pragma unroll
        for (int m = 0; m < TM; ++m)
#pragma unroll
          for (int n = 0; n < TN; ++n)
#pragma unroll
            for (int r = 0; r < 16; ++r)
              yf[(co_l + m * 32 + (r & 3) + 8 * (r >> 2)) * YS + wn * WN + n * 32 + l32] = acc[m][n][r];
        for (int u = tid; u < C * (K - 1); u += NT) {
          const int row = u / (K - 1);
          yf[row * YS + BN + u - row * (K - 1)] = 0.f;
        }
        __syncthreads();
        if (__any(done != 0u)) {
          form_again(done, G.f2, G.b2, [&](float(&B)[TN], int k, int c) {
#pragma unroll
            for (int n = 0; n < TN; ++n) B[n] = yf[(c + half) * YS + wn * WN + n * 32 + l32 + k];
          });
          store(done);
        }
#pragma unroll
        for (int m = 0; m < TM; ++m)
#pragma unroll
          for (int n = 0; n < TN; ++n)
#pragma unroll
            for (int r = 0; r < 16; ++r)
              acc[m][n][r] = yf[(co_l + m * 32 + (r & 3) + 8 * (r >> 2)) * YS + wn * WN + n * 32 + l32];
      }
      __syncthreads();  // the room is free again
    }
  }
  first(uniform_rsrc(G.w2.w, wbytes));
  uint2* ys = reinterpret_cast<uint2*>(sm);  // [part][C / 8][YW][half]
#pragma unroll
  for (int m = 0; m < TM; ++m)
#pragma unroll
    for (int n = 0; n < TN; ++n)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int at = ((wm * WM + m * 32) / 8 + q) * YW + wn * WN + n * 32 + l32;
        if constexpr (BF) {
          ys[2 * at + half] = make_uint2(pk_bf16(acc[m][n][4 * q], acc[m][n][4 * q + 1]),
                                         pk_bf16(acc[m][n][4 * q + 2], acc[m][n][4 * q + 3]));
        } else {
          uint2 h, l;
          split2(acc[m][n][4 * q] * sy, acc[m][n][4 * q + 1] * sy, h.x, l.x);
          split2(acc[m][n][4 * q + 2] * sy, acc[m][n][4 * q + 3] * sy, h.y, l.y);
          ys[2 * at + half] = h;
          ys[2 * (at + (C / 8) * YW) + half] = l;
        }
      }
  // the columns past BN, which only outputs past BO read
  for (int u = tid; u < PARTS * (C / 8) * (K - 1); u += NT) {
    const int row = u / (K - 1);
    sm[row * YW + BN + u - row * (K - 1)] = make_uint4(0u, 0u, 0u, 0u);
  }
  __syncthreads();

  // ---- conv2 over BN columns, the first BO of them outputs
  const __amdgpu_buffer_rsrc_t w2 = uniform_rsrc(G.w2.w, wbytes);
  zero();
#pragma unroll 1
  for (int c = 0; c < nchunk; ++c)
    taps(w2, sm + (XU * c + half) * YW + wn * WN + l32, BF ? 2 * YW : (C / 8) * YW, 1);
  unsigned nan2 = 0;  // NaN sums of fitting columns: the weights'
  if constexpr (!BF) {
    nan2 = nan_bits() & ~done;
#pragma unroll
    for (int n = 0; n < TN; ++n)
      if (wn * WN + n * 32 + l32 >= cols) nan2 &= ~(1u << n);
  }
  finish(G.w2.sc, 1.f / sy, G.b2);
  if (__any(nan2 != 0u)) {
    const float inv = 1.f / sy;
    form_again(nan2, G.f2, G.b2, [&](float(&B)[TN], int k, int c) {
      const int ci = c + half;
#pragma unroll
      for (int n = 0; n < TN; ++n) {
        const int col = wn * WN + n * 32 + l32 + k;
        const _Float16* p = reinterpret_cast<const _Float16*>(sm + (ci / 8) * YW + col) + ci % 8;
        B[n] = ((float)p[0] + (float)p[(C / 8) * YW * 8]) * inv;
      }
    });
  }
  store(~done);
}

template <bool BF, int C, int BN, int WM, int WN>
void launch_p(PairLaunch a, hipStream_t s) {
  constexpr int NT = (C / WM) * (BN / WN) * 64;
  size_t units = 0;
  long long items = 0;
  for (int g = 0; g < a.n; ++g) {
    const int K = a.g[g].K;
    units = std::max(units, (size_t)std::max(8 * (BN + (K - 1) * a.g[g].dil), BF ? C / 8 * (BN + K - 1) : C / 4 * (BN + kConvTapsMax - 1)));
    a.g[g].tiles = (a.L + BN - K) / (BN - K + 1);
    items += (long long)a.g[g].tiles * a.B;
  }
  RVC_CHECK(items < (1LL << 30), "resblock_pair: launch too large");
  const size_t lds = units * sizeof(uint4);
  constexpr size_t kMax = sizeof(uint4) * (size_t)std::max(8 * (BN + kConvHaloMax), C / (BF ? 8 : 4) * (BN + kConvTapsMax - 1));
  static_assert(kMax <= 160 * 1024, "LDS of one workgroup");
  if constexpr (kMax > 65536) {
    static bool attr = false;  // per instantiation
    if (!attr) {
      RVC_HIP(hipFuncSetAttribute((const void*)resblock_pair_kernel<BF, C, BN, WM, WN>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMax));
      attr = true;
    }
  }
  launch_timed(resblock_pair_kernel<BF, C, BN, WM, WN>, dim3((unsigned)items), dim3(NT), lds, s, a);
  check_launch("resblock_pair");
}

}  // namespace

bool resblock_pair_ok(int C, int L, float slope) {
  return (C == 32 || C == 64 || C == 128) && slope >= 0.f && slope <= 1.f && 4.0 * C * L < 2147483648.0;
}

void launch_resblock_pair(const PairLaunch& a, hipStream_t s) {
  RVC_CHECK(resblock_pair_ok(a.C, a.L, a.slope) && a.n >= 1 && a.n <= 3 && a.B >= 1, "resblock_pair: unsupported shape");
  for (int g = 0; g < a.n; ++g) {
    const PairGroup& G = a.g[g];
    RVC_CHECK(G.K % 2 == 1 && conv1d_mfma_supported(G.K, G.dil) && G.x != G.out && G.w1.w && G.w2.w && G.b1 && G.b2,
              "resblock_pair: unsupported group");
  }
  if (a.L < 1) return;
  // The widest tile that leaves one batch item 400 workgroups (of 256 CUs, two
  // to four resident on each); never by B, so that a batch equals its items
  // bit for bit also where a tile's own scale shows.  At 1000 frames of the
  // 40k model (stages 1 / 2 / 3): 1.19 / 0.69 / 0.45 ms with these tiles;
  // 64 x 256 columns on four 32 x 128 waves 0.73, 64 x 128 0.70, 32 x 512 0.53,
  // 32 x 128 0.51, 128 x 128 on 64 x 64 waves 1.22.  At 60 frames, a limit of
  // 128 instead: 0.224 / 0.112 / 0.068 against 0.183 / 0.096 / 0.062 ms.
  // tiles of one batch item
  auto wide = [&](int BN) {
    long long n = 0;
    for (int g = 0; g < a.n; ++g) n += (a.L + BN - a.g[g].K) / (BN - a.g[g].K + 1);
    return n >= 400;
  };
  if (!a.g[0].w1.sc) {
    // batch of 4 x 1000 frames, ms of stages 1 / 2 / 3 (one-shot bf16 tiles: 6.9
    // / 3.7 / 1.8): these 1.97 / 1.48 / 1.21; 128 x 128 on 64 x 64 waves 2.18,
    // 64 x 256 on 64 x 64 waves 1.53, 32 x 256 1.31
    if (a.C == 32) {
      if (wide(512)) return launch_p<true, 32, 512, 32, 64>(a, s);
      if (wide(256)) return launch_p<true, 32, 256, 32, 64>(a, s);
      if (wide(128)) return launch_p<true, 32, 128, 32, 32>(a, s);
      return launch_p<true, 32, 64, 32, 32>(a, s);
    }
    if (a.C == 64) {
      if (wide(256)) return launch_p<true, 64, 256, 32, 128>(a, s);
      if (wide(128)) return launch_p<true, 64, 128, 32, 64>(a, s);
      return launch_p<true, 64, 64, 32, 32>(a, s);
    }
    if (wide(256)) return launch_p<true, 128, 256, 64, 128>(a, s);
    if (wide(128)) return launch_p<true, 128, 128, 64, 64>(a, s);
    return launch_p<true, 128, 64, 32, 64>(a, s);
  }
  if (a.C == 32) {
    if (wide(256)) return launch_p<false, 32, 256, 32, 64>(a, s);
    if (wide(128)) return launch_p<false, 32, 128, 32, 32>(a, s);
    launch_p<false, 32, 64, 32, 32>(a, s);
  } else if (a.C == 64) {
    if (wide(256)) return launch_p<false, 64, 256, 32, 64>(a, s);
    if (wide(128)) return launch_p<false, 64, 128, 32, 64>(a, s);
    launch_p<false, 64, 64, 32, 32>(a, s);
  } else {
    if (wide(128)) return launch_p<false, 128, 128, 32, 128>(a, s);
    launch_p<false, 128, 64, 32, 64>(a, s);
  }
}

}  // namespace rvc
