// fp32 conv1d on the fp16 matrix cores: every operand split into two fp16
// parts, three products, fp32 accumulation.
//
// Two fp16 values hold 23 of a float's 24 significant bits and, three times in
// four, all of them: x = h + l with h = fp16(x), l = fp16(x - h), x - h exact,
// |x - h - l| <= 2^-23 |x|.  Then
//   w x = wh xh + wh xl + wl xh   (wl xl <= 2^-22 |w x| left out),
// each product exact in fp32.  The two errors are random in sign and stay, with
// the additions of one v_mfma_f32_32x32x16_f16 per 16 channels and product,
// below the rounding of an fp32 convolution's own additions, of which there
// are 2.7 times as many: whole waveforms against 64 bits, fp32 matrix cores ->
// here, 1 s at 40k 2.3e-6 -> 1.4e-6, 10 s 1.7e-6 -> 1.4e-6, 48k decoder 1.5e-6
// -> 1.3e-6.  The instruction does 16 times the multiply-adds per cycle of
// v_mfma_f32_32x32x2_f32; three products leave a factor of 16 / 3.  Under them
// the clock falls to 1.63 GHz, where matrix cores that never paused would do
// 1710 TFLOP/s, 570 of fp32 products (a loop of nothing but these instructions
// holds 1700).  The 256-channel launches at 10 000 columns keep them busy 0.57
// of the cycles (SQ counters), the rest being waits for operands and barriers:
// 320 TFLOP/s.  (Three bf16 parts, six products: the same
// launches at 190 - 220 TFLOP/s of fp32 products, error 1.6e-6.)
//
// Range: weights are scaled per output row to a largest value in [2^9, 2^10),
// inputs by 2^6, all exactly (powers of two).  At that scale the two parts hold
// a column whose largest input, of all channels and taps, is in [2^-6, 2^9.9]: a
// smaller one loses bits to fp16's subnormals, a larger one overflows.  A
// workgroup keeps the largest magnitude of each unit of 8 channels and a column
// that it stages.  Where none of them fits, it forms the tile again with the
// power of two that puts the largest into [2^14, 2^15); where some do, it looks
// at each output's own columns, and those that do not fit (an infinity among
// them, or a NaN among the sums) are formed on the fp32 matrix cores from the
// fp32 weights (fp32_sums), which gives what an fp32 convolution gives.  So an
// output has fp32's precision and reach whatever else is in its tile, as far
// as its inputs go.  Within an output's own inputs, channels or taps far below
// the largest keep 2^-31 absolute, and weights 2^-34 of their row's largest:
// where small inputs meet large weights and large inputs small ones, the error
// is the fp32 matrix cores' up to a spread of 2^10 between channels and
// grows with it from there (a ResBlock whose intermediate channels spread over
// 2^10 / 2^14 / 2^18, the next conv's weights making up for it: 2.2e-7 / 1.4e-6
// / 1.9e-5, fp32 2.1e-7).
//
// One workgroup forms a BM x BN tile, wave (wm, wn) a WM x WN part of it, over
// chunks of 16 input channels.  A chunk's input window (BN + (K - 1) dil
// columns) goes to LDS once, split on the way, for every tap:
//   xs[part][channel / 8][column] in units of 8 channels (16 bytes),
// so staging stores and operand reads are both 16 consecutive bytes per lane
// at consecutive columns (no bank conflicts, no padding).  The weights are
// split when they are packed, in MFMA operand order
//   wsp[chunk][tap][part][C_out / 32][lane][8],
// and go from L2 straight into registers: the waves of a workgroup that share
// rows read the same lines.
//
// S = 2: input stride 2 (HuBERT's feature extractor).  The window's even and
// odd columns lie apart in LDS, so that a tap's operand is again consecutive.
//
// BF: the same kernel on plain bf16 operands, for the mode that asks for bf16
// ResBlocks: chunks of 32 channels whose two halves of 16 take the place of the
// two parts, one product each, no scales.
//
// The order of an output's additions is (chunk, tap, product), whatever the
// tile, so the tile may follow the grid size and the batch.
#include <algorithm>
#include <type_traits>

#include "split.h"

namespace rvc {

namespace {

template <bool BF, int BM, int BN, int WM, int WN, int S>
struct CfgS {
  static constexpr int NWM = BM / WM;
  static constexpr int NWN = BN / WN;
  static constexpr int NW = NWM * NWN;
  static constexpr int NT = NW * 64;
  static constexpr int TM = WM / 32;
  static constexpr int TN = WN / 32;
  static constexpr int CH = BF ? 32 : 16;  // channels per chunk
  static constexpr int XU = CH / 8;
  static constexpr int XPT = (XU * (S == 2 ? 2 * (BN + 1) : BN + kConvHaloMax) + NT - 1) / NT;  // 8-channel units per thread and chunk
};

template <bool BF, int BM, int BN, int WM, int WN, int S>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * 64)
__attribute__((amdgpu_waves_per_eu(2)))
void conv1d_split_kernel(ConvLaunch a, int n_tx, int n_ty) {
  using C = CfgS<BF, BM, BN, WM, WN, S>;
  constexpr int NT = C::NT, TM = C::TM, TN = C::TN, XPT = C::XPT, XU = C::XU, CH = C::CH;
  const int per_b = n_tx * n_ty;
  const int per_group = per_b * a.B;
  const int gi = blockIdx.x / per_group;
  int lin = blockIdx.x - gi * per_group;
  const int b = lin / per_b;
  lin -= b * per_b;
  // the C_out tiles of one column tile 8 workgroups apart: on one XCD, whose
  // L2 then holds their input window
  int tx = lin, ty = 0;
  if (n_ty > 1) {
    const int full = (n_tx / 8) * 8 * n_ty;
    if (lin < full) {
      tx = (lin / (8 * n_ty)) * 8 + lin % 8;
      ty = (lin / 8) % n_ty;
    } else {
      tx = (n_tx / 8) * 8 + (lin - full) / n_ty;
      ty = (lin - full) % n_ty;
    }
  }
  const ConvGroup& G = a.g[gi];
  const int K = G.K, dil = G.dil, n_out = G.n_out;
  const int i0 = tx * BN, co0 = ty * BM;
  if (i0 >= n_out) return;  // uniform, before any barrier
  const int XW = S == 2 ? 2 * (BN + 1) : BN + (K - 1) * dil;
  const int nchunk = a.C_in / CH;

  extern __shared__ uint4 sm[];  // [2 buffers][2][2][XW]
  __shared__ float wmax[C::NW];
  __shared__ unsigned vote[C::NW];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave % C::NWM, wn = wave / C::NWM;
  const int half = lane >> 5, l32 = lane & 31;

  // ---- staging: unit u = (channel group u / XW, column u % XW) of a chunk
  const float* xb = G.x + (long long)b * a.xb;
  const unsigned xrow = 4u * (unsigned)a.xc;
  unsigned xo[XPT];
  int xu[XPT];
#pragma unroll
  for (int e = 0; e < XPT; ++e) {
    const int u = tid + e * NT;
    int c8 = u >= XW;
    if constexpr (BF) c8 += (u >= 2 * XW) + (u >= 3 * XW);
    const int p = u - c8 * XW;
    const int t = i0 * S + G.in_off + p;
    xu[e] = u < XU * XW ? (S == 2 ? c8 * XW + (p & 1) * (BN + 1) + (p >> 1) : u) : -1;
    xo[e] = u < XU * XW && t >= 0 && t < a.L_in ? 4u * (unsigned)(c8 * 8 * (int)a.xc + t) : kBufOut;
  }
  float xv[XPT][8];
  auto gload = [&](int c) {
    const __amdgpu_buffer_rsrc_t rs =
        uniform_rsrc(xb + (long long)c * CH * a.xc, 4u * (unsigned)((CH - 1) * (int)a.xc + a.L_in));
#pragma unroll
    for (int e = 0; e < XPT; ++e)
#pragma unroll
      for (int j = 0; j < 8; ++j) xv[e][j] = buf_load4(rs, xo[e], j * xrow);
  };
  float sx = kScaleX, xm[XPT];  // each unit's largest magnitude, scaled
  auto lstore_as = [&](int buf, auto act) __attribute__((always_inline)) {
    uint4* xs = sm + buf * 4 * XW;
#pragma unroll
    for (int e = 0; e < XPT; ++e) {
      if (xu[e] < 0) continue;
      float v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = decltype(act)::value ? leaky(xv[e][j], a.in_slope) : xv[e][j];
      stage_unit<BF>(v, sx, xm[e], xs + xu[e], 2 * XW);
    }
  };
  auto lstore = [&](int buf) __attribute__((always_inline)) {
    if (a.in_act == ACT_LEAKY)
      lstore_as(buf, std::true_type{});
    else
      lstore_as(buf, std::false_type{});
  };

  // ---- weights: part p of step (chunk c, tap k) at ((c K + k) 2 + p) nrb KiB
  const int nrb = a.C_out / 32;
  const __amdgpu_buffer_rsrc_t wrs = uniform_rsrc(G.wsp, (unsigned)(nchunk * K * 2 * nrb) * 1024u);
  const unsigned wvo = 16u * (unsigned)lane + 1024u * (unsigned)(co0 / 32 + wm * TM);
  const unsigned wpart = 1024u * (unsigned)nrb;
  uint4 Ah[2][TM], Al[2][TM];  // the current step's and the next one's
  auto lda = [&](uint4(&A)[TM], unsigned so) {
#pragma unroll
    for (int m = 0; m < TM; ++m) A[m] = buf_load16(wrs, wvo + 1024u * m, so);
  };

  floatx16 acc[TM][TN];
  auto prod = [&](const uint4(&A)[TM], const uint4(&B)[TN]) {
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
      for (int n = 0; n < TN; ++n)
        acc[m][n] = mma16<BF>(A[m], B[n], acc[m][n]);
  };

  bool mixed = false;  // some units lie outside the split's range
  for (bool again = false;; again = true) {
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
      for (int n = 0; n < TN; ++n)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[m][n][r] = 0.f;
#pragma unroll
    for (int e = 0; e < XPT; ++e) xm[e] = 0.f;
    gload(0);
    // last: the last step's weights; next: the ones to load
    const unsigned last = (unsigned)(nchunk * K - 1) * 2u * wpart;
    unsigned next = min(2u * wpart, last);
    lda(Al[0], wpart);
    lda(Ah[0], 0);
    lda(Al[1], next + wpart);
    lda(Ah[1], next);
    next = min(next + 2 * wpart, last);
    lstore(0);
    __syncthreads();
    for (int c = 0; c < nchunk; ++c) {
      const bool more = c + 1 < nchunk;
      if (more) gload(c + 1);
      const uint4* xh = sm + (c & 1) * 4 * XW + half * XW + wn * WN + l32;
      uint4 Bh[TN], Bl[TN];
      auto ldb = [&](uint4(&B)[TN], const uint4* p) {
#pragma unroll
        for (int n = 0; n < TN; ++n) B[n] = p[n * 32];
      };
      ldb(Bh, xh);
      ldb(Bl, xh + 2 * XW);
      // one tap: its products, the weights two steps on, the next tap's columns
      // (the last tap of a chunk reads its own again: the next chunk is behind
      // the barrier)
      auto tap = [&](int k, uint4(&H)[TM], uint4(&Lo)[TM]) __attribute__((always_inline)) {
        if constexpr (S == 2)
          xh += k + 1 < K ? ((k & 1) ? -BN : BN + 1) : 0;
        else
          xh += k + 1 < K ? dil : 0;
        if constexpr (BF) {
          prod(H, Bh);
          lda(H, next);
          ldb(Bh, xh);
          prod(Lo, Bl);
          lda(Lo, next + wpart);
          ldb(Bl, xh + 2 * XW);
        } else {
          prod(Lo, Bh);
          lda(Lo, next + wpart);
          prod(H, Bh);
          ldb(Bh, xh);
          prod(H, Bl);
          lda(H, next);
          ldb(Bl, xh + 2 * XW);
        }
        next = min(next + 2 * wpart, last);
        sched_tap<BF, TM, TN>();
      };
      int k = 0;
      for (; k + 1 < K; k += 2) {
        tap(k, Ah[0], Al[0]);
        tap(k + 1, Ah[1], Al[1]);
      }
      if (k < K) {
        tap(k, Ah[0], Al[0]);
        swap_sets(Ah, Al);
      }
      if (more) lstore((c & 1) ^ 1);
      __syncthreads();
    }
    if (BF) break;
    float top;
    const unsigned f = block_or<C::NW>(range_bits(xm, 1.f, top), vote);
    mixed = f & 1u;
    if (!mixed || again || (f & 2u)) break;
    top = block_max<C::NW>(top, wmax);
    if (top == 0.f) break;  // infinities and zeros
    sx = pow2_scale(top * (1.f / kScaleX));
  }

  const int co_l = co0 + wm * WM + 4 * half;
  if constexpr (!BF) {
    // ---- the lane's columns that the split does not hold (bit n)
    unsigned bad = 0;
    if (mixed) {
      unsigned* cm = reinterpret_cast<unsigned*>(sm);  // a column's largest magnitude; every wave is past its operands
      for (int u = tid; u < XW; u += NT) cm[u] = 0u;
      __syncthreads();
#pragma unroll
      for (int e = 0; e < XPT; ++e)
        if (xu[e] >= 0) atomicMax(cm + (xu[e] < XW ? xu[e] : xu[e] - XW), __builtin_bit_cast(unsigned, xm[e]));
      __syncthreads();
#pragma unroll
      for (int n = 0; n < TN; ++n) {
        const unsigned* p = cm + wn * WN + n * 32 + l32;
        unsigned t = 0;
        for (int k = 0; k < K; ++k) {
          t = max(t, *p);
          if (k + 1 < K) p += S == 2 ? ((k & 1) ? -BN : BN + 1) : dil;
        }
        if (!split_holds(__builtin_bit_cast(float, t))) bad |= 1u << n;
      }
    }
#pragma unroll
    for (int n = 0; n < TN; ++n) {
      float nan = 0.f;
#pragma unroll
      for (int m = 0; m < TM; ++m)
#pragma unroll
        for (int r = 0; r < 16; ++r) nan = fmaf(acc[m][n][r], 0.f, nan);
      if (nan != nan) bad |= 1u << n;
      if (i0 + wn * WN + n * 32 + l32 >= n_out) bad &= ~(1u << n);
    }
    const __amdgpu_buffer_rsrc_t srs = uniform_rsrc(G.wsc, 4u * (unsigned)a.C_out);
    const float inv = 1.f / sx;
#pragma unroll
    for (int m = 0; m < TM; ++m) {
      float sc[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) sc[r] = buf_load4(srs, 4u * (unsigned)co_l, 4 * (m * 32 + (r & 3) + 8 * (r >> 2)));
#pragma unroll
      for (int n = 0; n < TN; ++n)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[m][n][r] = acc[m][n][r] * (sc[r] * inv);
    }
    if (__any(bad != 0u)) {
      floatx16 f[TM][TN];
      const __amdgpu_buffer_rsrc_t frs = uniform_rsrc(G.w, 4u * (unsigned)(K * a.C_in * a.w_ld));
      const unsigned fo = 4u * (unsigned)(half * a.w_ld + co0 + wm * WM + l32);
      fp32_sums(
          f, a.C_in, K,
          [&](float(&A)[TM], int k, int c) {
#pragma unroll
            for (int m = 0; m < TM; ++m) A[m] = buf_load4(frs, fo + 128u * m, 4u * (unsigned)((k * a.C_in + c) * a.w_ld));
          },
          [&](float(&B)[TN], int k, int c) {
            const __amdgpu_buffer_rsrc_t rs = uniform_rsrc(xb + (long long)c * a.xc, 4u * (unsigned)((int)a.xc + a.L_in));
#pragma unroll
            for (int n = 0; n < TN; ++n) {
              const int t = (i0 + wn * WN + n * 32 + l32) * S + G.in_off + k * dil;
              const float v = buf_load4(rs, t >= 0 && t < a.L_in ? 4u * (unsigned)(half * (int)a.xc + t) : kBufOut, 0);
              B[n] = a.in_act == ACT_LEAKY ? leaky_mma(v, a.in_slope) : v;
            }
          });
#pragma unroll
      for (int m = 0; m < TM; ++m)
#pragma unroll
        for (int n = 0; n < TN; ++n)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[m][n][r] = bad >> n & 1u ? f[m][n][r] : acc[m][n][r];
    }
  }

  // ---- (sum + bias) + residual, activation, store
  const __amdgpu_buffer_rsrc_t ors =
      uniform_rsrc(G.out + (long long)b * a.ob, 4u * (unsigned)((a.C_out - 1) * (int)a.oc + n_out));
  const __amdgpu_buffer_rsrc_t brs = uniform_rsrc(G.bias, G.bias ? 4u * (unsigned)a.C_out : 0u);
  const bool res = G.res != nullptr;
  const __amdgpu_buffer_rsrc_t rrs = uniform_rsrc(
      res ? G.res + (long long)b * a.rb : nullptr, res ? 4u * (unsigned)((a.C_out - 1) * (int)a.rc + n_out) : 0u);
#pragma unroll
  for (int m = 0; m < TM; ++m) {
    float bias[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) bias[r] = buf_load4(brs, 4u * (unsigned)co_l, 4 * (m * 32 + (r & 3) + 8 * (r >> 2)));
#pragma unroll
    for (int n = 0; n < TN; ++n) {
      const int i = i0 + wn * WN + n * 32 + l32;
      const unsigned oo = i < n_out ? 4u * (unsigned)(co_l * (int)a.oc + i) : kBufOut;
      if (res) {
        const unsigned ro = i < n_out ? 4u * (unsigned)(co_l * (int)a.rc + i) : kBufOut;
        float pre[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) pre[r] = buf_load4(rrs, ro, 4 * (m * 32 + (r & 3) + 8 * (r >> 2)) * (int)a.rc);
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[m][n][r] = (acc[m][n][r] + bias[r]) + pre[r];
      } else {
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[m][n][r] = acc[m][n][r] + bias[r];
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        float v = acc[m][n][r];
        if (S == 2 ? a.out_act == ACT_GELU : a.out_act == ACT_LEAKY) v = S == 2 ? gelu_as(v) : leaky(v, a.out_slope);
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), ors, oo,
                                              4 * (m * 32 + (r & 3) + 8 * (r >> 2)) * (int)a.oc, 0);
      }
    }
  }
}

int max_n_out_s(const ConvLaunch& a) {
  int n = 0;
  for (int g = 0; g < a.n_groups; ++g) n = std::max(n, a.g[g].n_out);
  return n;
}

template <bool BF, int BM, int BN, int WM, int WN, int S = 1>
void launch_s(const ConvLaunch& a, hipStream_t s) {
  using C = CfgS<BF, BM, BN, WM, WN, S>;
  int halo = 0;
  for (int g = 0; g < a.n_groups; ++g) halo = std::max(halo, (a.g[g].K - 1) * a.g[g].dil);
  const size_t lds = 2 * 4 * sizeof(uint4) * (size_t)(S == 2 ? 2 * (BN + 1) : BN + halo);
  constexpr size_t kMax = 2 * 4 * sizeof(uint4) * (size_t)(S == 2 ? 2 * (BN + 1) : BN + kConvHaloMax);
  static_assert(kMax <= 160 * 1024, "LDS of one workgroup");
  if constexpr (kMax > 65536) {
    static bool attr = false;  // per instantiation
    if (!attr) {
      RVC_HIP(hipFuncSetAttribute((const void*)conv1d_split_kernel<BF, BM, BN, WM, WN, S>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMax));
      attr = true;
    }
  }
  const int n_tx = (max_n_out_s(a) + BN - 1) / BN, n_ty = a.C_out / BM;
  const long long items = (long long)n_tx * n_ty * a.B * a.n_groups;
  RVC_CHECK(items < (1LL << 30), "conv1d_split: launch too large");
  launch_timed(conv1d_split_kernel<BF, BM, BN, WM, WN, S>, dim3((unsigned)items), dim3(C::NT), lds, s, a, n_tx, n_ty);
  check_launch("conv1d_split");
}

}  // namespace

bool conv1d_split_supported(int C_in, int C_out, int K, int dil, bool bf16) {
  return C_in % (bf16 ? 32 : 16) == 0 && C_out % 32 == 0 && K >= 1 && conv1d_mfma_supported(K, dil);
}

bool conv1d_split_ok(const ConvLaunch& a) {
  if (a.bias2 || a.post != POST_NONE || a.ln_g || a.ln_stat || a.stat_out || a.res_stat) return false;
  if (a.in_act != ACT_NONE && !(a.in_act == ACT_LEAKY && a.in_slope >= 0.f && a.in_slope <= 1.f)) return false;
  // stride 2 (K <= 3, two fp16 parts): no activation in, none or GELU out
  const bool two = a.g[0].in_step == 2;
  if (a.out_act != ACT_NONE && !(two ? a.out_act == ACT_GELU
                                     : a.out_act == ACT_LEAKY && a.out_slope >= 0.f && a.out_slope <= 1.f))
    return false;
  // and at least 400 tiles of 64 x 64 in one batch item: below that the fp32
  // kernel's workgroups, which share a tile's channels between four waves, are
  // as fast and their sums shorter (HuBERT's six stride-2 convs, ms, fp32 ->
  // this rule / always: 1 s 0.273 -> 0.273 / 0.336, 10 s 0.70 -> 0.40 / 0.41, 30 s
  // 1.80 -> 0.83 / 0.77)
  if (two && (a.in_act != ACT_NONE || !a.g[0].wsc || a.C_out % 64 != 0 ||
              (long long)((max_n_out_s(a) + 63) / 64) * (a.C_out / 64) * a.n_groups < 400))
    return false;
  for (int g = 0; g < a.n_groups; ++g) {
    const ConvGroup& G = a.g[g];
    if (!G.wsp || (two ? G.in_step != 2 || G.K > 3 || G.dil != 1 : G.in_step > 1) || G.out_step != 1 || G.out_off != 0 || G.combine != COMB_STORE ||
        !conv1d_split_supported(a.C_in, a.C_out, G.K, G.dil, !G.wsc) || !G.wsc != !a.g[0].wsc)
      return false;
    // 32-bit buffer offsets
    if (4.0 * G.K * a.C_in * a.C_out >= 2147483648.0) return false;
  }
  const double n = max_n_out_s(a);
  return 4.0 * (31.0 * a.xc + a.L_in) < 2147483648.0 && 4.0 * (a.C_out * (double)a.oc + n) < 2147483648.0 &&
         4.0 * (a.C_out * (double)a.rc + n) < 2147483648.0;
}

void launch_conv1d_split(const ConvLaunch& a, hipStream_t s) {
  RVC_CHECK(conv1d_split_ok(a), "conv1d_split: unsupported launch");
  const int n = max_n_out_s(a);
  if (n == 0) return;
  // The widest tile that leaves one batch item 400 workgroups; never by B, so
  // that a batch equals its items bit for bit also where a tile's own scale
  // or its fp32 sums show.  C = 256 at 10 000 columns (40k stage 0, 1000 frames, ms
  // of its six launches): 64 x 128 0.60, 128 x 128 0.65, 64 x 256 0.76 (the fp32
  // matrix cores: 1.42).
  // tiles of one batch item
  auto wide = [&](int BM, int BN) { return (long long)((n + BN - 1) / BN) * (a.C_out / BM) * a.n_groups >= 400; };
  if (a.g[0].in_step == 2) {
    if (wide(64, 128)) return launch_s<false, 64, 128, 32, 64, 2>(a, s);
    return launch_s<false, 64, 64, 32, 32, 2>(a, s);
  }
  if (!a.g[0].wsc) {
    // C = 256, batch of 4 x 10 000 columns (six launches, ms): 128 x 128 0.84,
    // 64 x 128 0.93, 64 x 256 on 64 x 64 waves 0.92, on 64 x 128 waves 1.25
    // (spills); the one-shot bf16 tiles 3.0
    if (a.C_out % 128 == 0 && wide(128, 128)) return launch_s<true, 128, 128, 64, 64>(a, s);
    if (a.C_out % 64 == 0 && wide(64, 64)) return launch_s<true, 64, 64, 32, 32>(a, s);
    return launch_s<true, 32, 64, 32, 32>(a, s);
  }
  if (a.C_out % 64 == 0) {
    if (wide(64, 128)) return launch_s<false, 64, 128, 32, 64>(a, s);
    if (wide(64, 64)) return launch_s<false, 64, 64, 32, 32>(a, s);
  } else if (wide(32, 256)) {
    return launch_s<false, 32, 256, 32, 64>(a, s);
  }
  launch_s<false, 32, 64, 32, 32>(a, s);
}

}  // namespace rvc
