// The stride-1 2-D convolutions of the RMVPE U-Net on split fp16 products
// (conv_split.hip describes the split, its range and its error).
//
// Every U-Net convolution of ten seconds is 0.6 GFLOP, 1 us of these products;
// what bounds it is how long one wave's chain of steps is.  So the waves are
// many and their chains short: a workgroup forms 32 channels x 32 points, its
// NW waves each take a run of 16-channel chunks and all of the tile, and the
// partial tiles are added in wave order in LDS.  The fp32 kernel in rmvpe.hip,
// which staged 8 channels for a whole workgroup behind two barriers and split
// the deep levels' channels over workgroups with a reduce launch behind, took
// 16 - 26 us a convolution.
//
// The 32 points are 4 rows x 8 columns (8 x 4 where the image is 4 wide): a
// window of at most 60 positions serves all nine taps.  Each wave stages its own
// chunk, split on the way, into its own part of LDS as
//   xs[part][channel / 8][position] in units of 8 channels (16 bytes),
// without a barrier; the next chunk's loads are in flight during its taps.  The
// weights come from L2 in operand order (SessionBase::upload_split), two taps
// ahead.  Workgroups 8 apart hold the same weights where there are 8 row
// blocks: one XCD's L2 reads each weight of the deep levels once.
#include <algorithm>

#include "split.h"

namespace rvc {

namespace {

constexpr int kPos = 60;                // the window's positions
constexpr int kXsUnits = 4 * kPos;      // [part][channel group][position]
constexpr int kTileFloats = 32 * 32;    // one wave's partial tile

template <int NW>
__global__ __launch_bounds__(64 * NW) void conv2d_split_kernel(Conv2dLaunch a, int n_row, int n_pt, int ntc) {
  extern __shared__ uint4 sm[];  // NW windows, then NW partial tiles in the same place
  const int gi = blockIdx.y / a.B, bb = blockIdx.y - gi * a.B;
  const Conv2dGroup& G = a.g[gi];
  int lin = blockIdx.x;
  if (n_row < 8) {  // a run of neighbouring tiles per XCD (run_c2s)
    lin = (lin & 7) * (int)(gridDim.x >> 3) + (lin >> 3);
    if (lin >= n_row * n_pt) return;  // uniform, before any barrier
  }
  const int row = lin % n_row, pt = lin / n_row;
  const int TC = a.tile_c, TR = 32 / TC, tcs = __builtin_ctz(TC);
  const int tr = pt / ntc, a0 = tr * TR, b0 = (pt - tr * ntc) * TC, co0 = row * 32;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5, l32 = lane & 31;
  const int T = G.ntaps, n = a.C_in / 16;
  const int k_lo = blockIdx.z * a.csplit, k_n = min(a.csplit, n - k_lo);
  const int c_lo = k_lo + k_n * wave / NW, c_hi = k_lo + k_n * (wave + 1) / NW;

  // ---- staging: unit u = (channel group u / np, position u % np)
  const int WC = TC + G.dw_span, np = (TR + G.dh_span) * WC;
  const float* xb = a.x + (long long)bb * a.xb;
  const unsigned xrow = 4u * (unsigned)a.xc;
  uint4* xs = sm + wave * kXsUnits;
  unsigned xo[2];
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int u = lane + 64 * e, c8 = u >= np, p = u - c8 * np;
    const int rr = p / WC, h = a0 + G.dh_lo + rr, w = b0 + G.dw_lo + p - rr * WC;
    xo[e] = u < 2 * np && h >= 0 && h < a.H && w >= 0 && w < a.W ? c8 * 8u * xrow + 4u * (unsigned)(h * a.W + w) : kBufOut;
  }
  float xv[2][8];
  auto gload = [&](int c) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t rs = uniform_rsrc(xb + (long long)c * 16 * a.xc, 15u * xrow + 4u * (unsigned)(a.H * a.W));
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
      for (int j = 0; j < 8; ++j) xv[e][j] = buf_load4(rs, xo[e], j * xrow);
  };
  float sx = kScaleX, xm[2];  // each unit's largest magnitude, scaled
  auto lstore = [&]() __attribute__((always_inline)) {
    // a wave's LDS operations run in order; the fences keep the compiler to it
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int e = 0; e < 2; ++e)
      if (lane + 64 * e < 2 * np) stage_unit<false>(xv[e], sx, xm[e], xs + lane + 64 * e, 2 * np);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };

  // ---- weights: part q of step (chunk c, tap t) at ((c T + t) 2 + q) nrb KiB
  const unsigned wpart = 1024u * (unsigned)n_row;
  const __amdgpu_buffer_rsrc_t wrs = uniform_rsrc(G.wsp, (unsigned)(n * T) * 2u * wpart);
  const unsigned wvo = 16u * (unsigned)lane + 1024u * (unsigned)row;
  uint4 Ah[2], Al[2];
  // tap t's offset in the window
  auto tap_off = [&](int t) __attribute__((always_inline)) { return (G.tap_h >> 2 * t & 3) * WC + (G.tap_w >> 2 * t & 3); };
  const uint4* xp = xs + half * np + (l32 >> tcs) * WC + (l32 & (TC - 1));

  floatx16 acc;
  bool mixed = false;  // some units lie outside the split's range
  for (bool again = false;; again = true) {
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    xm[0] = xm[1] = 0.f;
    gload(c_lo);
    const unsigned last = (unsigned)(n * T - 1) * 2u * wpart;
    unsigned next = (unsigned)(c_lo * T) * 2u * wpart;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      Al[i] = buf_load16(wrs, wvo, next + wpart);
      Ah[i] = buf_load16(wrs, wvo, next);
      next = min(next + 2 * wpart, last);
    }
    for (int c = c_lo; c < c_hi; ++c) {
      lstore();
      if (c + 1 < c_hi) gload(c + 1);
      int off = tap_off(0);
      uint4 Bh = xp[off], Bl = xp[off + 2 * np];
      auto tap = [&](int t, uint4& H, uint4& Lo) __attribute__((always_inline)) {
        off = tap_off(min(t + 1, T - 1));
        acc = mma16<false>(Lo, Bh, acc);
        Lo = buf_load16(wrs, wvo, next + wpart);
        acc = mma16<false>(H, Bh, acc);
        Bh = xp[off];
        acc = mma16<false>(H, Bl, acc);
        H = buf_load16(wrs, wvo, next);
        Bl = xp[off + 2 * np];
        next = min(next + 2 * wpart, last);
      };
      int t = 0;
      for (; t + 1 < T; t += 2) {
        tap(t, Ah[0], Al[0]);
        tap(t + 1, Ah[1], Al[1]);
      }
      if (t < T) {
        tap(t, Ah[0], Al[0]);
        const uint4 h = Ah[0], l = Al[0];
        Ah[0] = Ah[1]; Al[0] = Al[1];
        Ah[1] = h; Al[1] = l;
      }
    }
    float top;
    const unsigned f = range_bits(xm, 1.f, top);
    mixed = __any(f & 1u);
    if (!mixed || again || __any(f & 2u)) break;
    // no unit fits: again with a scale of the wave's own
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) top = fmaxf(top, __shfl_xor(top, d));
    top = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, top)));
    if (top == 0.f) break;  // infinities and zeros
    sx = pow2_scale(top * (1.f / kScaleX));
  }

  const int pr = a0 + (l32 >> tcs), pc = b0 + (l32 & (TC - 1));
  // the points whose own inputs the scale does not hold, or whose sums are NaN
  bool bad = false;
  if (mixed) {
    unsigned* cm = reinterpret_cast<unsigned*>(xs);  // a position's largest magnitude, over the wave's window
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (lane < np) cm[lane] = 0u;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int u = lane + 64 * e;
      if (u < 2 * np) atomicMax(cm + (u < np ? u : u - np), __builtin_bit_cast(unsigned, xm[e]));
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    unsigned t = 0;
    for (int k = 0; k < T; ++k) t = max(t, cm[(l32 >> tcs) * WC + (l32 & (TC - 1)) + tap_off(k)]);
    bad = !split_holds(__builtin_bit_cast(float, t));
  }
  float nan = 0.f;
#pragma unroll
  for (int r = 0; r < 16; ++r) nan = fmaf(acc[r], 0.f, nan);
  bad = bad || nan != nan;
  const __amdgpu_buffer_rsrc_t srs = uniform_rsrc(G.wsc, 128u * (unsigned)n_row);
#pragma unroll
  for (int r = 0; r < 16; ++r)
    acc[r] *= buf_load4(srs, 4u * (unsigned)(co0 + 4 * half), 4 * ((r & 3) + 8 * (r >> 2))) * (1.f / sx);
  if (__any(bad)) {  // this wave's channels again in fp32
    floatx16 f[1][1];
    const __amdgpu_buffer_rsrc_t frs = uniform_rsrc(G.w, 4u * (unsigned)(T * a.C_in * a.w_ld));
    const unsigned fo = co0 + l32 < a.C_out ? 4u * (unsigned)(half * a.w_ld + co0 + l32) : kBufOut;
    fp32_sums(
        f, 16 * (c_hi - c_lo), T,
        [&](float(&A)[1], int t, int c) {
          A[0] = buf_load4(frs, fo, 4u * (unsigned)((t * a.C_in + 16 * c_lo + c) * a.w_ld));
        },
        [&](float(&B)[1], int t, int c) {
          const __amdgpu_buffer_rsrc_t rs =
              uniform_rsrc(xb + (long long)(16 * c_lo + c) * a.xc, xrow + 4u * (unsigned)(a.H * a.W));
          const int h = pr + G.dh[t], w = pc + G.dw[t];
          B[0] = buf_load4(rs, h >= 0 && h < a.H && w >= 0 && w < a.W ? half * xrow + 4u * (unsigned)(h * a.W + w) : kBufOut, 0);
        });
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = bad ? f[0][0][r] : acc[r];
  }

  // ---- partial tiles [wave][channel][point], added in wave order
  float* part = reinterpret_cast<float*>(sm);
  __syncthreads();  // every wave is done with its window
#pragma unroll
  for (int r = 0; r < 16; ++r) part[wave * kTileFloats + (4 * half + (r & 3) + 8 * (r >> 2)) * 32 + l32] = acc[r];
  __syncthreads();
  float* ob = a.out + (long long)bb * a.ob;
  const float* rb = a.res ? a.res + (long long)bb * a.ob : nullptr;
  const bool taps = pr < G.a_lim && pc < G.b_lim;
  if (pr >= G.oh_n || pc >= G.ow_n) return;
  const long long o = (long long)(pr * a.osh + G.oh0) * a.ors + (long long)(pc * a.osw + G.ow0) * a.ocs;
#pragma unroll
  for (int i = 0; i < 16 / NW; ++i) {
    const int r = tid / 32 + i * 2 * NW, co = co0 + r;
    if (co >= a.C_out) break;
    float v = part[r * 32 + l32];
#pragma unroll
    for (int w = 1; w < NW; ++w) v += part[w * kTileFloats + r * 32 + l32];
    if (!taps) v = 0.f;
    if (a.ksplit > 1) {
      a.part[((long long)(blockIdx.z * gridDim.y + blockIdx.y) * a.C_out + co) * a.OH * a.OW + pr * a.OW + pc] = v;
      continue;
    }
    if (a.bias) v += a.bias[co];
    if (a.relu) v = fmaxf(v, 0.f);
    if (rb) v += rb[co * a.oc + o];
    ob[co * a.oc + o] = v;
  }
}

template <int NW>
void run_c2s(const Conv2dLaunch& a, int n_row, int n_pt, int ntc, hipStream_t s) {
  const size_t lds = (size_t)NW * std::max<size_t>(sizeof(uint4) * kXsUnits, sizeof(float) * kTileFloats);
  // Below 8 row blocks the image is wide and the weights are few: neighbouring
  // tiles, which share 128-byte lines of the input and of the output, go to one
  // XCD; above, a row block's tiles do, for its weights.  (Ten seconds, a launch
  // of 16 / 32 / 64 channels 20.6 / 14.4 / 11.6 -> 15.5 / 11.3 / 9.6 us.)
  const unsigned gx = (unsigned)(n_row < 8 ? (n_row * n_pt + 7) / 8 * 8 : n_row * n_pt);
  hipLaunchKernelGGL(conv2d_split_kernel<NW>, dim3(gx, (unsigned)(a.n_groups * a.B), (unsigned)a.ksplit),
                     dim3(64 * NW), lds, s, a, n_row, n_pt, ntc);
  check_launch("conv2d_split");
}

}  // namespace

bool conv2d_split_supported(int C_in, int C_out) { return C_in >= 16 && C_in % 16 == 0 && C_out % 16 == 0; }

bool conv2d_split_ok(const Conv2dLaunch& a) {
  if (a.stride != 1 || !conv2d_split_supported(a.C_in, a.C_out) || a.OW < 4) return false;
  for (int g = 0; g < a.n_groups; ++g)
    if (!a.g[g].wsp || !a.g[g].wsc) return false;
  const long long n_row = (a.C_out + 31) / 32;
  const long long pts = (long long)((a.OH + 3) / 4 + 1) * ((a.OW + 3) / 4 + 1);
  // 32-bit byte offsets into 16 planes and into the weights
  return a.xc >= 0 && 64LL * std::max(a.xc, (long long)a.H * a.W) < (1LL << 31) &&
         a.C_in / 16 * 9 * 2048LL * n_row < (1LL << 31) && n_row * pts < (1LL << 30) &&
         (long long)a.n_groups * a.B <= 65535;
}

// The tile grid, and the split of long reductions (at 32 chunks a workgroup's
// weights are 590 KB, which one CU takes 10 us to stream) over workgroups where
// the tiles leave CUs idle, 8 chunks each, with a reduce launch behind: the
// intermediate level's 3x3 convs at ten seconds, 64 tiles, 18.3 -> 9.5 + 4.4 us.
// At 16 chunks (256 channels, 128 tiles, 12 us) the reduce launch would cost
// what the split gives.
void conv2d_split_plan(Conv2dLaunch& a, int& n_row, int& n_pt, int& ntc) {
  a.tile_c = a.OW <= 4 ? 4 : 8;
  const int TR = 32 / a.tile_c, n = a.C_in / 16;
  ntc = (a.OW + a.tile_c - 1) / a.tile_c;
  n_row = (a.C_out + 31) / 32;
  n_pt = (a.OH + TR - 1) / TR * ntc;
  bool nine = true;
  for (int g = 0; g < a.n_groups; ++g) nine = nine && a.g[g].ntaps == 9;
  a.ksplit = 1;
  a.csplit = n;
  if (nine && n >= 32 && (long long)n_row * n_pt * a.n_groups < 128) {
    a.csplit = 8;
    a.ksplit = (n + 7) / 8;
  }
}

size_t conv2d_split_part_floats(const Conv2dLaunch& a0) {
  Conv2dLaunch a = a0;
  int n_row, n_pt, ntc;
  conv2d_split_plan(a, n_row, n_pt, ntc);
  return a.ksplit > 1 ? (size_t)a.ksplit * a.n_groups * a.B * a.C_out * a.OH * a.OW : 0;
}

void launch_conv2d_split(Conv2dLaunch& a, hipStream_t s) {
  int n_row, n_pt, ntc;
  conv2d_split_plan(a, n_row, n_pt, ntc);
  if (a.ksplit > 1 && (!a.part || a.part_floats < (size_t)a.ksplit * a.n_groups * a.B * a.C_out * a.OH * a.OW)) {
    a.ksplit = 1;
    a.csplit = a.C_in / 16;
  }
  for (int g = 0; g < a.n_groups; ++g) {
    Conv2dGroup& G = a.g[g];
    G.tap_h = G.tap_w = 0;
    for (int t = 0; t < G.ntaps; ++t) {
      G.tap_h |= (unsigned)(G.dh[t] - G.dh_lo) << 2 * t;
      G.tap_w |= (unsigned)(G.dw[t] - G.dw_lo) << 2 * t;
    }
  }
  // waves per tile: 2048 waves or a wave per chunk of 16 channels
  const long long tiles = (long long)n_row * n_pt * a.n_groups * a.ksplit;
  int nw = 1;
  while (nw < 16 && 2 * nw <= a.csplit && tiles * nw < 2048) nw *= 2;
  if (nw == 16) run_c2s<16>(a, n_row, n_pt, ntc, s);
  else if (nw == 8) run_c2s<8>(a, n_row, n_pt, ntc, s);
  else if (nw == 4) run_c2s<4>(a, n_row, n_pt, ntc, s);
  else if (nw == 2) run_c2s<2>(a, n_row, n_pt, ntc, s);
  else run_c2s<1>(a, n_row, n_pt, ntc, s);
}

}  // namespace rvc
