// fp32 convolution as an implicit GEMM on the bf16 matrix cores, each fp32
// operand split into three bf16 terms (see gemm_x3.hip for the split, its
// error and its handling of infinities and NaNs): M = output channels, N =
// batch * OH * OW pixels, K = channels x filter taps.
//
// A gather of the input per tap reads and splits every element KH * KW times
// with one 4-byte load a lane, which costs the address units sixteen cycles
// per 256 bytes: they, not the matrix cores, bounded that form (a 64 x 64 x
// 32 step: 44 loads, 700 cycles, for 384 cycles of MFMAs). Here a workgroup
// stages the input its pixels read once per 16 * KS channels: the patch, the
// rows its pixels' windows touch (per image, stacked, with the padding as
// zeros), split once and kept in LDS as [8-channel chunk][h, m, l][position]
// [8 bf16]. A lane's B operand for a tap is then one 16-byte read per term at
// its pixel's position plus the tap's offset. Columns are stored by their
// remainder modulo the stride, so that neighbouring pixels are neighbouring
// positions for any stride. A 1x1 convolution's positions are its pixels.
//
// The weights come straight from memory to registers: they are packed
// [32-channel block][k step][h, m, l][lane][8 bf16], k ordered (16-channel
// block, tap, channel), a wave's block and k step one contiguous 3 KB, and
// the waves of a workgroup that share one read it together. The loop over a
// stage's k steps therefore has no barrier; one per stage separates reading
// a patch from writing the next.
//
// Measured against the fp32 implicit GEMM: batch 8, 192 -> 320, 27x27, 3x3
// stride 2 26.3 -> 19.0 us (error against 64 bits 3.7e-7 -> 1.4e-7); batch 32,
// 96 -> 576, 14x14, 1x1 13.2 -> 10.4 us; batch 16, 96 -> 200, 35x35, 3x3 106 ->
// 60 us. A 128 x 128 tile keeps the matrix cores busy 64 % of its time; grids of
// one to two workgroups a CU and the launch bound the rest.
//
// Waves: WGM x WGN, each 32 output channels x 32 * NI pixels. The patch has
// room for PMAX positions (a multiple of 64: a wave stages 64 positions of
// one chunk at a time).
namespace mdlc {

// n / d for 0 <= n < 2^21, 0 < d < 2^21, given inv = rcp(d)
__device__ __forceinline__ int x3_div(int n, int d, float inv) {
  int q = (int)((float)n * inv);
  const int r = n - __mul24(q, d);
  return q + (r >= d) - (r < 0);
}

// Scheduling hints of a k step, as compile-time recursion (their arguments
// must be constants): its memory reads, then its MFMAs each followed by VM
// vector instructions.
template <int I, int MF, int RD, int VM>
struct ConvX3Order {
  __device__ __forceinline__ static void emit() {
    if constexpr (I < MF) {
      if constexpr (I == 0) __builtin_amdgcn_sched_group_barrier(0x120, RD, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, VM, 0);
      ConvX3Order<I + 1, MF, RD, VM>::emit();
    }
  }
};

template <int WGM, int WGN, int NI, int KS, int PMAX, int D, int OUT, class Epi, class Win>
__device__ __forceinline__ void conv_x3(const GemmArgs& g, int bid = -1) {
  constexpr int NT = WGM * WGN * 64;
  constexpr int BM = 32 * WGM, WN = 32 * NI, BN = WN * WGN;
  constexpr int T = Win::KH * Win::KW;
  constexpr bool ONE = T == 1;
  constexpr int NK = KS * T;                      // k steps per stage
  constexpr int NW = WGM * WGN;
  constexpr int GR = PMAX / 64, NG = 2 * KS * GR; // 64-position groups per chunk and per stage
  constexpr int PT = (NG + NW - 1) / NW;          // and per wave
  constexpr int PLANE = PMAX * 16, CHUNK = 3 * PLANE, BUF = 2 * KS * CHUNK;
  static_assert(PMAX % 64 == 0, "whole waves stage one chunk");
  static_assert(NK % D == 0, "the weight registers rotate within a stage");
  __shared__ __attribute__((aligned(1024))) char patch[2 * BUF];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WGN, wn0 = (wave % WGN) * WN;
  const int li = lane & 31, lk = lane >> 5;

  const int tiles_m = (g.M + BM - 1) / BM;
  const int tiles_n = (g.N + BN - 1) / BN;
  const int tiles = tiles_m * tiles_n;
  const int t = xcd_remap(bid < 0 ? (int)blockIdx.x : bid, tiles * g.ksplit);
  const int ks = t / tiles;
  int mt, nt;
  grouped_tile<8>(t - ks * tiles, tiles_m, tiles_n, mt, nt);
  const int m0 = mt * BM, n0 = nt * BN;
  const int ksteps = g.K >> 4;
  const int step0 = ks * (g.kchunk >> 4);
  const int nst = (min(g.kchunk >> 4, ksteps - step0)) / NK;   // stages (K is packed in whole ones)
  const int cbeg = step0 / T * 16;                // first channel

  // ---- patch geometry ---------------------------------------------------------
  const int HW = g.H * g.W, OHW = g.OH * g.OW;
  const int WP = (g.OW - 1) * Win::SW + (Win::KW - 1) * Win::DW + 1;
  const int WPH = (WP + Win::SW - 1) / Win::SW;
  const int WR = WPH * Win::SW;                   // positions per row
  const int FR = (g.OH - 1) * Win::SH + (Win::KH - 1) * Win::DH + 1;   // padded rows of an image
  const int nf = n0 / OHW;
  const int plast = min(n0 + BN, g.N) - 1;
  const int nl = plast / OHW;
  const float iOW = __builtin_amdgcn_rcpf((float)g.OW), iOHW = __builtin_amdgcn_rcpf((float)OHW);
  const int rlo = (n0 - nf * OHW) / g.OW * Win::SH;
  const int rlast = (plast - nl * OHW) / g.OW * Win::SH + (Win::KH - 1) * Win::DH + 1;
  const int rows0 = (nl == nf ? rlast : FR) - rlo;
  const int PS = (rows0 + (nl > nf ? (nl - nf - 1) * FR + rlast : 0)) * WR;

  // wave w stages groups w, w + NW, ...: byte offset (channel 0) of the
  // lane's position in each, or kOutside
  int x_off[PT];
  {
    const float iWR = __builtin_amdgcn_rcpf((float)WR), iFR = __builtin_amdgcn_rcpf((float)FR);
    const float iWPH = __builtin_amdgcn_rcpf((float)WPH);
#pragma unroll
    for (int i = 0; i < PT; ++i) {
      const int e = (wave + i * NW) % GR * 64 + lane;
      int n, ih, iw;
      bool ok;
      if (ONE) {
        const int p = n0 - nf * OHW + e;          // from image nf's first pixel
        const int s1 = x3_div(p, OHW, iOHW);
        const int s = p - s1 * OHW;
        const int oh = x3_div(s, g.OW, iOW);
        n = nf + s1;
        ih = oh * Win::SH - Win::PT;
        iw = (s - oh * g.OW) * Win::SW - Win::PL;
        ok = n0 + e <= plast;
      } else {
        const int q = x3_div(e, WR, iWR);
        const int c = e - q * WR;
        const int cr = Win::SW == 1 ? 0 : x3_div(c, WPH, iWPH);
        const int col = (c - cr * WPH) * Win::SW + cr;
        int row = rlo + q;
        n = nf;
        if (q >= rows0) {
          const int R = q - rows0, s1 = x3_div(R, FR, iFR);
          n = nf + 1 + s1;
          row = R - s1 * FR;
        }
        ih = row - Win::PT;
        iw = col - Win::PL;
        ok = e < PS;
      }
      ok = ok && (unsigned)ih < (unsigned)g.H && (unsigned)iw < (unsigned)g.W;
      x_off[i] = ok ? (n * g.ximg + ih * g.W + iw) * 4 : kOutside;
    }
  }
  // the lane's pixels' positions, in bytes (plus its half's chunk)
  int pos[NI];
#pragma unroll
  for (int ni = 0; ni < NI; ++ni) {
    int p = n0 + wn0 + ni * 32 + li;
    p = p <= plast ? p : n0;                      // past the last pixel: any window, never stored
    int at;
    if (ONE) {
      at = p - n0;
    } else {
      const int r = p - nf * OHW;
      const int s1 = x3_div(r, OHW, iOHW);
      const int s = r - s1 * OHW;
      const int oh = x3_div(s, g.OW, iOW);
      at = (s1 == 0 ? oh * Win::SH - rlo : rows0 + (s1 - 1) * FR + oh * Win::SH) * WR + s - oh * g.OW;
    }
    pos[ni] = at * 16 + lk * CHUNK;
  }

  // ---- staging ------------------------------------------------------------------
  const __amdgpu_buffer_rsrc_t rsX = buffer_over(g.B, g.N / OHW * g.ximg * 4);
  float xv[PT][8];
  auto load_x = [&](int c0) {                     // the chunks of channels c0 .. c0 + 16 KS - 1
#pragma unroll
    for (int i = 0; i < PT; ++i) {
      if (NG % NW != 0 && wave + i * NW >= NG) break;
      const int c = c0 + (wave + i * NW) / GR * 8;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        xv[i][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
            rsX, c + j < g.Cin ? x_off[i] : kOutside, (c + j < g.Cin ? c + j : 0) * HW * 4, 0));
    }
  };
  auto store_x = [&](int i, char* buf) {
    if (NG % NW != 0 && wave + i * NW >= NG) return;
    uintx4_t p[3];
    split_bf16x3(xv[i], p);
    char* at = buf + (wave + i * NW) / GR * CHUNK + ((wave + i * NW) % GR * 64 + lane) * 16;
#pragma unroll
    for (int q = 0; q < 3; ++q) *reinterpret_cast<uintx4_t*>(at + q * PLANE) = p[q];
  };
  const int wblocks = (g.M + 31) >> 5;
  const __amdgpu_buffer_rsrc_t rsW = buffer_over(g.A, wblocks * ksteps * 3072);
  const int w_off = lane * 16;
  int w_at = (min((m0 >> 5) + wm, wblocks - 1) * ksteps + step0) * 3072;   // next k step to load
  bf16x8_t a[D][3];
  auto load_w = [&](int d) {
    // past the last k step of the constant: zeros (never used)
#pragma unroll
    for (int q = 0; q < 3; ++q)
      a[d][q] = __builtin_bit_cast(bf16x8_t, __builtin_amdgcn_raw_buffer_load_b128(rsW, w_off + w_at + q * 1024, 0, 0));
    w_at += 3072;
  };

  floatx16 acc[1][NI], small[1][NI];
#pragma unroll
  for (int ni = 0; ni < NI; ++ni)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[0][ni][r] = small[0][ni][r] = 0.f;

  auto tap_off = [&](int k) {                     // bytes from a window's first position
    const int kh = k % T / Win::KW, kw = k % Win::KW;
    return ONE ? 0 : (kh * Win::DH * WR + kw * Win::DW % Win::SW * WPH + kw * Win::DW / Win::SW) * 16;
  };
  auto read_b = [&](const char* rd, int k, bf16x8_t (&b)[NI][3]) {
    const char* at = rd + tap_off(k) + k / T * 2 * CHUNK;
#pragma unroll
    for (int ni = 0; ni < NI; ++ni)
#pragma unroll
      for (int q = 0; q < 3; ++q) b[ni][q] = *reinterpret_cast<const bf16x8_t*>(at + pos[ni] + q * PLANE);
  };

  load_x(cbeg);
#pragma unroll
  for (int d = 0; d < D - 1; ++d) load_w(d);
#pragma unroll
  for (int i = 0; i < PT; ++i) store_x(i, patch);
  __syncthreads();
  int cur = 0;
  bf16x8_t b[2][NI][3];                           // this k step's operands and the next's
  for (int st = 0; st < nst; ++st) {
    const bool more = st + 1 < nst;
    const char* rd = patch + cur;
    cur = BUF - cur;
    char* wr = patch + cur;
    read_b(rd, 0, b[0]);
    if (more) load_x(cbeg + (st + 1) * 16 * KS);
#pragma unroll
    for (int k = 0; k < NK; ++k) {
      __builtin_amdgcn_sched_barrier(0);
      load_w((k + D - 1) % D);
      if (k + 1 < NK) read_b(rd, k + 1, b[(k + 1) & 1]);
      constexpr int PA[6] = {2, 0, 1, 1, 0, 0}, PB[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
      for (int p = 0; p < 6; ++p)
#pragma unroll
        for (int ni = 0; ni < NI; ++ni) {
          floatx16& c = p < 5 ? small[0][ni] : acc[0][ni];
          c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[k % D][PA[p]], b[k & 1][ni][PB[p]], c, 0, 0, 0);
        }
      // the next stage's groups over the last k steps
      constexpr int PER = (PT + NK - 1) / NK;
      if (more) {
#pragma unroll
        for (int i = 0; i < PT; ++i)
          if (k == NK - 1 - (PT - 1 - i) / PER) store_x(i, wr);
      }
      ConvX3Order<0, 6 * NI, 3 + 3 * NI, 4>::emit();
    }
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
  }

  float z = 0.f;
#pragma unroll
  for (int ni = 0; ni < NI; ++ni)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      acc[0][ni][r] += small[0][ni][r];
      z += acc[0][ni][r] * 0.f;
    }
  if (__any(z != 0.f)) {
    // a NaN or an infinity: the wave's tile again, in fp32
    for (int e = lane; e < 32 * WN; e += 64) {
      const int row = m0 + wm * 32 + e / WN, col = n0 + wn0 + e % WN;
      if (row >= g.M || col >= g.N) continue;
      const int n = col / OHW, s = col - n * OHW;
      const int ih0 = s / g.OW * Win::SH - Win::PT, iw0 = s % g.OW * Win::SW - Win::PL;
      float v = 0.f;
      for (int k = step0 * 16; k < (step0 + nst * NK) * 16; ++k) {
        const int c = k / (16 * T) * 16 + k % 16, tap = k / 16 % T;
        if (c >= g.Cin) continue;
        const int ih = ih0 + tap / Win::KW * Win::DH, iw = iw0 + tap % Win::KW * Win::DW;
        const bool in = (unsigned)ih < (unsigned)g.H && (unsigned)iw < (unsigned)g.W;
        const float x = in ? g.B[(size_t)n * g.ximg + (size_t)c * HW + ih * g.W + iw] : 0.f;
        v = __builtin_fmaf(x3_weight(g.A, ksteps, row, k), x, v);
      }
      if (OUT == 2) {
        g.C[((size_t)ks * g.M + row) * g.N + col] = v;
      } else {
        const size_t o = (size_t)n * g.cimg + (size_t)row * OHW + s;
        v = Epi::apply(v, Epi::bias == 1 ? g.bias[row] : 0.f);
        if (Epi::residual) v = Epi::post(v, g.R[o]);
        g.C[o] = v;
      }
    }
    return;
  }
  x3_store<BM, BN, WGM, WGN, OUT, Epi>(g, acc, m0, n0, ks);
}

}  // namespace mdlc
