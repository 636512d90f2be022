// 3x3 stride-1 convolution by Winograd F(2x2, 3x3) (see conv_wino.hip for the
// algorithm and its matrices), the sixteen channel sums on the bf16 matrix
// cores with each fp32 operand split into three bf16 terms (gemm_x3.hip):
// the transforms stay in fp32, U and V are split, and a sum costs 16 / 6 = 2.7
// times less matrix-core time than with the fp32 instruction.
//
// A workgroup of eight waves owns 64 output channels x 64 tiles, like the fp32
// kernel, in chunks of 16 channels (one v_mfma_f32_32x32x16_bf16 deep). Wave w
// owns positions 2 w and 2 w + 1 (one window row pair, three columns) for all
// channels and tiles: 2 x 2 x 2 blocks of 32x32, 128 accumulators a lane, two
// waves a SIMD. So no filter operand is used by two waves: they are loaded
// from memory to registers in the lanes' order (12 KB a wave and chunk), and
// LDS holds only the input patch. A lane's B operand (tile li, channels 8 lk ..
// 8 lk + 7) is what it transforms and splits itself. (One position a wave,
// sixteen waves: four reads and three additions a channel and position instead
// of three and two and a half, and everything in step: 39.4 us against 34.)
//
// Per chunk and SIMD: 3072 cycles of MFMAs, 2050 of vector instructions; per CU
// 1540 of LDS reads and 3580 of the address unit (128 patch loads of 256 bytes
// and 96 filter loads of 1 KB, 16 each). They are woven by hand (the regions
// below). A chunk measured 2.7 us (2.2 without its loads, 1.5 only its MFMAs),
// prologue and epilogue 10 us, of which the LDS exchange and the output 6.5.
// Measured, fp32 kernel -> this one: 32 x 28x28, 128 -> 128 channels and residual
// 46.9 -> 33.9 us; 56x56, 64 -> 64 51.1 -> 45.5; 14x14, 256 -> 256 48.6 -> 33; 7x7,
// 512 -> 512 50 -> 39. Error against 64 bits 2.1e-7 - 2.4e-7 (fp32 kernel 2.6e-7 -
// 2.9e-7).
//
// The bf16 instruction rounds its sums down a little on average (a mean error
// of 1e-8 of the result's rms at 512 channels, 1e-10 with the fp32 one), which
// would add up over a network's layers. So U is negated on the odd rows of
// positions and, once more, on column 2: each output then has nearly as many
// positions whose error is turned up as down, instead of nine down.
//
// The patch of a chunk is loaded straight to LDS two regions to a chunk ahead;
// one barrier a chunk. The output transform sums over the waves through LDS, one
// tile half at a time. An output that is not finite is computed again in fp32
// (the split turns an infinity into NaN).
namespace mdlc {

constexpr int WINO_X3_NT = 512;
// Patch stride per channel. A patch is four planes, by the parities of row and
// column, so that one window position of neighbouring tiles is neighbouring
// floats; channels 8 - 15, the other half of a wave, sit on the other banks.
constexpr int WINO_X3_PSTR = WINO_PMAX + 4;
constexpr int WINO_X3_CHUNK = 16 * 2 * 3 * 1024;      // filter image bytes of a chunk

// Output (i, j) of one tile and channel (oc of the block of 64) over channels
// [c0, c1) in fp32, in conv_wino_f32's order of additions, so that what
// overflows is the same: the window's first row and column are ih, iw.
__device__ __forceinline__ float wino_x3_slow(const WinoArgs& g, const float* ublk, int c0, int c1, int oc, int n,
                                           int ih, int iw, int i, int j) {
  const unsigned short* img = reinterpret_cast<const unsigned short*>(ublk);
  float y = 0.f;
  for (int h = 0; h < 2; ++h) {                       // rows 2 h, 2 h + 1 of M: A^T = (1 1 1 0; 0 1 -1 -1)
    float yh = 0.f;
    for (int b = j; b < 3 + j; ++b) {
      float s = 0.f;
      for (int a = max(i, 2 * h); a < min(3 + i, 2 * h + 2); ++a) {
        float m = 0.f;
        for (int c = c0; c < c1; ++c) {
          const float* xc = g.x + ((size_t)n * g.C + c) * g.H * g.W;
          auto d = [&](int r, int k) {
            const int h = ih + r, w = iw + k;
            return (unsigned)h < (unsigned)g.H && (unsigned)w < (unsigned)g.W ? xc[(size_t)h * g.W + w] : 0.f;
          };
          auto row = [&](int k) {                     // (B^T d) at row a, column k
            return a == 0 ? d(0, k) - d(2, k) : a == 1 ? d(1, k) + d(2, k) : a == 2 ? d(2, k) - d(1, k) : d(1, k) - d(3, k);
          };
          const float v = b == 0 ? row(0) - row(2) : b == 1 ? row(1) + row(2) : b == 2 ? row(2) - row(1) : row(1) - row(3);
          const unsigned short* p = img + ((size_t)(c >> 4) * 32 + (4 * a + b) * 2 + (oc >> 5)) * 1536 +
                                    ((c >> 3 & 1) * 32 + (oc & 31)) * 8 + (c & 7);
          const float u = __builtin_bit_cast(float, (unsigned)p[0] << 16) +
                          (__builtin_bit_cast(float, (unsigned)p[512] << 16) +
                           __builtin_bit_cast(float, (unsigned)p[1024] << 16));
          m = __builtin_fmaf(u, v, m);
        }
        s = (i + h == 2) != (a % 2 != (b == 2)) ? s - m : s + m;
      }
      yh = j == 1 && b > 1 ? yh - s : yh + s;
    }
    y += yh;
  }
  return y;
}

template <bool SPLIT, int PL, bool FULL, class Epi>
__device__ __forceinline__ void conv_wino_x3(const WinoArgs& g) {
  static_assert(PL * 64 <= WINO_PMAX, "patch larger than its LDS");
  __shared__ __attribute__((aligned(1024))) float p0[16 * WINO_X3_PSTR], p1[16 * WINO_X3_PSTR];
  __shared__ __attribute__((aligned(1024))) float ex[16 * 4 * 64 * 4];
  __shared__ int poff[PL * 64];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int a = wave >> 1, bp = wave & 1;               // position row, column pair: positions 2 wave, 2 wave + 1
  const int li = lane & 31, lk = lane >> 5;

  const int P = g.N * g.TH * g.TW;                    // < 2^21 (checked by the host)
  const int tiles_n = (P + 63) >> 6;
  // the work item of this workgroup, as in conv_wino_f32
  const int slices = SPLIT ? (int)gridDim.y : 1;
  const int w = xcd_remap(blockIdx.x + (int)gridDim.x * (int)blockIdx.y, (int)gridDim.x * slices);
  const int os = wino_div(w, tiles_n, __builtin_amdgcn_rcpf((float)tiles_n));
  const int t0 = (w - os * tiles_n) * 64;
  const int ocb = SPLIT ? os / slices : os;
  const int slice = SPLIT ? os - ocb * slices : 0;
  const int chunk0 = slice * g.nchunk;
  const int nch = g.nchunk;
  const int HW = g.H * g.W;

  const float* ublk = g.U + (size_t)ocb * (g.CP / 16) * (WINO_X3_CHUNK / 4);
  bf16x8_t u[2][2][3];                                // the chunk's filter operands, [position][block]
  auto load_u = [&](int chunk, int pos, int q) {
    const __amdgpu_buffer_rsrc_t r = buffer_over(ublk + (size_t)chunk * (WINO_X3_CHUNK / 4), WINO_X3_CHUNK);
#pragma unroll
    for (int blk = 0; blk < 2; ++blk)
      u[pos][blk][q] = __builtin_bit_cast(bf16x8_t, __builtin_amdgcn_raw_buffer_load_b128(
          r, lane * 16, ((2 * wave + pos) * 2 + blk) * 3072 + q * 1024, 0));
  };
#pragma unroll
  for (int q = 2; q >= 0; --q) {
    load_u(chunk0, 0, q);
    load_u(chunk0, 1, q);
  }

  // ---- the patch, laid out as in conv_wino_f32 --------------------------------
  const int TT = g.TH * g.TW;
  const int WP = 2 * g.TW + 2;
  const int SR = 2 * g.TH + 2;
  const float iTT = __builtin_amdgcn_rcpf((float)TT), iTW = __builtin_amdgcn_rcpf((float)g.TW);
  const float iSR = __builtin_amdgcn_rcpf((float)SR);
  const int nfirst = wino_div(t0, TT, iTT);
  const int plast = min(t0 + 63, P - 1);
  const int nlast = wino_div(plast, TT, iTT);
  const int rlo0 = 2 * wino_div(t0 - nfirst * TT, g.TW, iTW) - g.PT;
  const int rhil = 2 * wino_div(plast - nlast * TT, g.TW, iTW) + 3 - g.PT;
  const int rows0 = (nlast == nfirst ? rhil : 2 * g.TH + 1 - g.PT) - rlo0 + 1;
  const int seg = SR * WP;
  const int PS = rows0 * WP + (nlast > nfirst ? (nlast - nfirst - 1) * seg + (rhil + g.PT + 1) * WP : 0);

  // tile th * 32 + li: image, tile row, tile column and window base
  auto tile_at = [&](int th, int& n, int& ty, int& tx) {
    const int p = t0 + 32 * th + li;
    const int pc = p < P ? p : t0;                    // tiles past the batch: any window, never stored
    n = wino_div(pc, TT, iTT);
    ty = wino_div(pc - n * TT, g.TW, iTW);
    tx = pc - n * TT - ty * g.TW;
  };
  // the wave's rows of B^T d: d[r1] + s2 d[r2]
  const int r1 = a == 0 ? 0 : a == 2 ? 2 : 1, r2 = a == 0 ? 2 : a == 1 ? 2 : a == 2 ? 1 : 3;
  const float s2 = a == 1 ? 1.f : -1.f;
  // and columns of t = B^T d: tx - ty, ty + sz tz (t0 - t2, t2 + t1; t2 - t1, t1 - t3)
  const int PW = g.TW + 1, PP = PS >> 2;               // plane row, plane
  const int cx = bp, cy = bp ? PP : 1, cz = bp ? 1 + PP : PP;
  const float sz = bp ? -1.f : 1.f;
  // window of the lane's tiles, channel 8 lk, row r1, column 0
  int win[2];
#pragma unroll
  for (int th = 0; th < 2; ++th) {
    int n, ty, tx;
    tile_at(th, n, ty, tx);
    const int row = n == nfirst ? 2 * ty - g.PT - rlo0 : rows0 + (n - nfirst - 1) * SR + 2 * ty;   // even
    win[th] = (row >> 1) * PW + tx + lk * 8 * WINO_X3_PSTR + (r1 & 1) * 2 * PP + (r1 >> 1) * PW;
  }
  const float iPW = __builtin_amdgcn_rcpf((float)PW), iPP = __builtin_amdgcn_rcpf((float)PP);
  const int drow = ((r2 & 1) - (r1 & 1)) * 2 * PP + ((r2 >> 1) - (r1 >> 1)) * PW;
  // byte offset (channel 0) of each patch position, or kOutside: the same for
  // every channel, kept in LDS
  for (int e = tid; e < PL * 64; e += WINO_X3_NT) {
    const int pl = wino_div(e, PP, iPP), f = e - pl * PP;
    const int qh = wino_div(f, PW, iPW);
    const int q = 2 * qh + (pl >> 1), col = 2 * (f - qh * PW) + (pl & 1);
    int sg = 0, row = rlo0 + q;
    if (q >= rows0) {
      const int R = q - rows0;
      const int s1 = wino_div(R, SR, iSR);
      sg = 1 + s1;
      row = R - s1 * SR - g.PT;
    }
    const int ix = col - g.PL;
    const bool ok = e < PS && (unsigned)row < (unsigned)g.H && (unsigned)ix < (unsigned)g.W;
    poff[e] = ok ? ((nfirst + sg) * g.C * HW + row * g.W + ix) * 4 : kOutside;
  }
  __syncthreads();
  const int xbytes = g.N * g.C * HW * 4;
  // loads [i0, i1) of the wave's 2 PL of a chunk's patch (channels `wave` and
  // `wave` + 8), straight to LDS; positions outside the image and channels past
  // the last read as zeros
  auto load_x = [&](int chunk, float* patch, int i0, int i1) {
#pragma unroll
    for (int part = 0; part < 2; ++part) {
      const int c = chunk * 16 + wave + 8 * part;
      const __amdgpu_buffer_rsrc_t r = buffer_over(g.x + (size_t)min(c, g.C - 1) * HW,
                                                   c < g.C ? xbytes - c * HW * 4 : 0);
#pragma unroll
      for (int i = 0; i < PL; ++i)
        if (part * PL + i >= i0 && part * PL + i < i1)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(
              r, (__attribute__((address_space(3))) void*)(patch + (wave + 8 * part) * WINO_X3_PSTR + i * 64), 4,
              poff[i * 64 + lane], 0, 0, 0);
    }
  };
  struct Operand { uintx4_t v[2][3]; };               // B operands of a tile half, [position][h, m, l]
  Operand va, vb;
  // channels 2 j, 2 j + 1 of a tile half: the window values, then the operands
  float raw[2][12];
  auto fetch = [&](const float* patch, int th, int j) {
    const float* at = patch + win[th] + 2 * j * WINO_X3_PSTR;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const float* p = at + e * WINO_X3_PSTR;
      float* x = raw[j & 1] + 6 * e;
      x[0] = p[cx];
      x[1] = p[drow + cx];
      x[2] = p[cy];
      x[3] = p[drow + cy];
      x[4] = p[cz];
      x[5] = p[drow + cz];
    }
  };
  auto transform = [&](int j, Operand& o) {
    float x[2][2];                                    // [position][channel]
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const float* p = raw[j & 1] + 6 * e;
      const float tx = __builtin_fmaf(s2, p[1], p[0]);
      const float ty = __builtin_fmaf(s2, p[3], p[2]);
      const float tz = __builtin_fmaf(s2, p[5], p[4]);
      x[0][e] = tx - ty;
      x[1][e] = __builtin_fmaf(sz, tz, ty);
    }
#pragma unroll
    for (int pos = 0; pos < 2; ++pos) split_bf16x3_pair(x[pos][0], x[pos][1], o.v[pos], j);
  };

  floatx16 acc[2][2][2];                              // [position][channel block][tile half]
#pragma unroll
  for (int pos = 0; pos < 2; ++pos)
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int th = 0; th < 2; ++th)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[pos][k][th][r] = 0.f;
  // half h of a position's twelve products
  auto multiply = [&](int pos, int th, int h, const Operand& o) {
    constexpr int PA[6] = {2, 1, 1, 0, 0, 0}, PB[6] = {0, 1, 0, 2, 1, 0};
#pragma unroll
    for (int q = 3 * h; q < 3 * h + 3; ++q)
#pragma unroll
      for (int blk = 0; blk < 2; ++blk)
        acc[pos][blk][th] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            u[pos][blk][PA[q]], __builtin_bit_cast(bf16x8_t, o.v[pos][PB[q]]), acc[pos][blk][th], 0, 0, 0);
  };

  // ---- chunks ---------------------------------------------------------------------
  // Eight regions a chunk, each six MFMAs interleaved with the transform of two
  // channels of the tile half after (of the next chunk in regions 4 - 7) and the
  // LDS reads of the two after these. Before region 3, the first that reads the
  // next chunk's patch, the barrier: that patch has arrived, and nothing reads
  // this chunk's any more.
  constexpr int X0 = 2 * PL * 5 / 16, X1 = 2 * PL * 10 / 16, X2 = 2 * PL * 13 / 16;
  load_x(chunk0, p0, 0, 2 * PL);
  load_x(chunk0 + min(1, nch - 1), p1, 0, X2);
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(X2) : "memory");
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    fetch(p0, 0, j);
    transform(j, va);
  }
  fetch(p0, 1, 0);
  auto weave = [&](int vmem) {
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);   // MFMA
      __builtin_amdgcn_sched_group_barrier(0x2, 6, 0);   // vector instructions
      __builtin_amdgcn_sched_group_barrier(0x100, 3, 0); // LDS reads
      if (k > 0 && k <= vmem) __builtin_amdgcn_sched_group_barrier(0x10, 1, 0);
      if (k > 0 && k + 5 <= vmem) __builtin_amdgcn_sched_group_barrier(0x10, 1, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto step = [&](int c, float* cur, float* next) {
    // past the last chunk: that chunk again (nothing branches)
    const int c1 = chunk0 + min(c + 1, nch - 1), c2 = chunk0 + min(c + 2, nch - 1), c0 = chunk0 + min(c, nch - 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      if (r == 3) asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
      const int j = r & 3;
      if (r == 0) {
        load_x(c1, next, X2, 2 * PL);
        load_u(c0, 1, 0);
      } else if (r == 3) {
        load_x(c2, cur, 0, X0);
      } else if (r == 4) {
        load_x(c2, cur, X0, X1);
      } else if (r == 6) {
        load_x(c2, cur, X1, X2);
        load_u(c1, 0, 0);
      }
      if (r < 3) fetch(cur, 1, j + 1);
      if (r >= 3 && r < 7) fetch(next, 0, r - 3);
      if (r == 7) fetch(next, 1, 0);
      if (r < 4) {
        transform(j, vb);
        multiply(j >> 1, 0, j & 1, va);
      } else {
        transform(j, va);
        multiply(j >> 1, 1, j & 1, vb);
      }
      if (r == 5 || r == 7) {
        load_u(c1, j >> 1, 2);
        load_u(c1, j >> 1, 1);
      }
      weave(r == 0 ? 2 * PL - X2 + 2 : r == 3 || r == 4 ? X0 : r == 6 ? X2 - X1 + 2 : r == 5 || r == 7 ? 4 : 0);
    }
  };
  for (int c = 0; c < nch; c += 2) {
    step(c, p0, p1);
    if (c + 1 < nch) step(c + 1, p1, p0);
  }
  // the loads past the last chunk land in the patches, which other waves reuse
  // after the next barrier
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  // ---- output transform, a tile half at a time -------------------------------------
  // A wave writes its positions' sums to [xi][r group][lane], four channels a
  // float4. Wave f then finishes channels 8 (f & 3) + 4 lk + 0 .. 3 of pixel row
  // i = f >> 2, both columns: Y = A^T M A, A^T = (1 1 1 0; 0 1 -1 -1), M's signs
  // undone: (1 -1 1 0; 0 -1 -1 1) on rows, (1 1 -1 0; 0 1 1 -1) on columns.
  const int OHW = g.OH * g.OW;
  const int ocs = SPLIT ? g.N * OHW : OHW;            // stride between channels
  const int rq = wave & 3, i = wave >> 2;
  const float sg = i == 0 ? 1.f : -1.f;                 // sign of the first row
  const int oc0 = ocb * 64 + 8 * rq + 4 * lk;   // the lane's first channel of block 0
  int obase[2];                                       // byte offset of the lane's pixels, channel 0, or kOutside
  bool xok[2];
#pragma unroll
  for (int th = 0; th < 2; ++th) {
    int n, ty, tx;
    tile_at(th, n, ty, tx);
    const bool ok = t0 + 32 * th + li < P && (FULL || 2 * ty + i < g.OH);
    obase[th] = ok ? ((SPLIT ? n : n * g.OC) * OHW + (2 * ty + i) * g.OW + 2 * tx) * 4 : kOutside;
    xok[th] = FULL || 2 * tx + 1 < g.OW;
  }
  // bias and residual before any store: a load after a store waits for it
  float bv[2][4] = {};
  float2 rv[2][2][4] = {};                            // [th][k][channel]
  if (!SPLIT) {
    if (Epi::bias == 1) {
      const __amdgpu_buffer_rsrc_t rbias = buffer_over(g.bias, g.OC * 4);
#pragma unroll
      for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          bv[k][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rbias, (oc0 + 32 * k + e) * 4, 0, 0));
    }
    if (Epi::residual) {
      const __amdgpu_buffer_rsrc_t rres = buffer_over(g.R, g.N * g.OC * OHW * 4);
#pragma unroll
      for (int th = 0; th < 2; ++th)
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int oc = oc0 + 32 * k + e;
            const int o = obase[th] != kOutside && oc < g.OC ? obase[th] + oc * OHW * 4 : kOutside;
            if (FULL) {
              rv[th][k][e] = __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(rres, o, 0, 0));
            } else {
              rv[th][k][e].x = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rres, o, 0, 0));
              rv[th][k][e].y = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                  rres, o != kOutside && xok[th] ? o + 4 : kOutside, 0, 0));
            }
          }
    }
  }
  const __amdgpu_buffer_rsrc_t rout =
      buffer_over(g.y + (SPLIT ? (size_t)slice * g.OC * g.N * OHW : 0), g.OC * g.N * OHW * 4);
  // sums of position xi, channel block k: [r group][lane] of 4 KB in ex, or where
  // the patches were
  auto sums = [&](int xi, int k) { return k == 0 ? ex + xi * 1024 : xi < 8 ? p0 + xi * 1024 : p1 + (xi - 8) * 1024; };
#pragma unroll
  for (int th = 0; th < 2; ++th) {
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int pos = 0; pos < 2; ++pos)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const floatx16& s = acc[pos][k][th];
          st4(sums(2 * wave + pos, k) + q * 256 + lane * 4,
              make_float4(s[4 * q], s[4 * q + 1], s[4 * q + 2], s[4 * q + 3]));
        }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      float2 o[4];                                    // [channel], both pixel columns
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        floatx4 m[4];
#pragma unroll
        for (int q = 0; q < 4; ++q)
          m[q] = *reinterpret_cast<const floatx4*>(sums((i + r) * 4 + q, k) + rq * 256 + lane * 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float y0 = m[0][e] + m[1][e] - m[2][e], y1 = m[1][e] + m[2][e] - m[3][e];
          if (r == 0) {
            o[e] = make_float2(sg * y0, sg * y1);
          } else if (r == 1) {
            o[e] = make_float2(o[e].x - y0, o[e].y - y1);
          } else {
            o[e] = make_float2(o[e].x + y0, o[e].y + y1);
          }
        }
      }
      float z = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) z += o[e].x * 0.f + o[e].y * 0.f;
      if (__any(z != 0.f) && z != 0.f && obase[th] != kOutside) {
        int n, ty, tx;
        tile_at(th, n, ty, tx);
#pragma unroll 1
        for (int q = 0; q < 8; ++q) {                 // one copy of the loops: o by selects
          const int oc = oc0 + 32 * k + (q >> 1);
          float old = 0.f;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            old = q == 2 * e ? o[e].x : old;
            old = q == 2 * e + 1 ? o[e].y : old;
          }
          if (old * 0.f == 0.f || oc >= g.OC) continue;
          const float w1 = wino_x3_slow(g, ublk, chunk0 * 16, min(g.C, (chunk0 + nch) * 16), oc & 63, n,
                                        2 * ty - g.PT, 2 * tx - g.PL, i, q & 1);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            o[e].x = q == 2 * e ? w1 : o[e].x;
            o[e].y = q == 2 * e + 1 ? w1 : o[e].y;
          }
        }
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int oc = oc0 + 32 * k + e;
        if (!SPLIT) {
          o[e].x = Epi::apply(o[e].x, bv[k][e]);
          o[e].y = Epi::apply(o[e].y, bv[k][e]);
          if (Epi::residual) {
            o[e].x = Epi::post(o[e].x, rv[th][k][e].x);
            o[e].y = Epi::post(o[e].y, rv[th][k][e].y);
          }
        }
        const int at = obase[th] != kOutside && oc < g.OC ? obase[th] + oc * ocs * 4 : kOutside;
        if (FULL) {
          __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(v2u32_t, o[e]), rout, at, 0, 0);
        } else {
          __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, o[e].x), rout, at, 0, 0);
          __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, o[e].y), rout,
                                                at != kOutside && xok[th] ? at + 4 : kOutside, 0, 0);
        }
      }
    }
  }
}

}  // namespace mdlc
