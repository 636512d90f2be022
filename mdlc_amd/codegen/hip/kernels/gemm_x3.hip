// Dense fp32 GEMM on the bf16 matrix cores, each fp32 operand split into three
// bf16 terms (conv_x3.hip is the convolution).
//
//   C = epi(A[M x K] * B[K x N], bias)
//
// v_mfma_f32_32x32x16_bf16 does 16 times the multiply-adds per cycle of
// v_mfma_f32_32x32x2_f32. A float is the exact sum of three bf16 values,
// x = h + m + l (h = bf16(x), m = bf16(x - h), l = x - h - m, each rounded to
// nearest: 8 + 8 + 8 significand bits), so a product of two floats is the sum
// of nine bf16 products, each exact in fp32. Six of them are accumulated
// (in fp32, smallest first: l h, h l, m m, m h, h m, h h); the other three
// (m l, l m, l l) are below 2^-25 of the product, under half a unit in the
// last place of the float it would be rounded to. Measured against 64 bits
// the result is closer than the fp32 instruction's (which rounds the
// accumulator eight times where this rounds it six times), at 16 / 6 = 2.7
// times its peak rate.
//
// The split needs finite operands: an infinity splits into inf + NaN, and a
// float within half a bf16 ulp of FLT_MAX rounds its h to infinity. Either
// leaves a NaN or an infinity in the accumulators, so a wave that finds one
// there recomputes its tile with plain fp32 fmas: infinities, NaNs
// and overflow come out as the fp32 kernel gives them. Operands below 2^-102
// may lose the bits of m and l under 2^-126.
//
// B is a constant, split and packed on the host as [32-column block][16-deep k
// step][h, m, l][lane][8 bf16] in the instruction's lane order (lane = 32 *
// (k % 16 / 8) + column % 32), so its tiles are copied into LDS as they are:
// through registers two stages ahead, or (DMA) by loads straight to LDS one
// stage ahead, where a wave's 64 x 128 tile leaves no registers. A is fp32 rows
// of depth lda; the thread that stages eight k of a row splits them, 5.5
// vector instructions an element between the MFMAs, into three 16-byte LDS
// writes. K is the depth B is packed to (zeros past A's).
//
// Tiling: WGM x WGN waves, each with MI x NI blocks of 32x32. LDS holds two
// stages of KST k steps.
//
// Measured (fused bias + ReLU): 4096^3 1067 -> 607 us (256 x 256 tiles, 1.36
// PFLOP/s of bf16, what a plain bf16 product of that size reaches here; the
// chip's power holds the clock near 1.9 GHz), error against 64 bits 1.1e-6 ->
// 1.0e-6; 1000 x 1511 x 777 33.3 -> 25.4 us (64 x 64 tiles, two slices: vector,
// LDS and matrix work of a 32-deep step take about 400 cycles each and barely
// overlap in so small a tile), error 3.5e-7 -> 1.2e-7; 16 x 333 x 1000 17.1 ->
// 7.3 us.
namespace mdlc {

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float floatx2_t __attribute__((ext_vector_type(2)));
typedef unsigned uintx4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ unsigned cvt_bf16_pair(float a, float b) {
  const floatx2_t v = {a, b};
  return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2_t));
}

// eight floats -> three vectors of eight bf16: h, m, l. Eleven instructions a
// pair, all of which run beside MFMAs. (v_dot2_f32_bf16 with {-1, 0} subtracts a
// half of a pair without unpacking it, seven instructions, but waits for the
// matrix cores: four of them between MFMAs cost 12 ns, four additions 1 ns.
// 4096^3 612 -> 590 us with the additions.)
__device__ __forceinline__ void split_bf16x3_pair(float a, float b, uintx4_t (&p)[3], int j) {
#pragma unroll
  for (int t = 0; t < 3; ++t) {
    const unsigned w = cvt_bf16_pair(a, b);
    p[t][j] = w;
    if (t < 2) {
      a -= __builtin_bit_cast(float, w << 16);
      b -= __builtin_bit_cast(float, w & 0xffff0000u);
    }
  }
}

__device__ __forceinline__ void split_bf16x3(const float (&x)[8], uintx4_t (&p)[3]) {
#pragma unroll
  for (int j = 0; j < 4; ++j) split_bf16x3_pair(x[2 * j], x[2 * j + 1], p, j);
}

// element (row, k) of a packed constant: h + m + l, the original float
__device__ __forceinline__ float x3_weight(const float* img, int ksteps, int row, int k) {
  const unsigned short* p = reinterpret_cast<const unsigned short*>(img) +
                            (size_t)((row >> 5) * ksteps + (k >> 4)) * 1536 +
                            ((k >> 3 & 1) * 32 + (row & 31)) * 8 + (k & 7);
  const float h = __builtin_bit_cast(float, (unsigned)p[0] << 16);
  const float m = __builtin_bit_cast(float, (unsigned)p[512] << 16);
  const float l = __builtin_bit_cast(float, (unsigned)p[1024] << 16);
  return h + (m + l);                             // exact in this order, also next to FLT_MAX
}

// The epilogue of one tile, like gemm_f32_store's, through buffer resources:
// a row past M or a column past N gets an offset out of range, which reads
// zero and drops the store, so nothing branches.
template <int BM, int BN, int WGM, int WGN, int OUT, class Epi, class Acc>
__device__ __forceinline__ void x3_store(const GemmArgs& g, const Acc& acc, int m0, int n0, int ks) {
  constexpr int WM = BM / WGM, WN = BN / WGN;
  constexpr int MI = WM / 32, NI = WN / 32;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 31, lk = lane >> 5;
  const int mw = m0 + (wave / WGN) * WM, nw = n0 + (wave % WGN) * WN;
  const int rs = OUT == 2 ? g.N : OUT == 1 ? g.hw : g.ldc;     // stride between rows
  const int row0 = mw + lk * 4;
  const int nbytes = OUT == 1 ? g.N / g.hw * g.cimg * 4 : ((g.M - 1) * rs + g.N) * 4;
  const __amdgpu_buffer_rsrc_t rC = buffer_over(g.C + (OUT == 2 ? (size_t)ks * g.M * g.N : 0), nbytes);
  const bool full = mw + WM <= g.M;
  int off[NI];
#pragma unroll
  for (int ni = 0; ni < NI; ++ni) {
    const int col = nw + ni * 32 + li;
    int o = col;
    if (OUT == 1) {
      const int n = col / g.hw;
      o = n * g.cimg + (col - n * g.hw);
    }
    off[ni] = col < g.N ? (o + row0 * rs) * 4 : kOutside;
  }
  float4 brow[MI][4];
  float bcol[NI];
  float rv[NI][MI][16];
  if (OUT != 2) {
    const __amdgpu_buffer_rsrc_t rb = buffer_over(g.bias, Epi::bias == 0 ? 0 : (Epi::bias == 1 ? g.M : g.N) * 4);
    if (Epi::bias == 1) {
#pragma unroll
      for (int mi = 0; mi < MI; ++mi)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          brow[mi][q] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(
              rb, (row0 + mi * 32 + q * 8) * 4, 0, 0));
    }
#pragma unroll
    for (int ni = 0; ni < NI; ++ni)
      bcol[ni] = Epi::bias == 2 ? __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                      rb, (nw + ni * 32 + li) * 4, 0, 0)) : 0.f;
    if (Epi::residual) {
      const __amdgpu_buffer_rsrc_t rR = buffer_over(g.R, nbytes);
#pragma unroll
      for (int ni = 0; ni < NI; ++ni)
#pragma unroll
        for (int mi = 0; mi < MI; ++mi)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int dr = mi * 32 + (r / 4) * 8 + r % 4;
            rv[ni][mi][r] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                rR, full || row0 + dr < g.M ? off[ni] : kOutside, dr * rs * 4, 0));
          }
    }
  }
#pragma unroll
  for (int ni = 0; ni < NI; ++ni)
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int dr = mi * 32 + (r / 4) * 8 + r % 4;
        float v = acc[mi][ni][r];
        if (OUT != 2) {
          v = Epi::apply(v, Epi::bias == 1 ? pick(brow[mi][r / 4], r % 4) : bcol[ni]);
          if (Epi::residual) v = Epi::post(v, rv[ni][mi][r]);
        }
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), rC,
                                              full || row0 + dr < g.M ? off[ni] : kOutside, dr * rs * 4, 0);
      }
}

// Scheduling hints of a stage, as compile-time recursion (their arguments must
// be constants): per k step its LDS reads, then its MFMAs each followed by VM
// vector instructions.
template <int I, int KST, int MF, int RD, int VM>
struct X3Order {
  __device__ __forceinline__ static void emit() {
    if constexpr (I < KST * MF) {
      if constexpr (I == 0) __builtin_amdgcn_sched_group_barrier(0x100, KST * RD, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, VM, 0);
      X3Order<I + 1, KST, MF, RD, VM>::emit();
    }
  }
};

// V4: A's depth is a multiple of 4 (its rows are read as aligned float4).
template <int BM, int BN, int KST, int WGM, int WGN, bool DMA, bool V4, int OUT, class Epi>
__device__ __forceinline__ void gemm_x3(const GemmArgs& g) {
  constexpr int NT = WGM * WGN * 64, NW = WGM * WGN;
  constexpr int WM = BM / WGM, WN = BN / WGN;
  constexpr int MI = WM / 32, NI = WN / 32;
  constexpr int BK = 16 * KST;
  constexpr int CPT = 2 * KST;                    // 8-deep chunks of k per row and stage
  constexpr int XPT = BM * CPT / NT;              // chunks a thread splits per stage
  constexpr int WPC = BN / 32 * KST * 3;          // 1 KB pieces of the constant per stage
  constexpr int WPT = (WPC + NW - 1) / NW;        // and per wave
  constexpr int XB = BM * BK * 6, WB = BN * BK * 6;
  constexpr bool DUAL = MI * NI <= 4;             // registers for a second accumulator
  static_assert(WM % 32 == 0 && WN % 32 == 0, "wave tile must be a multiple of the MFMA");
  static_assert(BM * CPT % NT == 0, "A's chunks must cover the workgroup evenly");
  // two stages, as separate arrays so that the compiler knows one's writes
  // from the other's reads
  __shared__ __attribute__((aligned(1024))) char xs0[XB], xs1[XB], ws0[WB], ws1[WB];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm0 = (wave / WGN) * WM, wn0 = (wave % WGN) * WN;
  const int li = lane & 31, lk = lane >> 5;

  const int tiles_m = (g.M + BM - 1) / BM;
  const int tiles_n = (g.N + BN - 1) / BN;
  const int tiles = tiles_m * tiles_n;
  const int t = xcd_remap(blockIdx.x, tiles * g.ksplit);
  const int ks = t / tiles;
  int mt, nt;
  grouped_tile<8>(t - ks * tiles, tiles_m, tiles_n, mt, nt);
  const int m0 = mt * BM, n0 = nt * BN;
  // K steps of this slice: g.K is the padded depth (a multiple of 16) the
  // constant is packed to, g.kchunk a multiple of BK
  const int ksteps = g.K >> 4;
  const int kbeg = ks * g.kchunk, kend = min(g.K, kbeg + g.kchunk);
  const int nk = (kend - kbeg + BK - 1) / BK;

  // ---- the packed constant: its 1 KB pieces [row block][k step][h, m, l] of
  // a stage. Row blocks past the constant repeat its last one (their rows are
  // never stored), k steps past K read zeros. ----------------------------------
  const int wblocks = (g.N + 31) >> 5;
  const __amdgpu_buffer_rsrc_t rsW = buffer_over(g.B, wblocks * ksteps * 3072);
  int w_off[WPT], w_step[WPT];
#pragma unroll
  for (int i = 0; i < WPT; ++i) {
    const int j = wave + i * NW, rb = j / (3 * KST), r = j - rb * (3 * KST);
    w_step[i] = r / 3;
    w_off[i] = (min((n0 >> 5) + rb, wblocks - 1) * ksteps + r / 3) * 3072 + (r % 3) * 1024;
  }
  auto w_at = [&](int i, int k0) {                // byte offset of the lane's 16 bytes of piece i
    const int step = k0 >> 4;
    return step + w_step[i] < ksteps ? w_off[i] + step * 3072 + lane * 16 : kOutside;
  };
  auto dma_w = [&](int k0, char* ws) {
#pragma unroll
    for (int i = 0; i < WPT; ++i)
      if (WPC % NW == 0 || wave + i * NW < WPC)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            rsW, (__attribute__((address_space(3))) void*)(ws + (wave + i * NW) * 1024), 16, w_at(i, k0), 0, 0, 0);
  };

  // ---- A: chunk q = tid + i * NT of a stage, CPT chunks a row ---------------
  int x_off[XPT], x_lds[XPT], x_k[XPT];
  const __amdgpu_buffer_rsrc_t rsX = buffer_over(g.A, g.M * g.lda * 4);
#pragma unroll
  for (int i = 0; i < XPT; ++i) {
    const int q = tid + i * NT, c = q % CPT, r = q / CPT;
    // consecutive threads hold a row's chunks: rows are permuted by the chunk
    // so that their writes (and any 16 lanes' reads) hit distinct banks
    x_lds[i] = ((r >> 5) * KST + (c >> 1)) * 3072 + ((c & 1) * 32 + ((r & 31) ^ ((c & 3) << 2))) * 16;
    x_k[i] = c * 8;
    x_off[i] = m0 + r < g.M ? ((m0 + r) * g.lda + c * 8) * 4 : kOutside;
  }

  // One stage in registers: the loads of stage k0 (called for every stage in
  // order), then its splits and LDS writes.
  struct Stage {
    float x[XPT][8];
    uintx4_t w[DMA ? 1 : WPT];
  };
  auto load = [&](int k0, Stage& st) {
    if (!DMA) {
#pragma unroll
      for (int i = 0; i < WPT; ++i)
        if (WPC % NW == 0 || wave + i * NW < WPC)
          st.w[i] = __builtin_bit_cast(uintx4_t, __builtin_amdgcn_raw_buffer_load_b128(rsW, w_at(i, k0), 0, 0));
    }
#pragma unroll
    for (int i = 0; i < XPT; ++i) {
      const int k = k0 + x_k[i];
      const int off = x_off[i] + k0 * 4;
      const bool in = x_off[i] != kOutside;
      if (V4 || k0 + BK <= g.lda) {
        // 16-byte loads, dword aligned; with V4 a quad lies inside the row or past it
#pragma unroll
        for (int j = 0; j < 8; j += 4) {
          const float4 v = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(
              rsX, in && (!V4 || k + j < g.lda) ? off + j * 4 : kOutside, 0, 0));
          st.x[i][j] = v.x; st.x[i][j + 1] = v.y; st.x[i][j + 2] = v.z; st.x[i][j + 3] = v.w;
        }
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j)
          st.x[i][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
              rsX, in && k + j < g.lda ? off + j * 4 : kOutside, 0, 0));
      }
    }
  };
  auto store = [&](char* xs, char* ws, const Stage& st) {
    if (!DMA) {
#pragma unroll
      for (int i = 0; i < WPT; ++i)
        if (WPC % NW == 0 || wave + i * NW < WPC)
          *reinterpret_cast<uintx4_t*>(ws + (wave + i * NW) * 1024 + lane * 16) = st.w[i];
    }
#pragma unroll
    for (int i = 0; i < XPT; ++i) {
      uintx4_t p[3];
      split_bf16x3(st.x[i], p);
#pragma unroll
      for (int q = 0; q < 3; ++q) *reinterpret_cast<uintx4_t*>(xs + x_lds[i] + q * 1024) = p[q];
    }
  };

  // acc[0]: the h h products (and all the others without a second
  // accumulator), acc[1]: the five small ones, whose roundings are then
  // 2^-8 of the result's
  floatx16 acc[DUAL ? 2 : 1][MI][NI];
#pragma unroll
  for (int d = 0; d < (DUAL ? 2 : 1); ++d)
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
      for (int ni = 0; ni < NI; ++ni)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[d][mi][ni][r] = 0.f;

  auto compute = [&](const char* xs, const char* ws) {
#pragma unroll
    for (int s = 0; s < KST; ++s) {
      const int plain = lane * 16;
      const int swz = (lk * 32 + (li ^ (((2 * s + lk) & 3) << 2))) * 16;
      bf16x8_t a[MI][3], b[NI][3];
#pragma unroll
      for (int q = 0; q < 3; ++q) {
#pragma unroll
        for (int mi = 0; mi < MI; ++mi)
          a[mi][q] = *reinterpret_cast<const bf16x8_t*>(
              xs + ((wm0 / 32 + mi) * KST + s) * 3072 + q * 1024 + swz);
#pragma unroll
        for (int ni = 0; ni < NI; ++ni)
          b[ni][q] = *reinterpret_cast<const bf16x8_t*>(
              ws + ((wn0 / 32 + ni) * KST + s) * 3072 + q * 1024 + plain);
      }
      constexpr int PA[6] = {2, 0, 1, 1, 0, 0}, PB[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
      for (int p = 0; p < 6; ++p)
#pragma unroll
        for (int mi = 0; mi < MI; ++mi)
#pragma unroll
          for (int ni = 0; ni < NI; ++ni) {
            floatx16& c = acc[DUAL && p < 5 ? 1 : 0][mi][ni];
            c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[mi][PA[p]], b[ni][PB[p]], c, 0, 0, 0);
          }
    }
  };

  // the MFMAs of the stage in (xs, ws), the splits of stage st between them
  // into (xt, wt)
  auto step = [&](const char* xs, const char* ws, char* xt, char* wt, const Stage& st) {
    __builtin_amdgcn_sched_barrier(0);
    compute(xs, ws);
    store(xt, wt, st);
    constexpr int MF = MI * NI * 6;               // MFMAs per k step
    constexpr int VM = (XPT * 48 + MF * KST - 1) / (MF * KST);   // vector instructions after each
    X3Order<0, KST, MF, (MI + NI) * 3, VM>::emit();
    __builtin_amdgcn_sched_barrier(0);
    if (DMA) __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): the constant's pieces are in LDS
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
  };

  if (DMA) {
    Stage st;
    dma_w(kbeg, ws0);
    load(kbeg, st);
    store(xs0, ws0, st);
    __builtin_amdgcn_s_waitcnt(0x0f70);
    __syncthreads();
    int kt = 0;
    for (; kt + 2 <= nk; kt += 2) {
      dma_w(kbeg + (kt + 1) * BK, ws1);
      load(kbeg + (kt + 1) * BK, st);
      step(xs0, ws0, xs1, ws1, st);
      dma_w(kbeg + (kt + 2) * BK, ws0);
      load(kbeg + (kt + 2) * BK, st);
      step(xs1, ws1, xs0, ws0, st);
    }
    if (kt < nk) compute(xs0, ws0);
  } else {
    // two stages of loads in flight; loads past the slice are stored to a
    // stage nobody reads
    Stage s0, s1;
    load(kbeg, s0);
    load(kbeg + BK, s1);
    store(xs0, ws0, s0);
    __syncthreads();
    int kt = 0;
    for (; kt + 2 <= nk; kt += 2) {
      load(kbeg + (kt + 2) * BK, s0);
      step(xs0, ws0, xs1, ws1, s1);
      load(kbeg + (kt + 3) * BK, s1);
      step(xs1, ws1, xs0, ws0, s0);
    }
    if (kt < nk) compute(xs0, ws0);
  }

  // a NaN or an infinity anywhere in the wave's tile: v * 0 is then NaN
  float z = 0.f;
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int ni = 0; ni < NI; ++ni)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        if (DUAL) acc[0][mi][ni][r] += acc[1][mi][ni][r];
        z += acc[0][mi][ni][r] * 0.f;
      }
  if (__any(z != 0.f)) {
    for (int e = lane; e < WM * WN; e += 64) {
      const int row = m0 + wm0 + e / WN, col = n0 + wn0 + e % WN;
      if (row >= g.M || col >= g.N) continue;
      float v = 0.f;
      for (int k = kbeg; k < min(kend, g.lda); ++k)
        v = __builtin_fmaf(g.A[(size_t)row * g.lda + k], x3_weight(g.B, ksteps, col, k), v);
      if (OUT == 2) {
        g.C[((size_t)ks * g.M + row) * g.N + col] = v;
      } else {
        g.C[(size_t)row * g.ldc + col] = Epi::apply(v, Epi::bias == 2 ? g.bias[col] : 0.f);
      }
    }
    return;
  }
  x3_store<BM, BN, WGM, WGN, OUT, Epi>(g, acc[0], m0, n0, ks);
}

}  // namespace mdlc
