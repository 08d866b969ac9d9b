// Cell-stationary kernels of the pair grid: every wave owns 32 cells for a whole tile and keeps
// their LayerNormed channels in registers as MFMA fragments, while the weights stream past all
// waves of the workgroup through LDS. Nothing of a tile but its inputs and its outputs touches
// memory.
#include "common.h"
#include "kernels.h"

namespace esm {

namespace {
constexpr int kCsWaves = 8;                  // two per SIMD: one's VALU work runs under the other's MFMAs
constexpr int kCsThreads = 64 * kCsWaves;
constexpr int kEmWaves = 4;                  // of the kernels that run two workgroups per CU
constexpr int kCsCells = 32;                 // cells per wave: the columns of one 32x32x16 MFMA

// Sum over the N = 16 or 32 aligned lanes of a group; every lane gets it.
template <int N>
DEV float lane_sum(float v) {
  static_assert(N == 16 || N == 32, "one or two DPP rows");
  v = row16_sum(v);
  if constexpr (N == 32) {
    const auto w = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(w[0]) + __uint_as_float(w[1]);
  }
  return v;
}
// Ends a value's live range in other forms: the next use starts from these registers.
DEV void pin(half8& v) { __asm__ volatile("" : "+v"(v)); }
// The lane number, formed anew at each use: where the registers are full, addresses are computed from it
// instead of being kept.
DEV int fresh_lane() {
  int l;
  __asm__ volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
  return l;
}
// LayerNorm in place of a wave's 32 cells in LDS (rows of C halfs, 16-byte piece j of cell c at
// j ^ (c % (C / 8))), two-pass fp32 statistics, 1 KB at a time in a rolled loop: straight-line code that
// runs once per tile is bound by its instruction fetches (unrolled, staging and LayerNorm took 36 us
// of a launch at one tile per CU instead of 20).
template <int C>
DEV void ln_rows_lds(char* zs, const float* w, const float* b, float eps) {
  constexpr int LPC = C / 8, CPI = 64 / LPC;  // lanes per cell, cells per KB
  const int l = fresh_lane(), l0 = l & (LPC - 1), cl = l / LPC;
  float g[8], bb[8];
#pragma unroll
  for (int e = 0; e < 8; e++) {
    g[e] = w[8 * l0 + e];
    bb[e] = b[8 * l0 + e];
  }
#pragma unroll 4
  for (int i = 0; i < kCsCells / CPI; i++) {
    char* piece = zs + i * 1024 + cl * (2 * C) + 16 * (l0 ^ ((i * CPI + cl) & (LPC - 1)));
    const half8 x = *reinterpret_cast<const half8*>(piece);
    const half2v one = {(half_t)1.0f, (half_t)1.0f};
    const float s0 = __builtin_amdgcn_fdot2(half2v{x[2], x[3]}, one,
                                            __builtin_amdgcn_fdot2(half2v{x[0], x[1]}, one, 0.f, false), false);
    const float s1 = __builtin_amdgcn_fdot2(half2v{x[6], x[7]}, one,
                                            __builtin_amdgcn_fdot2(half2v{x[4], x[5]}, one, 0.f, false), false);
    const float mean = lane_sum<LPC>(s0 + s1) * (1.0f / C);
    float q0 = 0.f, q1 = 0.f, d[8];
#pragma unroll
    for (int e = 0; e < 8; e++) d[e] = (float)x[e] - mean;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      q0 += d[e] * d[e];
      q1 += d[e + 4] * d[e + 4];
    }
    const float rstd = rsqrtf(lane_sum<LPC>(q0 + q1) * (1.0f / C) + eps);
    half8 v;
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = (half_t)(d[e] * rstd * g[e] + bb[e]);
    *reinterpret_cast<half8*>(piece) = v;
  }
}
// The rows' MFMA fragments: channels 16 k + 8 (lane / 32) .. + 7 of cell lane % 32.
template <int C>
DEV void rows_to_frags(const char* zs, half8 (&f)[C / 16]) {
  const int l = fresh_lane();
#pragma unroll
  for (int k = 0; k < C / 16; k++)
    f[k] = *reinterpret_cast<const half8*>(zs + (l & 31) * (2 * C) + 16 * ((2 * k + (l >> 5)) ^ (l & (C / 8 - 1))));
#pragma unroll
  for (int k = 0; k < C / 16; k++) pin(f[k]);
}
// The rows' accumulator pieces: channels 4 j2 + 0..3 with j2 = 2 (4 ob + q) + lane / 32, as the 32x32
// MFMA leaves rows 8 q + 4 (lane / 32) + 0..3 of output block ob for cell lane % 32.
template <int C>
DEV char* acc_piece(char* zs, int l, int ob, int q) {
  return zs + (l & 31) * (2 * C) + 8 * (l >> 5) + 16 * ((4 * ob + q) ^ (l & (C / 8 - 1)));
}
DEV void cs_lds_fence() {  // a wave's own LDS operations complete in order: a compiler fence only
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
}  // namespace

// ---- transition: out = z + W3 act(W1 LN(z) [, W2 LN(z)]) ----------------------------------------
// One launch in place of a LayerNorm pass and two GEMMs with the hidden plane (4 z planes at
// H = 4 C) written and read between them. A wave's 32 cells are the columns of every product:
// LN(z) stays in 64 registers as the B operand of the first GEMM, its 32 hidden units per step
// become the B operand of the second one where they stand, and the output's 128 accumulators
// start as z. The weights (96 KB per 64 units) come from L2 once per 256 cells.
// Bound by the matrix cores' load: over a launch at L=476 they are busy in 44% of the cycles (32% at L=238, 222
// tiles on 256 CUs), at a clock below 1.8 GHz (2.2 in the contraction). C=256, H=1024, back to back: L=238
// SwiGLU 171 -> 100 us, ReLU 129 -> 69; L=476 655 -> 377 and 496 -> 261 (89 GFLOP at L=238: 0.89 PFLOP/s); a
// call among others 173 -> 92 at L=238, SwiGLU. What is not the loop (~20 us at one tile per CU): z's arrival,
// the LayerNorm, the stores.
template <int C, bool SWIGLU>
struct CsTransGeo {
  static constexpr int G = SWIGLU ? 2 : 1;             // matrices of the first GEMM
  static constexpr int W1B = 32 * C * 2;               // 32 hidden units of one of them
  static constexpr int W12B = G * W1B, W3B = C * 64;   // and of W3: C rows of 32 units
  static constexpr int OFF3 = 3 * W12B;                // three ring slots of each
  static constexpr int N12 = W12B / 1024 / kCsWaves, N3 = W3B / 1024 / kCsWaves;  // 1 KB loads per wave
  static constexpr int ZW = kCsCells * C * 2;          // a wave's cells
  static constexpr int OFFZ = W12B;                    // z rows lie behind ring slot 0 until they are fragments
  static constexpr int SMEM0 = OFF3 + 3 * W3B, SMEM1 = OFFZ + kCsWaves * ZW;
  static constexpr int SMEM = SMEM0 > SMEM1 ? SMEM0 : SMEM1;
  static_assert(SMEM <= 160 * 1024, "LDS");
  static_assert(W12B % (1024 * kCsWaves) == 0 && W3B % (1024 * kCsWaves) == 0, "whole loads per wave");
};

template <int C, bool SWIGLU>
__global__ __launch_bounds__(kCsThreads, 1) void transition_stream_kernel(TransitionArgs p) {
  using T = CsTransGeo<C, SWIGLU>;
  static_assert(C % 128 == 0 && C <= 256, "64 + 128 registers of LN(z) and outputs at C = 256");
  constexpr int KS = C / 16, OB = C / 32;
  __shared__ __align__(1024) char smem[T::SMEM];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t lds0 = lds_address(smem);
  const int H = p.H, U = H / 32;
  const dma_src_t r1 = dma_src(p.w1, (uint32_t)H * C * 2u);
  const dma_src_t r2 = dma_src(SWIGLU ? p.w2 : p.w1, (uint32_t)H * C * 2u);
  const dma_src_t r3 = dma_src(p.w3, (uint32_t)H * C * 2u);

  // Weight loads: 8 rows of 128 bytes (64 k) per instruction of W1 / W2, 16 rows of 64 bytes (32
  // units) of W3; the 16-byte pieces of a row XOR-swizzled so that a fragment read (32 rows, one
  // piece) covers the banks evenly.
  auto load12 = [&](int u) {
    const uint32_t s12 = lds0 + (u % 3) * T::W12B;
    constexpr int N1 = T::W1B / 1024;
    const int l = fresh_lane();
    const uint32_t l1 = (uint32_t)(l >> 3) * (C * 2), x1 = 16u * (uint32_t)((l & 7) ^ (l >> 4));
#pragma unroll
    for (int i = 0; i < T::N12; i++) {
      const int q = wave * T::N12 + i, m = q / N1, qm = q % N1, st = qm / 4, rq = qm % 4;
      dma16(m ? r2 : r1, s12 + q * 1024, l1 + (x1 ^ (64u * (rq & 1))), (uint32_t)(32 * u + 8 * rq) * (C * 2) + st * 128);
    }
  };
  auto load3 = [&](int u) {
    const uint32_t s3 = lds0 + T::OFF3 + (u % 3) * T::W3B;
    const int l = fresh_lane();
    const uint32_t l3 = (uint32_t)(l >> 2) * (uint32_t)H * 2u + 16u * ((l & 3) ^ (l >> 4));
#pragma unroll
    for (int i = 0; i < T::N3; i++) {
      const int q = wave * T::N3 + i;
      dma16(r3, s3 + q * 1024, l3, (uint32_t)(16 * q) * (uint32_t)H * 2u + 64u * u);
    }
  };

  for (int tile = blockIdx.x; tile < p.ntiles; tile += gridDim.x) {
    const size_t cell0 = ((size_t)tile * kCsWaves + wave) * kCsCells;  // this wave's first cell
    const long long left = (long long)p.ncells - (long long)cell0;
    const int nv = left < 0 ? 0 : left < kCsCells ? (int)left : kCsCells;   // its cells inside the grid
    char* zs = smem + T::OFFZ + wave * T::ZW;
    constexpr int LPC = C / 8, CPI = 64 / LPC, NKB = T::ZW / 1024;  // lanes per cell, cells per KB, KBs
    load12(0);

    // 1. The wave's z into its LDS rows, the 16-byte pieces of a row XOR-swizzled by its cell; the
    // accumulators start from it (the residual); LayerNorm in place; fragments.
    half8 nf[KS];
    f32x16 o[OB];
    {
      const dma_src_t dz = dma_src(p.z + (nv ? cell0 * C : 0), (uint32_t)nv * C * 2u);
      const int l = fresh_lane(), l0 = l & (LPC - 1), cl = l / LPC;
#pragma unroll 4
      for (int i = 0; i < NKB; i++) {
        const int c = i * CPI + cl;
        dma16(dz, lds0 + (uint32_t)(zs - smem) + i * 1024, (uint32_t)(c * (2 * C) + 16 * (l0 ^ (c & (LPC - 1)))), 0);
      }
      wait_vm(0);
#pragma unroll
      for (int ob = 0; ob < OB; ob++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const half4 v = *reinterpret_cast<const half4*>(acc_piece<C>(zs, l, ob, q));
#pragma unroll
          for (int e = 0; e < 4; e++) o[ob][4 * q + e] = (float)v[e];
        }
      cs_lds_fence();
      ln_rows_lds<C>(zs, p.ln_w, p.ln_b, p.eps);
      cs_lds_fence();
      rows_to_frags<C>(zs, nf);
    }
    __syncthreads();  // every wave's rows are read: the ring takes their place
    load3(0);
    if (U > 1) {
      load12(1);
      load3(1);
    }

    // 2. The hidden units, 32 per step, in two phases: W1 (and W2) against LN(z), then the
    // activation and W3. W1's row index rho = 16 j + 8 a + 4 b + c holds unit 16 j + 8 b + 4 a + c: the
    // accumulator registers 8 j .. 8 j + 7 of lane half b are then 8 consecutive units 16 j + 8 b ..
    // + 7, which is the B fragment of the second GEMM with no data movement. Waves 4-7 run one phase
    // behind waves 0-3 (each SIMD holds one of both): one wave's activation runs under the other's
    // MFMAs. A fragment is read four MFMAs before its use, across the phases' barriers too: a ring slot
    // is complete one barrier before the phase that multiplies it.
    int s1, s3;
    auto addr1 = [&](int u) {
      const int l = fresh_lane(), ur = (l & 0x13) | ((l & 4) << 1) | ((l & 8) >> 1);
      s1 = (u % 3) * T::W12B + ur * 128 + 16 * ((l >> 5) ^ ((ur >> 1) & 7));
    };
    auto addr3 = [&](int u) {
      const int l = fresh_lane();
      s3 = T::OFF3 + (u % 3) * T::W3B + (l & 31) * 64 + 16 * ((l >> 5) ^ ((l >> 2) & 3));
    };
    auto frag1 = [&](int q) {  // q = G k + matrix
      const int k = q / T::G, m = q % T::G;
      return *reinterpret_cast<const half8*>(smem + (s1 ^ (32 * (k & 3))) + m * T::W1B + (k >> 2) * 4096);
    };
    auto frag3 = [&](int q) { return *reinterpret_cast<const half8*>(smem + (s3 ^ (32 * (q / OB))) + (q % OB) * 2048); };
    half8 w[4];
    f32x16 d1, d2;
    // Ends a phase: this wave's share of every ring slot loaded two phases ago or earlier is in LDS,
    // and after the barrier everyone's. `more`: the last two phases both issued loads.
    auto phase_end = [&](bool more) {
      if (more)
        wait_vm(T::N12 + T::N3);
      else
        wait_vm(0);
      __syncthreads();
    };
    const int late = wave / (kCsWaves / 2);
    phase_end(U > 1);
    if (late) {
      if (U > 2) load12(2);
      phase_end(U > 2);
    }
    addr1(0);
#pragma unroll
    for (int q = 0; q < 4; q++) w[q] = frag1(q);
    int u = 0;
    do {
      constexpr int Q1 = T::G * KS, Q3 = 2 * OB;
#pragma unroll
      for (int i = 0; i < 16; i++) d1[i] = d2[i] = 0.f;
#pragma unroll
      for (int q = 0; q < Q1; q += 2) {
        d1 = mfma32(w[q & 3], nf[q / T::G], d1);
        d2 = mfma32(w[(q + 1) & 3], nf[(q + 1) / T::G], d2);
        if (q + 4 == Q1) addr3(u);
        w[q & 3] = q + 4 < Q1 ? frag1(q + 4) : frag3(q + 4 - Q1);
        w[(q + 1) & 3] = q + 5 < Q1 ? frag1(q + 5) : frag3(q + 5 - Q1);
        __builtin_amdgcn_sched_barrier(0);
        if (q == 2 && u + 2 < U) {
          if (late)
            load3(u + 2);
          else
            load12(u + 2);
        }
      }
      phase_end(u + 2 < U);
      half8 act[2];
      auto activate = [&](int i) {
        const float v = SWIGLU ? d1[i] * sigmoidf_fast(d1[i]) * d2[i] : fmaxf(d1[i] + d2[i], 0.f);
        act[i >> 3][i & 7] = (half_t)v;
      };
#pragma unroll
      for (int i = 0; i < 8; i++) activate(i);
      const int un = u + 2 + late;
      if (un < U) {
        if (late)
          load12(un);
        else
          load3(un);
      }
#pragma unroll
      for (int q = 0; q < Q3; q += 2) {
        o[q % OB] = mfma32(w[q & 3], act[q / OB], o[q % OB]);
        o[q % OB + 1] = mfma32(w[(q + 1) & 3], act[q / OB], o[q % OB + 1]);
        if (q < OB) {
#pragma unroll
          for (int i = 0; i < 16 / OB; i++) activate(8 + q * (8 / OB) + i);
        }
        if (q + 4 == Q3) addr1(u + 1);
        w[q & 3] = q + 4 < Q3 ? frag3(q + 4) : frag1(q + 4 - Q3);
        w[(q + 1) & 3] = q + 5 < Q3 ? frag3(q + 5) : frag1(q + 5 - Q3);
        __builtin_amdgcn_sched_barrier(0);
      }
      phase_end(un < U);
    } while (++u < U);
    if (!late) __syncthreads();
    __syncthreads();  // (and the late waves are done with the ring)

    // 3. Rounded once, through the wave's LDS rows, out as whole cell rows.
    {
      const int l = fresh_lane();
#pragma unroll
      for (int ob = 0; ob < OB; ob++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
          half4 v;
#pragma unroll
          for (int e = 0; e < 4; e++) v[e] = (half_t)o[ob][4 * q + e];
          *reinterpret_cast<half4*>(acc_piece<C>(zs, l, ob, q)) = v;
        }
      cs_lds_fence();
      const rsrc_t ro = make_rsrc_n(p.out + (nv ? cell0 * C : 0), (uint32_t)nv * C * 2u);
      const int l0 = l & (LPC - 1), cl = l / LPC;
#pragma unroll 4
      for (int i = 0; i < NKB; i++) {
        const half8 v = *reinterpret_cast<const half8*>(zs + i * 1024 + cl * (2 * C) + 16 * (l0 ^ ((i * CPI + cl) & (LPC - 1))));
        bstore16(ro, (uint32_t)(i * 1024 + l * 16), v);
      }
    }
    __syncthreads();  // the rows are the next tile's ring slots
  }
}

// ---- projection: a, b = (LN(z) Ws^T) * sigmoid(LN(z) Wg^T) [* mask], in FragLayout ---------------------
// One launch in place of the LayerNorm pass and the weight-stationary GEMM. No single limit: at L=476 its 165
// us hold ~62 us of vector work (the gates' exp and rcp above all), ~26 us of MFMAs and 68 us of memory
// traffic, and leaving any one of them out saved 20 to 60 us, so what it loses is overlap. Tried on top and not
// faster: the gate of a block between the products of the next one (100 us for the update at L=238 either
// way), and 8 waves per workgroup with a ring of three slots (440 us against 414 at L=476).
template <int C>
struct CsProjGeo {
  static constexpr int WB = 32 * C * 2, WSB = 2 * WB;       // 32 signal rows and their gate rows: a ring slot
  static constexpr int NL = WSB / 1024 / kEmWaves;
  static constexpr int ZW = kCsCells * C * 2;
  static constexpr int OFFS = 2 * WSB > kEmWaves * ZW ? 2 * WSB : kEmWaves * ZW;  // z rows, then the ring; then staging
  static constexpr int STG = 32 * 256;                      // 32 channels x 16 operand rows x 8 k
  static constexpr int SMEM = OFFS + 2 * STG;               // (the LayerNorm parameters lie in the staging's place)
  static_assert(2 * SMEM <= 160 * 1024 && 2 * C * 4 <= 2 * STG, "LDS: two workgroups per CU");
};

// A workgroup takes 16 operand rows x 8 k, a wave four of the rows: its cells c = 8 dr + dc are the
// rows of D[cell][channel], so a lane ends with 4 consecutive k of one channel and row.
template <int C, bool MASK>
__global__ __launch_bounds__(64 * kEmWaves, 2) void project_stream_kernel(ProjectArgs p) {
  using T = CsProjGeo<C>;
  constexpr int KS = C / 16, NB = 2 * C / 32, LPC = C / 8, CPI = 64 / LPC, NKB = T::ZW / 1024;
  static_assert(C % (64 * kEmWaves) == 0, "whole parameter loads");
  __shared__ __align__(1024) char smem[T::SMEM];
  float* lnp = reinterpret_cast<float*>(smem + T::OFFS);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t lds0 = lds_address(smem);
  const int L = p.L;
  const int nr = (L + 15) / 16, t0 = xcd_remap(blockIdx.x, gridDim.x), bi = t0 / (nr * p.tiles_per_line);
  const int tt = t0 - bi * nr * p.tiles_per_line, tr = tt / p.tiles_per_line;
  const int R0 = 16 * tr, K0 = 8 * (tt - tr * p.tiles_per_line);   // first operand row, first k
  const int row0 = R0 + 4 * wave;
  const size_t cb = (size_t)bi * L * L + (p.transpose ? (size_t)K0 * L + row0 : (size_t)row0 * L + K0);
  char* zs = smem + wave * T::ZW;
  // offset in cells of the wave's cell c from its first one, and whether it lies inside the grid
  auto coff = [&](int c) { return p.transpose ? (c & 7) * L + (c >> 3) : (c >> 3) * L + (c & 7); };
  auto cin = [&](int c) { return row0 + (c >> 3) < L && K0 + (c & 7) < L; };

  // 1. z rows into LDS (XOR-swizzled as ln_rows_lds reads them), LayerNorm, fragments; zeros for the cells
  // past the grid, whose operands are then 0
  half8 nf[KS];
  float mv[MASK ? 16 : 1];
  {
    const dma_src_t dz = dma_src(p.z + cb * C, (uint32_t)kBufRange);
    const int l = fresh_lane(), l0 = l & (LPC - 1), cl = l / LPC;
#pragma unroll 4
    for (int t = 0; t < NKB; t++) {
      const int c = t * CPI + cl;
      dma16(dz, lds0 + wave * T::ZW + t * 1024,
            cin(c) ? (uint32_t)coff(c) * (2 * C) + 16 * (l0 ^ (c & (LPC - 1))) : kOOB, 0);
    }
    for (int c = threadIdx.x; c < C; c += 64 * kEmWaves) {
      lnp[c] = p.ln_w[c];
      lnp[C + c] = p.ln_b[c];
    }
    if constexpr (MASK) {
      const rsrc_t rm = make_rsrc(p.mask + cb);
#pragma unroll
      for (int e = 0; e < 16; e++) {
        const int c = 8 * (e >> 2) + 4 * (l >> 5) + (e & 3);
        mv[e] = h2f(bload2(rm, cin(c) ? (uint32_t)coff(c) * 2u : kOOB));
      }
    }
  }
  wait_vm(0);
  __syncthreads();  // the parameters are in LDS
  ln_rows_lds<C>(zs, lnp, lnp + C, p.eps);
  cs_lds_fence();
  rows_to_frags<C>(zs, nf);
  if (row0 + 4 > L || K0 + 8 > L) {
    const int l = fresh_lane();
    const bool in = cin(l & 31);
#pragma unroll
    for (int k = 0; k < KS; k++) nf[k] = in ? nf[k] : zero_half8();
  }
  __syncthreads();  // every wave's rows are read: the ring takes their place

  // 2. 32 channels at a time (a's, then b's): both products, the gate, the staged tile out as 256-byte
  // segments (16 rows x 8 k of one channel) while the next block's products run
  const dma_src_t rw = dma_src(p.w, 4u * C * C * 2u);
  auto load_w = [&](int ob) {
    const uint32_t dst = lds0 + (ob & 1) * T::WSB;
    const int l = fresh_lane();
    const uint32_t l1 = (uint32_t)(l >> 3) * (C * 2), x1 = 16u * (uint32_t)((l & 7) ^ (l >> 4));
#pragma unroll
    for (int t = 0; t < T::NL; t++) {
      constexpr int N1 = T::WB / 1024;
      const int q = wave * T::NL + t, m = q / N1, qm = q % N1, st = qm / 4, rq = qm % 4;
      dma16(rw, dst + q * 1024, l1 + (x1 ^ (64u * (rq & 1))), (uint32_t)(m * 2 * C + 32 * ob + 8 * rq) * (C * 2) + st * 128);
    }
  };
  const size_t plane_h = (size_t)p.rbn * p.kbn * FragLayout::kTileHalfs;
  const size_t tile_h = ((size_t)(R0 >> 5) * p.kbn + (K0 >> 4)) * FragLayout::kTileHalfs +
                        (size_t)((R0 & 31) + 32 * ((K0 >> 3) & 1)) * 8;
  // this wave's share of block ob's staged tile: 2 x 4 channels of 256 bytes
  auto store = [&](int ob) {
    const int l = fresh_lane();
    const char* sg = smem + T::OFFS + (ob & 1) * T::STG;
    const int ch0 = 32 * ob % C;
    const rsrc_t ro = make_rsrc((ob < NB / 2 ? p.a : p.b) + ((size_t)bi * C + ch0) * plane_h + tile_h);
#pragma unroll
    for (int t = 0; t < 2; t++) {
      const int ch = 8 * wave + 4 * t + (l >> 4);
      bstore16(ro, (uint32_t)(ch * plane_h + 8 * (l & 15)) * 2u,
               *reinterpret_cast<const half8*>(sg + ch * 256 + 16 * ((l & 15) ^ (ch & 15))));
    }
  };
  load_w(0);
  wait_vm(0);
  __syncthreads();
#pragma unroll 1
  for (int ob = 0; ob < NB; ob++) {
    if (ob + 1 < NB) load_w(ob + 1);
    if (ob > 0) store(ob - 1);
    const int l = fresh_lane(), s1 = (ob & 1) * T::WSB + (l & 31) * 128 + 16 * ((l >> 5) ^ ((l >> 1) & 7));
    auto frag = [&](int q) {
      const int k = q >> 1, m = q & 1;
      return *reinterpret_cast<const half8*>(smem + (s1 ^ (32 * (k & 3))) + m * T::WB + (k >> 2) * 4096);
    };
    constexpr int PF = 6;  // fragments in flight
    half8 w[PF];
#pragma unroll
    for (int q = 0; q < PF; q++) w[q] = frag(q);
    f32x16 d1, d2;
#pragma unroll
    for (int e = 0; e < 16; e++) d1[e] = d2[e] = 0.f;
#pragma unroll
    for (int q = 0; q < 2 * KS; q += 2) {
      d1 = mfma32(nf[q / 2], w[q % PF], d1);
      d2 = mfma32(nf[q / 2], w[(q + 1) % PF], d2);
      if (q + PF < 2 * KS) {
        w[q % PF] = frag(q + PF);
        w[(q + 1) % PF] = frag(q + PF + 1);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    char* sg = smem + T::OFFS + (ob & 1) * T::STG + (l & 31) * 256 + 8 * (l >> 5);
#pragma unroll
    for (int dr = 0; dr < 4; dr++) {
      half4 hv;
#pragma unroll
      for (int e = 0; e < 4; e++) {
        float v = d1[4 * dr + e] * sigmoidf_fast(d2[4 * dr + e]);
        if constexpr (MASK) v *= mv[4 * dr + e];
        __asm__ volatile("" : "+v"(v));  // fp32 then fp16 at every position
        hv[e] = (half_t)v;
      }
      *reinterpret_cast<half4*>(sg + 16 * ((4 * wave + dr) ^ (l & 15))) = hv;
    }
    if (ob > 0)
      wait_vm(2);  // the next block's weights; the two stores behind them may still be on their way
    else
      wait_vm(0);
    __syncthreads();
  }
  store(NB - 1);
}

hipError_t launch_project_stream(const ProjectArgs& a, hipStream_t s) {
  ProjectArgs t = a;
  t.tiles_per_line = (a.L + 7) / 8;  // k tiles per row tile
  const long long nt = (long long)a.B * ((a.L + 15) / 16) * t.tiles_per_line;
  if (nt > 0x7fffffffLL) return hipErrorInvalidValue;
  const dim3 grid((unsigned)nt), blk(64 * kEmWaves);
  if (a.mask)
    ESM_LAUNCH((project_stream_kernel<256, true>), grid, blk, 0, s, t);
  else
    ESM_LAUNCH((project_stream_kernel<256, false>), grid, blk, 0, s, t);
  return hipGetLastError();
}

// ---- emit and gate: out = [z +] (LN_mix(x) We^T) * sigmoid(LN_in(z) Wg^T) [* mask] ------------------
// One launch in place of the transposing LayerNorm of x and the dual GEMM, which wrote and read LN(x) and
// read a kept LN(z): x and z are read once, both LayerNorms happen on the way into the fragments, z stays in
// registers (in accumulator order) for the residual. Bound by memory and latency phases: a workgroup loads x
// (its ~16,000 cycles at the chip's rate), then z, normalises (~10,000), multiplies (8 blocks of ~3,000) and
// stores. Two workgroups of 4 waves per CU, each with its own weight ring, run these phases against each
// other; one of 8 waves made the update 499 us at L=476 instead of 457 and 116 instead of 110 at L=238.
// Traced, the two launches against this one: L=238 15.1 + 42.7 -> 39.9 us, L=476 64.7 + 149.5 -> 113.4 us (348
// MB of x, z and out: 3.1 TB/s).
template <int C>
struct CsEmitGeo {
  static constexpr int WB = 32 * C * 2, WSB = 2 * WB;       // 32 outputs of We, of Wg; a ring slot holds both
  static constexpr int NL = WSB / 1024 / kEmWaves;          // 1 KB loads per wave and slot
  static constexpr int ZW = kCsCells * C * 2;               // a wave's x, then z, then output rows
  static constexpr int OFFZ = 4 * C * 4;                    // behind the LayerNorm parameters; both ring slots
  static constexpr int SMEM0 = OFFZ + 2 * WSB, SMEM1 = OFFZ + kEmWaves * ZW;  // take their place
  static constexpr int SMEM = SMEM0 > SMEM1 ? SMEM0 : SMEM1;
  static_assert(2 * SMEM <= 160 * 1024, "LDS: two workgroups per CU");
};

template <int C, bool MASK, bool RES>
__global__ __launch_bounds__(64 * kEmWaves, 2) void emit_stream_kernel(EpilogueArgs p) {
  using T = CsEmitGeo<C>;
  constexpr int KS = C / 16, OB = C / 32, LPC = C / 8, CPI = 64 / LPC, NKB = T::ZW / 1024;
  static_assert(OB % 2 == 0 && C % (64 * kEmWaves) == 0, "output blocks in pairs; whole parameter loads");
  __shared__ __align__(1024) char smem[T::SMEM];
  float* lnp = reinterpret_cast<float*>(smem);  // LN_mix w, b, LN_in w, b
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t lds0 = lds_address(smem);
  const int L = p.L;
  // this wave's unit: 32 cells (bi, i, pos0 ..) of one pair row; nv of them inside the row. The XCD-aware
  // order gives neighbouring units, which share lines of x, one L2.
  const int u = xcd_remap(blockIdx.x, gridDim.x) * kEmWaves + wave, bl = u / p.tiles_per_line;
  const int pos0 = (u - bl * p.tiles_per_line) * kCsCells, bi = bl / L, i = bl - bi * L;
  const bool live = bi < p.B;
  const int nv = !live ? 0 : L - pos0 < kCsCells ? L - pos0 : kCsCells;
  const size_t cell0 = live ? ((size_t)bi * L + i) * L + pos0 : 0;
  const int zoff = T::OFFZ + wave * T::ZW;
  char* zs = smem + zoff;

  // 1. x: channel rows of 32 cells (64 bytes) into the wave's LDS, transposing reads into fragments,
  // LayerNorm in registers; z takes x's place meanwhile.
  half8 nx[KS], nz[KS];
  half4 zo[OB][4];  // z, then the output, in accumulator order
  float mv = 1.f;
  {
    const int l = fresh_lane();
    const bool okx = live && pos0 + 8 * (l & 3) < p.ldx;
    const uint32_t xo = okx ? (uint32_t)((size_t)(l >> 2) * L * p.ldx + 8 * (l & 3)) * 2u : kOOB;
    const half_t* xb = p.x + (((size_t)(live ? bi : 0) * C) * L + (live ? i : 0)) * p.ldx + (live ? pos0 : 0);
#pragma unroll 4
    for (int q = 0; q < C / 16; q++)
      dma16(dma_src(xb + (size_t)16 * q * L * p.ldx, (uint32_t)kBufRange), lds0 + zoff + q * 1024, xo, 0);
    for (int c = threadIdx.x; c < C; c += 64 * kEmWaves) {
      lnp[c] = p.ln_mix_w[c];
      lnp[C + c] = p.ln_mix_b[c];
      lnp[2 * C + c] = p.ln_in_w[c];
      lnp[3 * C + c] = p.ln_in_b[c];
    }
    if constexpr (MASK) mv = (l & 31) < nv ? (float)p.mask[cell0 + (l & 31)] : 0.f;
  }
  wait_vm(0);
  __syncthreads();  // the parameters are in LDS
  {
    const int l = fresh_lane(), h = l >> 5, n0 = 16 * ((l >> 4) & 1), j = l & 15;
    const half_t* xs = reinterpret_cast<const half_t*>(zs);
    float s = 0.f, q = 0.f;
#pragma unroll
    for (int k = 0; k < KS; k++) {
      const half4 lo = ds_read_tr16x4(xs + (16 * k + 8 * h + (j >> 2)) * kCsCells + n0 + 4 * (j & 3));
      const half4 hi = ds_read_tr16x4(xs + (16 * k + 8 * h + 4 + (j >> 2)) * kCsCells + n0 + 4 * (j & 3));
      nx[k] = half8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    }
#pragma unroll
    for (int k = 0; k < KS; k++) pin(nx[k]);
    {
      const dma_src_t dz = dma_src(p.z + cell0 * C, (uint32_t)nv * C * 2u);
      const int l0 = l & (LPC - 1), cl = l / LPC;
#pragma unroll 4
      for (int t = 0; t < NKB; t++) {
        const int c = t * CPI + cl;
        dma16(dz, lds0 + zoff + t * 1024, (uint32_t)(c * (2 * C) + 16 * (l0 ^ (c & (LPC - 1)))), 0);
      }
    }
#pragma unroll
    for (int k = 0; k < KS; k++) dot2_moments(nx[k], s, q);
    s += __shfl_xor(s, 32);
    q += __shfl_xor(q, 32);
    float rstd, shift;
    ln_scale_shift(s, q, 1.0f / C, p.eps_mix, rstd, shift);
#pragma unroll
    for (int k = 0; k < KS; k++) {
      const f32x4* w = reinterpret_cast<const f32x4*>(lnp + 16 * k + 8 * h);
      const f32x4* b = reinterpret_cast<const f32x4*>(lnp + C + 16 * k + 8 * h);
      const f32x4 w0 = w[0], w1 = w[1], b0 = b[0], b1 = b[1];
#pragma unroll
      for (int e = 0; e < 4; e++) {
        nx[k][e] = ln_value(nx[k][e], rstd, shift, w0[e], b0[e]);
        nx[k][e + 4] = ln_value(nx[k][e + 4], rstd, shift, w1[e], b1[e]);
      }
    }
#pragma unroll
    for (int k = 0; k < KS; k++) pin(nx[k]);
  }
  wait_vm(0);
  if constexpr (RES) {
    const int l = fresh_lane();
#pragma unroll
    for (int ob = 0; ob < OB; ob++)
#pragma unroll
      for (int q = 0; q < 4; q++) zo[ob][q] = *reinterpret_cast<const half4*>(acc_piece<C>(zs, l, ob, q));
    cs_lds_fence();
  }
  ln_rows_lds<C>(zs, lnp + 2 * C, lnp + 3 * C, p.eps_in);
  cs_lds_fence();
  rows_to_frags<C>(zs, nz);
  __syncthreads();  // every wave's rows are read: the ring takes their place

  // 2. The outputs, 32 at a time: both products, the gate. The next block's weights arrive meanwhile.
  const dma_src_t re = dma_src(p.w_emit, C * C * 2u), rg = dma_src(p.w_gate, C * C * 2u);
  auto load_w = [&](int ob) {
    const uint32_t dst = lds0 + T::OFFZ + (ob & 1) * T::WSB;
    const int l = fresh_lane();
    const uint32_t l1 = (uint32_t)(l >> 3) * (C * 2), x1 = 16u * (uint32_t)((l & 7) ^ (l >> 4));
#pragma unroll
    for (int t = 0; t < T::NL; t++) {
      constexpr int N1 = T::WB / 1024;
      const int q = wave * T::NL + t, m = q / N1, qm = q % N1, st = qm / 4, rq = qm % 4;
      dma16(m ? rg : re, dst + q * 1024, l1 + (x1 ^ (64u * (rq & 1))), (uint32_t)(32 * ob + 8 * rq) * (C * 2) + st * 128);
    }
  };
  load_w(0);
  wait_vm(0);
  __syncthreads();
  auto block = [&](int ob, half4 (&zb)[4]) {
    if (ob + 1 < OB) load_w(ob + 1);
    const int l = fresh_lane(), s1 = T::OFFZ + (ob & 1) * T::WSB + (l & 31) * 128 + 16 * ((l >> 5) ^ ((l >> 1) & 7));
    auto frag = [&](int q) {
      const int k = q >> 1, m = q & 1;
      return *reinterpret_cast<const half8*>(smem + T::OFFZ + ((s1 - T::OFFZ) ^ (32 * (k & 3))) + m * T::WB + (k >> 2) * 4096);
    };
    half8 w[4];
#pragma unroll
    for (int q = 0; q < 4; q++) w[q] = frag(q);
    f32x16 d1, d2;
#pragma unroll
    for (int e = 0; e < 16; e++) d1[e] = d2[e] = 0.f;
#pragma unroll
    for (int q = 0; q < 2 * KS; q += 2) {
      d1 = mfma32(w[q & 3], nx[q / 2], d1);
      d2 = mfma32(w[(q + 1) & 3], nz[q / 2], d2);
      if (q + 4 < 2 * KS) {
        w[q & 3] = frag(q + 4);
        w[(q + 1) & 3] = frag(q + 5);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        float v = d1[4 * q + e] * sigmoid_from_t(d2[4 * q + e] * kNegLog2e);
        if constexpr (MASK) v *= mv;
        if constexpr (RES) v += (float)zb[q][e];
        __asm__ volatile("" : "+v"(v));  // fp32 then fp16 at every position
        zb[q][e] = (half_t)v;
      }
    wait_vm(0);
    __syncthreads();
  };
#pragma unroll 1
  for (int ob = 0; ob < OB; ob += 2) {
    block(ob, zo[0]);
    block(ob + 1, zo[1]);
    // the pieces turn by two blocks, so that the loop body names fixed registers
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const half4 t0 = zo[0][q], t1 = zo[1][q];
#pragma unroll
      for (int b = 0; b + 2 < OB; b++) zo[b][q] = zo[b + 2][q];
      zo[OB - 2][q] = t0;
      zo[OB - 1][q] = t1;
    }
  }

  // 3. Out through the wave's LDS rows as whole cell rows.
  {
    const int l = fresh_lane();
#pragma unroll
    for (int ob = 0; ob < OB; ob++)
#pragma unroll
      for (int q = 0; q < 4; q++) *reinterpret_cast<half4*>(acc_piece<C>(zs, l, ob, q)) = zo[ob][q];
    cs_lds_fence();
    const rsrc_t ro = make_rsrc_n(p.out + cell0 * C, (uint32_t)nv * C * 2u);
    const int l0 = l & (LPC - 1), cl = l / LPC;
#pragma unroll 4
    for (int t = 0; t < NKB; t++) {
      const half8 v = *reinterpret_cast<const half8*>(zs + t * 1024 + cl * (2 * C) + 16 * (l0 ^ ((t * CPI + cl) & (LPC - 1))));
      bstore16(ro, (uint32_t)(t * 1024 + l * 16), v);
    }
  }
}

hipError_t launch_emit_stream(const EpilogueArgs& a, hipStream_t s) {
  EpilogueArgs e = a;
  e.tiles_per_line = (a.L + kCsCells - 1) / kCsCells;
  const long long units = (long long)a.B * a.L * e.tiles_per_line, nt = (units + kEmWaves - 1) / kEmWaves;
  if (nt * kEmWaves > 0x7fffffffLL) return hipErrorInvalidValue;
  const dim3 grid((unsigned)nt), blk(64 * kEmWaves);
  const bool m = a.out_mask && a.mask;
  if (m && a.residual)
    ESM_LAUNCH((emit_stream_kernel<256, true, true>), grid, blk, 0, s, e);
  else if (m)
    ESM_LAUNCH((emit_stream_kernel<256, true, false>), grid, blk, 0, s, e);
  else if (a.residual)
    ESM_LAUNCH((emit_stream_kernel<256, false, true>), grid, blk, 0, s, e);
  else
    ESM_LAUNCH((emit_stream_kernel<256, false, false>), grid, blk, 0, s, e);
  return hipGetLastError();
}

hipError_t launch_transition_stream(const TransitionArgs& a, int C, int cus, hipStream_t s) {
  TransitionArgs t = a;
  const size_t nt = (a.ncells + kCsWaves * kCsCells - 1) / (kCsWaves * kCsCells);
  t.ntiles = (int)nt;
  const dim3 grid((unsigned)(nt < (size_t)cus ? nt : cus)), blk(kCsThreads);
  if (C == 256 && a.w2)
    ESM_LAUNCH((transition_stream_kernel<256, true>), grid, blk, 0, s, t);
  else if (C == 256)
    ESM_LAUNCH((transition_stream_kernel<256, false>), grid, blk, 0, s, t);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

}  // namespace esm
