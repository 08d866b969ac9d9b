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
constexpr int kCsCells = 32;                 // cells per wave: the columns of one 32x32x16 MFMA

// 1 KB of a matrix into LDS, 16 bytes per lane from anywhere in the resource, landing in lane order
// at a wave-uniform LDS address. Written as assembly because the compiler, which cannot tell a
// ring's slots apart, waits for every such load in flight before the next LDS read; here the wait is
// where the slot is handed over (wait_vm and a barrier). Nothing is written to a register.
typedef u32x4 dma_src_t;
DEV dma_src_t dma_src(const void* base, uint32_t bytes) {
  const uint64_t a = reinterpret_cast<uint64_t>(base);
  return u32x4{(uint32_t)a, (uint32_t)(a >> 32) & 0xffffu, bytes, (uint32_t)kBufWord3};
}
DEV void dma16(dma_src_t r, uint32_t l, uint32_t off, uint32_t soff) {
  __asm__ volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                   :
                   : "s"(l), "v"(off), "s"(r), "s"(soff)
                   : "memory");
}
#define wait_vm(N) \
  do { \
    __builtin_amdgcn_s_waitcnt(0xF70 | (N));  /* vmcnt(N), N < 16 */ \
    __asm__ volatile("" ::: "memory"); \
  } while (0)
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
// Bound by the matrix cores' power: the loop runs them at ~72% of its cycles, and under that load
// the shader clock falls to ~1.6 GHz (2.2 without the MFMAs). L=238, C=256, H=1024: SwiGLU 174 ->
// 108 us, ReLU 133 -> 77; L=476: 656 -> 406 and 513 -> 288 (89 GFLOP at L=238: 0.83 PFLOP/s). What is
// not the loop (~20 us at one tile per CU): z's arrival, the LayerNorm, the stores.
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
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
  const int H = p.H, U = H / 32;
  const dma_src_t r1 = dma_src(p.w1, (uint32_t)H * C * 2u);
  const dma_src_t r2 = dma_src(SWIGLU ? p.w2 : p.w1, (uint32_t)H * C * 2u);
  const dma_src_t r3 = dma_src(p.w3, (uint32_t)H * C * 2u);

  // (each address is computed where it is used from a lane number the compiler cannot hoist: the
  // loop has no registers left to keep them in)
  auto fresh_lane = [&]() {
    int l = lane;
    __asm__ volatile("" : "+v"(l));
    return l;
  };
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
    // accumulators start from it (the residual); LayerNorm in place, 1 KB at a time in a rolled loop
    // (straight-line code that runs once per tile is bound by its instruction fetches); fragments.
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
      float g[8], bb[8];
#pragma unroll
      for (int e = 0; e < 8; e++) {
        g[e] = p.ln_w[8 * l0 + e];
        bb[e] = p.ln_b[8 * l0 + e];
      }
      wait_vm(0);
      {
        const char* zr = zs + (l & 31) * (2 * C) + 8 * (l >> 5);
#pragma unroll
        for (int ob = 0; ob < OB; ob++)
#pragma unroll
          for (int q = 0; q < 4; q++) {
            const half4 v = *reinterpret_cast<const half4*>(zr + 16 * ((4 * ob + q) ^ (l & (LPC - 1))));
#pragma unroll
            for (int e = 0; e < 4; e++) o[ob][4 * q + e] = (float)v[e];
          }
      }
      cs_lds_fence();
#pragma unroll 4
      for (int i = 0; i < NKB; i++) {
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
        const float rstd = rsqrtf(lane_sum<LPC>(q0 + q1) * (1.0f / C) + p.eps);
        half8 v;
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = (half_t)(d[e] * rstd * g[e] + bb[e]);
        *reinterpret_cast<half8*>(piece) = v;
      }
      cs_lds_fence();
#pragma unroll
      for (int k = 0; k < KS; k++)
        nf[k] = *reinterpret_cast<const half8*>(zs + (l & 31) * (2 * C) + 16 * ((2 * k + (l >> 5)) ^ (l & (LPC - 1))));
#pragma unroll
      for (int k = 0; k < KS; k++) pin(nf[k]);
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
      char* zr = zs + (l & 31) * (2 * C) + 8 * (l >> 5);
#pragma unroll
      for (int ob = 0; ob < OB; ob++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
          half4 v;
#pragma unroll
          for (int e = 0; e < 4; e++) v[e] = (half_t)o[ob][4 * q + e];
          *reinterpret_cast<half4*>(zr + 16 * ((4 * ob + q) ^ (l & (LPC - 1)))) = v;
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
