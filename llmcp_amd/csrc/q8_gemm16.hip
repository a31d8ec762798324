// q8_gemm16.hip -- Q8_0 GEMM on 16 x 16 MFMA tiles, for few rows or columns.
//
// The same function as gemm_kernel (q8_gemm.hip): exact int32 block dots,
// acc = fma(f32(I), sa * dw, acc) or acc + f32(I) * (sa * dw) in block
// order, bit for bit; for the shapes whose 128 x 96 or 64 x 64 workgroups
// leave most of the GPU idle.  There the time is one wave's serial walk
// over K, so a wave gets the smallest tile a matrix instruction has (16 x
// 16, four accumulators per lane) and as few other instructions per block
// as possible:
//   - v_mfma_i32_16x16x32_i8: one block's dots;
//   - v_mfma_f32_16x16x1_4b_f32: the scale tiles sa x dw of four blocks at
//     once (one exact product, one rounding, as a multiply);
//   - every operand comes from LDS, where producer waves put it by DMA; a
//     compute wave has no global load and waits for none.
// A workgroup computes RT x CN tiles, one compute wave each, so that the
// chip's 1024 SIMDs get close to the same number of tiles at every shape;
// shape16 chooses RT and CN, gemm16_takes the shapes (figures of both there).
#include "q8_kernels.h"

#include <algorithm>

#include "q8_device.h"

namespace llmcp_q8 {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v2i __attribute__((ext_vector_type(2)));
typedef unsigned v2u __attribute__((ext_vector_type(2)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void lds_void;

struct Gemm16Weight {
  const uint8_t *w0, *w1;  // unit layout; w1: the up matrix of a SwiGLU
  void *y;
  int64_t ldy;
  int32_t rows;   // N
  int32_t act;
  int32_t group0;  // first column group (CN tiles) of this weight in the grid
};

struct Gemm16Args {
  const int8_t *qa;    // Q8_1 rows in 16-row tiles (launch_quantize_tiled)
  const float *sa;
  const void *add;     // residual [m, ldr] of y's element type, or null
  int64_t ldr;
  int64_t m_rows;
  int32_t row_tiles;   // 16-row tiles in qa / sa
  int32_t units;       // units per lane group
  int32_t m_groups;    // workgroups along M
  int32_t n_groups;    // column groups over all weights
  int32_t count;       // weights
  int32_t y_bf16;
  Gemm16Weight g[kMaxGroup];
};

// The LDS of a workgroup.  Activations: a ring of NA stages of eight blocks,
// [row tile][block pair][1 KiB] and the scales [row tile][block][16].  Weights: a ring of NB stages
// of SB blocks (S = 1: one unit; S = 4, 6: four lane slots of the pass's S
// units), per column tile the values and then the scale blocks.
template <int SEG, int RT, int CN, bool DUAL>
struct Gemm16Shape {
  static constexpr int NM = DUAL ? 2 : 1;          // matrices
  static constexpr int CB = CN * NM;               // column tiles of B
  static constexpr int W = RT * CB;                // compute waves
  static constexpr int P = W > 4 || CB >= 4 ? 2 : 1;  // producers of A, and of B
  static constexpr int SB = SEG == 6 ? 24 : 16;    // blocks per weight stage
  static constexpr int SUB = SB / 8;               // A stages per weight stage
  static constexpr int QOPS = SB / 2;              // 1 KiB DMA ops of a tile's values
  // and of its scales: S = 1 the 128 B scale blocks of its four groups (one
  // op of 16 B per lane, half of it unused), S = 4, 6 the four slots' 8 B of
  // (unit, row) (4 B per lane)
  static constexpr int SOPS = SEG == 6 ? 3 : SEG == 4 ? 2 : 1;
  static constexpr int SLANE = SEG == 1 ? 16 : 4;
  static constexpr int TILE = QOPS * 1024 + SOPS * 64 * SLANE;
  static constexpr int PAIRS = (RT + 1) / 2;
  static constexpr int ASCALE = RT * 4096;         // the scales' place in an A stage
  static constexpr int ASZ = ASCALE + PAIRS * 1024;
  static constexpr int BSZ = CB * TILE;
  // Ring depths: as deep as the LDS allows (weights come from HBM, and a
  // stage has the time of NB - 1 others to land), within unrolled loops of
  // eight A stages (S = 6: nine).  The SwiGLU pair of one row tile leaves
  // room for three workgroups per CU instead: at N = 9216 that puts all 576
  // in flight at once (19.3 us against 25.9 with four pairs of tiles in 144
  // deep workgroups, M = 16, K = 2560; 16.8 with the non-temporal loads).
  static constexpr int BUDGET = (DUAL && RT == 1 ? 53 : 160) * 1024;
  static constexpr bool fits(int na, int nb) { return na * ASZ + nb * BSZ <= BUDGET; }
  static constexpr int NA = SEG != 6 && (fits(4, 4) || (!fits(3, 3) && fits(4, 2))) ? 4 : 3;
  static constexpr int NB = SEG != 6 && fits(4, 4) ? 4 : fits(3, 3) ? 3 : 2;
  static constexpr int BOFF = NA * ASZ;
  static constexpr int LDS = BOFF + NB * BSZ;
  static constexpr int AOPS = RT * 4 + PAIRS, DA = (AOPS + P - 1) / P;
  static constexpr int DQ = (CB * QOPS + P - 1) / P, DS = (CB * SOPS + P - 1) / P;
  static constexpr int DB = DQ + DS;
  // the stages of both rings at the same place again: A stages to unroll
  static constexpr int PERIOD = NB * SUB % NA == 0 ? NB * SUB
                                : NB * SUB * 2 % NA == 0 ? NB * SUB * 2 : NB * SUB * NA;
  static constexpr int THREADS = 64 * (W + 2 * P);
  // Declared: eight waves at least.  As a smaller workgroup, its LDS makes
  // the compiler assume one wave per SIMD, and it then keeps the MFMA
  // results in accumulation registers (a move per value to read them).
  static constexpr int BOUND = THREADS < 512 ? 512 : THREADS;
  static_assert(LDS <= 160 * 1024, "LDS");
};

// The resource of a stage's operands (no load is ever branched around: one past
// the last stage returns zeros without touching memory, dma_stage).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc_of(const void *p, const DmaStage &st) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, st.extent, 0x00020000);
}

template <int N>
__device__ __forceinline__ void wait_vmcnt16() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | 0x70 | 0xF00 | ((N >> 4) << 14));
}
__device__ __forceinline__ void barrier16() {
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_barrier();
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

__device__ __forceinline__ const uint8_t *uniform_base(const void *p) {
  const uint64_t v = (uint64_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return (const uint8_t *)(((uint64_t)hi << 32) | lo);
}

// Compute waves run a sequence of steps, one per quad of four blocks, two per
// A stage.  Entering step k a wave holds step k's dots and scale tiles and step k+1's
// operands; it issues step k+1's MFMAs and the LDS reads of step k+2's
// operands, and then runs step k's 32-operation epilogue, which covers
// both.  In the first step of A stage t every operand of the stage has been
// taken by an MFMA, so there the workgroup's barrier hands stage t + 1 to the
// compute waves and stage t's buffer back to the producers.
// DUAL, the SwiGLU pair: a wave for the tile of the gate matrix and one for
// the same columns of the up matrix, which hands its sums over through LDS
// at the end.
template <int SEG, bool FMA, int RT, int CN, bool DUAL>
__global__ __launch_bounds__((Gemm16Shape<SEG, RT, CN, DUAL>::BOUND))
void gemm16_kernel(const Gemm16Args p) {
#ifdef __HIP_DEVICE_COMPILE__  // the host pass needs the stub only (and drops
                               // it where it meets the operand pins below)
  typedef Gemm16Shape<SEG, RT, CN, DUAL> Sh;
  constexpr int NM = Sh::NM, NA = Sh::NA, NB = Sh::NB, SUB = Sh::SUB;
  __shared__ __align__(1024) uint8_t smem[Sh::LDS];

  // all row groups of a column group on one XCD (ids equal modulo 8)
  const int id = blockIdx.x;
  const int kk = id >> 3;
  const int ng = (kk / p.m_groups) * 8 + (id & 7);
  const int mg = kk % p.m_groups;
  if (ng >= p.n_groups) return;
  int gi = 0;
  while (gi + 1 < p.count && ng >= p.g[gi + 1].group0) ++gi;
  const Gemm16Weight &gw = p.g[gi];
  const int nc0 = 16 * CN * (ng - gw.group0);  // the workgroup's first column
  const int n_rows = gw.rows;
  const int stages = 2 * p.units;  // A stages
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

  if (wave >= Sh::W) {
    // ---- producers
    const int pw = wave - Sh::W;
    const int32_t nblk = p.units * kPassBlocks;
    if (pw < Sh::P) {
      // A: per stage RT * 4 ops of values and one op of scales per two tiles
      uint32_t voff[Sh::DA], ustep[Sh::DA], dst[Sh::DA];
      const uint8_t *base[Sh::DA];
      int32_t ends[Sh::DA];  // stages, none for a row tile past the last
#pragma unroll
      for (int u = 0; u < Sh::DA; ++u) {
        int o = pw + u * Sh::P;
        if (o >= Sh::AOPS) o -= Sh::AOPS;  // again: the same bytes, the same place
        const bool sc = o >= RT * 4;
        dst[u] = o * 1024;
        if (sc) {
          // lanes 0-31 the eight blocks' scales of one tile, 32-63 of the next
          const int t0 = mg * RT + 2 * (o - RT * 4);
          const int tl = min(t0 + (lane >> 5), p.row_tiles - 1) - t0;
          ends[u] = t0 < p.row_tiles ? stages : 0;
          ustep[u] = 512;
          base[u] = uniform_base(p.sa + (int64_t)t0 * nblk * 16);
          voff[u] = (uint32_t)max(tl, 0) * nblk * 64 + (lane & 31) * 16;
        } else {
          const int t0 = mg * RT + (o >> 2);
          ends[u] = t0 < p.row_tiles ? stages : 0;
          ustep[u] = 4096;
          base[u] = uniform_base(p.qa + (int64_t)t0 * nblk * 512 + (o & 3) * 1024);
          voff[u] = lane * 16;
        }
      }
      auto issue = [&](int t, int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < Sh::DA; ++u) {
          const DmaStage st = dma_stage(t, ends[u], (uint32_t)t * ustep[u]);
          __builtin_amdgcn_raw_ptr_buffer_load_lds(
              rsrc_of(base[u], st), (lds_void *)(smem + buf * Sh::ASZ + dst[u]), 16, voff[u],
              st.offset, 0, 0);
        }
      };
#pragma unroll
      for (int i = 0; i < NA; ++i) issue(i, i);
      wait_vmcnt16<(NA - 1) * Sh::DA>();
      barrier16();
      for (int t = 0, buf = 0; t < stages; ++t) {
        wait_vmcnt16<(NA - 2) * Sh::DA>();  // stage t + 1 is there
        barrier16();
        issue(t + NA, buf);
        buf = buf + 1 == NA ? 0 : buf + 1;
      }
    } else {
      // B.  S = 1: op (lane group gg, half h) is that group's 1 KiB half
      // unit, lane l taking row l / 16, slot (l % 16) ^ (4 gg + row).  S > 1:
      // op (unit i, half h) is 16 rows x 64 B, lane l taking row l / 4, slot
      // piece (l % 4) ^ (row / 4).  Either way the pieces that sixteen
      // lanes of a ds_read_b128 take lie in different banks.
      const uint32_t wrow = (uint32_t)p.units * kPassBytes;
      const int groups = n_rows >> 2;
      uint32_t voff[Sh::DB], uoff[Sh::DB], uslot[Sh::DB], dst[Sh::DB];
      const uint8_t *base[Sh::DB];
#pragma unroll
      for (int u = 0; u < Sh::DB; ++u) {
        const bool sc = u >= Sh::DQ;
        const int per = sc ? Sh::SOPS : Sh::QOPS;
        int o = pw - Sh::P + (sc ? u - Sh::DQ : u) * Sh::P;
        if (o >= Sh::CB * per) o -= Sh::CB * per;
        const int tl = o / per, oo = o % per;
        const int g0 = (nc0 >> 2) + 4 * (DUAL ? tl >> 1 : tl);  // the tile's first group
        base[u] = uniform_base(DUAL && (tl & 1) ? gw.w1 : gw.w0);
        dst[u] = tl * Sh::TILE + (sc ? Sh::QOPS * 1024 + oo * 64 * Sh::SLANE : oo * 1024);
        uoff[u] = uslot[u] = 0;
        if (sc && SEG == 1) {
          voff[u] = (uint32_t)min(g0 + ((lane >> 3) & 3), groups - 1) * wrow + kPassQs +
                    (lane & 7) * 16;
        } else if (sc) {
          const int idx = oo * 64 + lane, n = (idx >> 1) & 15;
          voff[u] = (uint32_t)min(g0 + (n >> 2), groups - 1) * wrow + (idx >> 5) * kPassBytes +
                    kPassQs + 32 * (n & 3) + 4 * (idx & 1);
          uslot[u] = 8;
        } else if (SEG == 1) {
          const int gg = oo >> 1, r = lane >> 4;
          voff[u] = (uint32_t)min(g0 + gg, groups - 1) * wrow + r * 256 +
                    (((lane & 15) ^ (4 * gg + r)) << 4);
          uoff[u] = (oo & 1) * 1024;
        } else {
          const int n = lane >> 2;
          voff[u] = (uint32_t)min(g0 + (n >> 2), groups - 1) * wrow + (n & 3) * 256 +
                    (((lane & 3) ^ (n >> 2)) << 4);
          uoff[u] = (oo >> 1) * kPassBytes + (oo & 1) * 1024;
          uslot[u] = 64;
        }
      }
      const int bstages = stages / SUB;
      auto issue = [&](int s, int buf) __attribute__((always_inline)) {
        // the stage's first unit (and four slots of its pass)
        const uint32_t unit = SEG == 1 ? (uint32_t)s : (uint32_t)(s >> 2) * SEG;
        const uint32_t quarter = SEG == 1 ? 0u : (uint32_t)(s & 3);
        static_for<Sh::DB>([&](auto U) __attribute__((always_inline)) {
          constexpr int u = decltype(U)::value;
          const DmaStage st =
              dma_stage(s, bstages, unit * kPassBytes + uoff[u] + quarter * uslot[u]);
          const auto r = rsrc_of(base[u], st);
          const auto to = (lds_void *)(smem + Sh::BOFF + buf * Sh::BSZ + dst[u]);
          // up to 16 rows one workgroup alone reads these weights: non-temporal
          // (M = 16, N = 9216, K = 2560 13.9 -> 12.9 us from HBM; at 32 rows
          // 4 % less from HBM, 10 % more for weights that fit the 256 MB
          // cache behind it)
          constexpr int kNt = RT == 1 ? 2 : 0;
          if constexpr (u < Sh::DQ || SEG == 1)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(r, to, 16, voff[u], st.offset, 0, kNt);
          else
            __builtin_amdgcn_raw_ptr_buffer_load_lds(r, to, 4, voff[u], st.offset, 0, kNt);
        });
      };
#pragma unroll
      for (int i = 0; i < NB; ++i) issue(i, i);
      wait_vmcnt16<((NB - 1) * Sh::DB < 63 ? (NB - 1) * Sh::DB : 63)>();
      barrier16();
      for (int s = 0, buf = 0; s < bstages; ++s) {
#pragma unroll
        for (int i = 0; i < SUB - 1; ++i) barrier16();
        wait_vmcnt16<(NB - 2) * Sh::DB>();  // weight stage s + 1 is there
        barrier16();
        issue(s + NB, buf);
        buf = buf + 1 == NB ? 0 : buf + 1;
      }
    }
    // no DMA may land in LDS after the workgroup has released it (or, with
    // DUAL, after the compute waves have taken the rings for their sums)
    wait_vmcnt16<0>();
    if constexpr (DUAL) barrier16();
    return;
  }

  // ---- compute waves
  const int wr = wave % RT, wt = wave / RT;  // its row tile and tile of B
  const int wc = wt / NM;
  const int rt16 = mg * RT + wr;  // this wave's 16-row tile
  if ((int64_t)rt16 * 16 >= p.m_rows) {
    for (int t = 0; t <= stages; ++t) barrier16();
    if constexpr (DUAL) barrier16();
    return;
  }
  const int li = lane & 15, lq = lane >> 4;
  // A: lane (row li, quarter lq) of a block pair; scales: (row li, block lq)
  const uint32_t aaddr = wr * 4096 + lane * 16;
  const uint32_t saddr = Sh::ASCALE + wr * 512 + lq * 64 + li * 4;
  // B: lane (row n = li, half lq & 1 of block lq >> 1 of a pair)
  constexpr int BA = SEG == 1 ? 8 : 4;
  uint32_t baddr[BA];
#pragma unroll
  for (int j = 0; j < BA; ++j) {
    if constexpr (SEG == 1)
      baddr[j] = ((li >> 2) * 2 + (lq & 1)) * 1024 + (li & 3) * 256 +
                 (((2 * j + (lq >> 1)) ^ li) << 4);
    else
      baddr[j] = (lq & 1) * 1024 + (lq >> 1) * 2048 + li * 64 + ((j ^ (li >> 2)) << 4);
    baddr[j] += Sh::BOFF + wt * Sh::TILE;
  }
  // weight scales: lane (row li, block 4q + lq of the weight stage)
  constexpr int QB = Sh::SB / 4;  // quads per weight stage
  uint32_t daddr[SEG == 6 ? QB : 1];
#pragma unroll
  for (int q = 0; q < (SEG == 6 ? QB : 1); ++q) {
    const int e = 4 * q + lq;
    const int i = SEG == 1 ? 0 : e % SEG, sl = SEG == 1 ? e : e / SEG;
    daddr[q] = Sh::BOFF + wt * Sh::TILE + Sh::QOPS * 1024 +
               (SEG == 1 ? (li >> 2) * 128 + 2 * (16 * (li & 3) + sl) : i * 128 + li * 8 + 2 * sl);
  }

  // operands of two block pairs: A as the MFMAs take them, B as read
  v4i fa[2], fb[2];
  float fs;
  uint16_t fd;
  // Operands of the step of the A stage at place T of the unrolled rings and
  // its quad Q (0, 1).
  auto read_ops = [&](auto T, auto Q) __attribute__((always_inline)) {
    constexpr int T_ = decltype(T)::value, q = decltype(Q)::value;
    constexpr int a0 = T_ % NA * Sh::ASZ;
    constexpr int b0 = T_ / SUB % NB * Sh::BSZ;
    constexpr int qb = T_ % SUB * 2 + q;  // quad of the weight stage
#pragma unroll
    for (int j = 0; j < 2; ++j) fa[j] = *(const v4i *)(smem + aaddr + (a0 + (2 * q + j) * 1024));
    fs = *(const float *)(smem + saddr + (a0 + q * 256));
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int e = 4 * qb + 2 * j;  // the pair's even block
      if constexpr (SEG == 1) fb[j] = *(const v4i *)(smem + baddr[e >> 1] + b0);
      else fb[j] = *(const v4i *)(smem + baddr[e / SEG] + (b0 + e % SEG * 2048));
    }
    fd = *(const uint16_t *)(smem + daddr[SEG == 6 ? qb : 0] +
                             (b0 + (SEG == 1 ? 8 * qb : SEG == 4 ? 2 * qb : 0)));
  };

  v4i cc[4], cn[4];
  v16f fc, fn;
  float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  // Lanes 0-31 of fb hold the even block of the pair (both halves of its
  // values), lanes 32-63 the odd one: swapping the upper lanes of the first
  // eight bytes with the lower lanes of the last eight gives each block an
  // operand of its own, its values in the order of tile16_offset.
  auto dots = [&](v4i (&c)[4]) __attribute__((always_inline)) {
    const v4i zero = {0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const auto lo = __builtin_amdgcn_permlane32_swap(fb[j][0], fb[j][2], false, false);
      const auto hi = __builtin_amdgcn_permlane32_swap(fb[j][1], fb[j][3], false, false);
      const v2u b0 = {lo[0], hi[0]}, b1 = {lo[1], hi[1]};
      const v2i a0 = {fa[j][0], fa[j][1]}, a1 = {fa[j][2], fa[j][3]};
      c[2 * j] = __builtin_amdgcn_mfma_i32_16x16x32_i8(
          __builtin_bit_cast(long, a0), __builtin_bit_cast(long, b0), zero, 0, 0, 0);
      c[2 * j + 1] = __builtin_amdgcn_mfma_i32_16x16x32_i8(
          __builtin_bit_cast(long, a1), __builtin_bit_cast(long, b1), zero, 0, 0, 0);
    }
  };
  auto scales = [&]() __attribute__((always_inline)) -> v16f {
    const v16f z = {};
    return __builtin_amdgcn_mfma_f32_16x16x1f32(fs, half_bits_to_float(fd), z, 0, 0, 0);
  };

  auto stage_steps = [&](auto T) __attribute__((always_inline)) {
    static_for<2>([&](auto K) __attribute__((always_inline)) {
      constexpr int T_ = decltype(T)::value;
      dots(cn);
      fn = scales();
#pragma unroll
      for (int j = 0; j < 4; ++j) asm volatile("" ::"v"(cn[j]));
      asm volatile("" ::"v"(fn));
      if constexpr (decltype(K)::value == 0) barrier16();
      read_ops(std::integral_constant<int, (T_ + 1) % Sh::PERIOD>{}, K);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const float dotf = (float)cc[j][v];
          const float f = fc[4 * j + v];
          if (FMA) {
            acc[v] = __builtin_fmaf(dotf, f, acc[v]);
          } else {
            const float contrib = dotf * f;
            acc[v] = acc[v] + contrib;
          }
        }
#pragma unroll
      for (int v = 0; v < 4; ++v) asm volatile("" : "+v"(acc[v]));
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < 4; ++j) cc[j] = cn[j];
      fc = fn;
    });
  };

  barrier16();
  {
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    read_ops(I0{}, I0{});
    dots(cc);
    fc = scales();
    read_ops(I0{}, I1{});
  }
  for (int t0 = 0; t0 < stages; t0 += Sh::PERIOD)
    static_for<Sh::PERIOD>([&](auto T) __attribute__((always_inline)) {
      const int t = t0 + decltype(T)::value;
      if (t < stages) stage_steps(T);
    });

  typedef float v4f __attribute__((ext_vector_type(4)));
  float up[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  if constexpr (DUAL) {
    // every DMA has landed and every operand has been read: the up waves'
    // sums take the rings' place
    barrier16();
    v4f *const box = (v4f *)(smem + (wc * RT + wr) * 1024 + lane * 16);
    if (wt & 1) {
      *box = v4f{acc[0], acc[1], acc[2], acc[3]};
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    }
    barrier16();
    if (wt & 1) return;
    const v4f u = *box;
#pragma unroll
    for (int v = 0; v < 4; ++v) up[v] = u[v];
  }

  const int n = nc0 + 16 * wc + li;
  const int64_t m0 = (int64_t)rt16 * 16 + 4 * lq;
  float o[4];
  activate_array(acc, DUAL ? ACT_SILU : gw.act);
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    o[v] = acc[v];
    if constexpr (DUAL)
      o[v] = p.y_bf16 ? bf16_to_float(float_to_bf16(o[v])) * bf16_to_float(float_to_bf16(up[v]))
                      : o[v] * up[v];
  }
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int64_t m = m0 + v;
    if (m >= p.m_rows || n >= n_rows) continue;
    if (p.y_bf16) {
      if (p.add)
        o[v] = bf16_to_float(float_to_bf16(o[v])) +
               bf16_to_float(((const uint16_t *)p.add)[m * p.ldr + n]);
      ((uint16_t *)gw.y)[m * gw.ldy + n] = float_to_bf16(o[v]);
    } else {
      if (p.add) o[v] = o[v] + ((const float *)p.add)[m * p.ldr + n];
      ((float *)gw.y)[m * gw.ldy + n] = o[v];
    }
  }
#endif
}

template <int SEG, bool FMA, int RT, int CN, bool DUAL>
hipError_t launch16(Gemm16Args &a, const Gemm16Launch &l, int32_t row_tiles16, hipStream_t s) {
  a.m_groups = (row_tiles16 + RT - 1) / RT;
  a.n_groups = 0;
  for (int i = 0; i < l.count; ++i) {
    a.g[i].group0 = a.n_groups;
    a.n_groups += (int32_t)((l.w[i].rows + 16 * CN - 1) / (16 * CN));
  }
  const int64_t grid = (int64_t)((a.n_groups + 7) / 8 * 8) * a.m_groups;
  typedef Gemm16Shape<SEG, RT, CN, DUAL> Sh;
  hipLaunchKernelGGL((gemm16_kernel<SEG, FMA, RT, CN, DUAL>), dim3((unsigned)grid),
                     dim3(Sh::THREADS), 0, s, a);
  return hipGetLastError();
}

// The workgroup shape for rts 16-row tiles and `tiles` column tiles: rows
// first (a column tile's weights are fetched once per RT rows), then the
// fewest columns that put every workgroup on a CU of its own.  `per_block`
// is a round's time per block of K, in us, fitted with 5 us of launch, fill
// and input quantization to op times within 2 us (f32, aarch64): (1, 1) 8.0 ..
// 8.4 us at K = 2560, 19.0 at 9216; (1, 4) 12.5 at N = 9216, K = 2560; (4, 1)
// 10.9 / 13.7 / 24.0 at K = 2560 / 4096 / 9216; (4, 2) 13.4 / - / 31.8; (4, 3)
// 16.0 / 21.9 / 43.3; SwiGLU (1, 1) 10.9 at N = 2560, 16.8 at 9216, (2, 3)
// 23.5, (4, 1) 13.8 .. 14.9 at K = 2560.
struct Shape16 {
  int rt, cn;
  double per_block;
};
Shape16 shape16(int64_t rts, int64_t tiles, int seg, bool dual) {
  const int64_t cus = cu_count();
  if (dual) {
    if (rts == 1) return {1, 1, 0.06};
    // three column pairs do not fit the LDS with S = 6
    if (rts == 2) return tiles <= cus || seg == 6 ? Shape16{2, 1, 0.11} : Shape16{2, 3, 0.24};
    return {4, 1, 0.14};
  }
  if (rts == 1) {
    if (tiles <= cus) return {1, 1, 0.05};
    return tiles <= 2 * cus ? Shape16{1, 2, 0.06} : Shape16{1, 4, 0.10};
  }
  if (rts == 2) {
    if (tiles <= cus) return {2, 1, 0.055};
    return tiles <= 2 * cus ? Shape16{2, 2, 0.08} : Shape16{2, 4, 0.15};
  }
  const int64_t wgs = (rts + 3) / 4 * tiles;
  if (wgs <= cus) return {4, 1, 0.065};
  return wgs <= 2 * cus ? Shape16{4, 2, 0.10} : Shape16{4, 3, 0.14};
}

// Rounds of workgroups, at most one per CU.
int64_t rounds16(const Shape16 &sh, int64_t rts, int64_t tiles) {
  const int64_t wgs = (rts + sh.rt - 1) / sh.rt * ((tiles + sh.cn - 1) / sh.cn);
  const int64_t cus = cu_count();
  return (wgs + cus - 1) / cus;
}

template <int SEG, bool FMA>
hipError_t launch16_f(Gemm16Args &a, const Gemm16Launch &l, int32_t rts, const Shape16 &sh,
                      bool dual, hipStream_t s) {
  const int code = sh.rt * 10 + sh.cn;
  if (dual) {
    switch (code) {
      case 11: return launch16<SEG, FMA, 1, 1, true>(a, l, rts, s);
      case 21: return launch16<SEG, FMA, 2, 1, true>(a, l, rts, s);
      case 41: return launch16<SEG, FMA, 4, 1, true>(a, l, rts, s);
    }
    if constexpr (SEG != 6)
      if (code == 23) return launch16<SEG, FMA, 2, 3, true>(a, l, rts, s);
    return hipErrorInvalidValue;
  }
  switch (code) {
    case 11: return launch16<SEG, FMA, 1, 1, false>(a, l, rts, s);
    case 12: return launch16<SEG, FMA, 1, 2, false>(a, l, rts, s);
    case 14: return launch16<SEG, FMA, 1, 4, false>(a, l, rts, s);
    case 21: return launch16<SEG, FMA, 2, 1, false>(a, l, rts, s);
    case 22: return launch16<SEG, FMA, 2, 2, false>(a, l, rts, s);
    case 24: return launch16<SEG, FMA, 2, 4, false>(a, l, rts, s);
    case 41: return launch16<SEG, FMA, 4, 1, false>(a, l, rts, s);
    case 42: return launch16<SEG, FMA, 4, 2, false>(a, l, rts, s);
    case 43: return launch16<SEG, FMA, 4, 3, false>(a, l, rts, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace

// The cheaper of the two GEMMs by the fitted op times.  launch_gemm, exact:
// up to 64 rows 1 + 0.18 us per block for one 64 x 64 workgroup per CU (13.9
// .. 15.8 us at K = 2560, 27 at 4096, 53 .. 56 at 9216) and 1 + 0.28 for each
// two (188 us at N = 248320, K = 2560, M = 32), above 0.33 us per block and
// round of 128 x 96 ones (26 .. 30 us at K = 2560, 45 at 4096, 105 at 9216),
// for each weight apart.  Op times launch_gemm -> launch_gemm16:
// N = 2560, K = 9216 M = 2 / 64 / 256 / 512 53.1 / 55.8 / 105.5 / 106.8 ->
// 18.5 / 24.0 / 42.9 / 76.9; N = 2560, K = 2560 M = 64 / 256 / 320 13.9 /
// 26.1 / 26.6 -> 10.9 / 16.0 / 25.5 (the last not taken); N = 9216, K = 2560
// M = 16 / 32 / 64 15.0 / 15.3 / 15.8 -> 11.9 / 14.6 / 16.7 (the last two not
// taken); its SwiGLU M = 16 / 32 / 64 29.5 / 30.2 / 31.0 -> 16.7 / 23.5 / 36.0
// (the last not taken); N = 2560, K = 9216 / 4096, M = 333 106.2 / 46.1 -> 69.2 /
// 36.5.
// SPLIT_K is no choice to make here: what splits K must depend on the one
// linear, whatever else shares its launch, so the caller keeps linears that
// split on launch_gemm.
bool gemm16_takes(int64_t m, const int64_t *rows, int count, int64_t cols, bool dual) {
  if (m <= 1) return false;
  const int64_t cus = cu_count(), units = passes_for(cols), rts = (m + 15) / 16;
  const double blocks = (double)units * kPassBlocks;
  int64_t tiles = 0;
  double old_us = 0;
  for (int i = 0; i < count; ++i) {
    tiles += (rows[i] + 15) / 16;
    const int64_t wgs = m <= 64 ? (rows[i] + 63) / 64 : (m + 127) / 128 * ((rows[i] + 95) / 96);
    const double us = m > 64     ? (double)((wgs + cus - 1) / cus) * 0.33 * blocks
                      : wgs <= cus ? 1.0 + 0.18 * blocks
                                   : (double)((wgs + 2 * cus - 1) / (2 * cus)) * (1.0 + 0.28 * blocks);
    old_us += us * (dual ? 2 : 1);
  }
  const Shape16 sh = shape16(rts, tiles, seg_for(units), dual);
  return 5.0 + (double)rounds16(sh, rts, tiles) * sh.per_block * blocks < old_us;
}

void gemm16_instance(int64_t m, const int64_t *rows, int count, int64_t cols, bool dual,
                     int32_t *seg, int32_t *row_tiles, int32_t *col_tiles) {
  int64_t tiles = 0;
  for (int i = 0; i < count; ++i) tiles += (rows[i] + 15) / 16;
  *seg = seg_for(passes_for(cols));
  const Shape16 sh = shape16((m + 15) / 16, tiles, *seg, dual);
  *row_tiles = sh.rt;
  *col_tiles = sh.cn;
}

hipError_t launch_gemm16(const Gemm16Launch &l, hipStream_t s) {
  Gemm16Args a = {};
  a.qa = l.qa;
  a.sa = l.sa;
  a.add = l.add;
  a.ldr = l.ldr;
  a.m_rows = l.m;
  a.row_tiles = (int32_t)((l.m + 15) / 16);
  a.units = (int32_t)passes_for(l.cols);
  a.y_bf16 = l.y_bf16 ? 1 : 0;
  a.count = l.count;
  const int32_t rts = a.row_tiles;
  bool dual = false;
  int64_t tiles = 0;
  for (int i = 0; i < l.count; ++i) {
    const Gemm16Launch::Weight &w = l.w[i];
    a.g[i] = {w.w, w.up, w.y, w.ldy, (int32_t)w.rows, w.activation, 0};
    tiles += (w.rows + 15) / 16;
    dual |= w.up != nullptr;
  }
  if (dual && (l.count != 1 || l.add)) return hipErrorInvalidValue;
  const int seg = seg_for(a.units);
  const Shape16 sh = shape16(rts, tiles, seg, dual);
  switch (seg) {
    case 6:
      return l.fma ? launch16_f<6, true>(a, l, rts, sh, dual, s)
                   : launch16_f<6, false>(a, l, rts, sh, dual, s);
    case 4:
      return l.fma ? launch16_f<4, true>(a, l, rts, sh, dual, s)
                   : launch16_f<4, false>(a, l, rts, sh, dual, s);
    default:
      return l.fma ? launch16_f<1, true>(a, l, rts, sh, dual, s)
                   : launch16_f<1, false>(a, l, rts, sh, dual, s);
  }
}

}  // namespace llmcp_q8
