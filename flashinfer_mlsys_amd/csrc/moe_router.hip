// Router GEMM: routing_logits [T, 256] fp32 = hidden [T, 7168] bf16 x gate [256, 7168]^T bf16,
// the linear layer that produces the operator's routing_logits input (reference
// moe/weight_origins_dataflow.md:21, :151-154: "x @ gate_weight.T (linear layer,
// no activation)"). bf16 x bf16 products are exact in fp32; sums run in fp32 on the
// bf16 MFMA (v_mfma_f32_16x16x32_bf16).
//
// Small T (< 576 tokens): one launch; a workgroup computes 16 tokens x 16 experts
// over the whole K, its 8 waves taking 7 of the 56 K blocks each with operands
// loaded straight into MFMA fragment registers (all 56 loads in flight at once),
// then the 8 partial tiles are added through LDS in wave order (deterministic, no
// atomics, no workspace).
//
// With QUANT the kernels also write the operator's FP8 activation inputs (e4m3 rows [T,
// 7168] and 1 x 128 block scales [56, T]) from the hidden states they read anyway, with
// the quantiser kernel's arithmetic, each (token, K block) exactly once. In the small-T
// kernel the workgroup of expert tile y quantises the K blocks kb with kb % 16 == y from
// the fragments it holds (one pass over x instead of two: 15 us instead of 20 at T=64).
// In the tiled kernels 4 more waves do it beside the GEMM (see rq_run; the same work in the
// GEMM's compute waves took 84 us at T=8192, against 49 + 40 for the two kernels).
//
// Larger T: LDS-staged tiles of 128 tokens x 64 experts, 8 compute waves of
// 32 x 32 (v_mfma_f32_32x32x16_bf16) and 4 loader waves that stream each 128-wide
// K block (hidden rows and gate rows, whole 128 B lines, 32-row swizzle) into a
// 3-slot LDS ring two blocks ahead. Between 576 tokens
// and the token count whose 32-token items fill the CUs once (2,048 on 256 CUs),
// router_ksplit_kernel: 32 x 64 tiles, a 5-slot ring, each K block's MFMA steps
// split over the 8 compute waves and the four K quarters added in LDS in a
// fixed order.
#include "moe_common.h"
#include "moe_host.h"
#include "moe_tile.h"
#include "moe_quant_block.h"

namespace moe {

constexpr int RT_M = 16;  // tokens per small-T tile

__device__ __forceinline__ v8bf load_bf16x8(const uint16_t* p) {
  return __builtin_bit_cast(v8bf, *reinterpret_cast<const v4i*>(p));
}

constexpr int RS_WAVES = 8;
constexpr int RS_KPW = NB_H / RS_WAVES;  // 7 K blocks per wave

template <bool QUANT>
__global__ __launch_bounds__(64 * RS_WAVES) void router_small_kernel(const uint16_t* __restrict__ x,
                                                                     const uint16_t* __restrict__ g, int T,
                                                                     float* __restrict__ logits, uint8_t* __restrict__ q,
                                                                     float* __restrict__ qs) {
  __shared__ float red[RS_WAVES][4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int fr = lane & 15, kg = lane >> 4;
  const int t0 = blockIdx.x * RT_M, e0 = blockIdx.y * 16;
  const int k0 = wave * RS_KPW * BLK;
  const uint16_t* xp = x + (size_t)min(t0 + fr, T - 1) * H + k0 + 8 * kg;
  const uint16_t* gp = g + (size_t)(e0 + fr) * H + k0 + 8 * kg;
  v8bf a[RS_KPW][4], b[RS_KPW][4];
#pragma unroll
  for (int kk = 0; kk < RS_KPW; ++kk)
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      a[kk][s] = load_bf16x8(xp + kk * BLK + 32 * s);
      b[kk][s] = load_bf16x8(gp + kk * BLK + 32 * s);
    }
  __builtin_amdgcn_sched_barrier(0);  // all 56 loads in flight before the first product waits
  v4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kk = 0; kk < RS_KPW; ++kk)
#pragma unroll
    for (int s = 0; s < 4; ++s) acc = mfma_bf16_k32(a[kk][s], b[kk][s], acc);
#pragma unroll
  for (int r = 0; r < 4; ++r) red[wave][r][lane] = acc[r];
  if (QUANT) {
    // lane (fr, kg) holds K 32 s + 8 kg + [0, 8) of token row fr for s = 0..3; the
    // row's 4 lanes are fr, fr + 16, fr + 32, fr + 48
    const int t = t0 + fr;
#pragma unroll
    for (int kk = 0; kk < RS_KPW; ++kk) {
      const int kb = wave * RS_KPW + kk;
      if (kb % 16 != (int)blockIdx.y) continue;  // wave-uniform
      float v[4][8];
      float m = 0.f;
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4) {
        const v4i w = __builtin_bit_cast(v4i, a[kk][s4]);
        const uint32_t wu[4] = {(uint32_t)w[0], (uint32_t)w[1], (uint32_t)w[2], (uint32_t)w[3]};
        bf16x8_to_f32(wu, v[s4]);
#pragma unroll
        for (int i = 0; i < 8; ++i) m = fmaxf(m, fabsf(v[s4][i]));
      }
      m = fmaxf(m, __shfl_xor(m, 16));
      m = fmaxf(m, __shfl_xor(m, 32));
      const float sc = qblock_scale(m);
      const QDiv dv = qblock_div(sc);
      if (t < T) {
#pragma unroll
        for (int s4 = 0; s4 < 4; ++s4) {
          const uint32_t p0 = qblock_pack4(v[s4][0], v[s4][1], v[s4][2], v[s4][3], dv);
          const uint32_t p1 = qblock_pack4(v[s4][4], v[s4][5], v[s4][6], v[s4][7], dv);
          *reinterpret_cast<uint2*>(q + (size_t)t * H + kb * BLK + 32 * s4 + 8 * kg) = uint2{p0, p1};
        }
        if (kg == 0) qs[(size_t)kb * T + t] = sc;
      }
    }
  }
  __syncthreads();
  if (threadIdx.x < 256) {  // entry (r, lane): token row 4 (lane / 16) + r, expert column lane % 16
    const int r = threadIdx.x >> 6, ln = threadIdx.x & 63;
    float v = red[0][r][ln];
#pragma unroll
    for (int w = 1; w < RS_WAVES; ++w) v += red[w][r][ln];
    const int t = t0 + 4 * (ln >> 4) + r;
    if (t < T) logits[(size_t)t * E_GLOBAL + e0 + (ln & 15)] = v;
  }
}

// Quantiser waves of the tiled kernels (QUANT): 4 more waves a workgroup quantise its
// items' tokens while the others run the GEMM, the workgroup of expert tile nt the K
// blocks 14 nt .. 14 nt + 13 of them, so each (token, block) once. They take every
// barrier of the K loop (a barrier counts all of a workgroup's waves) and do an equal
// share of the item between two of them, their loads RQ_D steps ahead; x comes from
// the caches, where the GEMM's own loads of the same rows bring it. A unit is 4 tokens
// x 1 block: 16 lanes per token, 8 values (16 B) per lane. What bounds them is their
// vector instructions between two barriers (with a division per value a K block took
// 1.3 us instead of the GEMM's 0.6), hence the 3-instruction quotients and the paths of
// finite blocks.
constexpr int RQ_WAVES = 4, RQ_D = 4;
constexpr int RQ_KB = NB_H / (E_GLOBAL / 64);  // 14 blocks per expert tile
typedef unsigned int v2u __attribute__((ext_vector_type(2)));
struct RQuant {
  __amdgpu_buffer_rsrc_t rx, rq, rs;
  int T, lane, p;  // p: quantiser wave
};
__device__ __forceinline__ RQuant rq_make(const uint16_t* x, int T, uint8_t* q, float* qs, int p) {
  RQuant r;
  r.rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(x), (short)0, (int)((uint32_t)T * (H * 2)), 0x00020000);
  r.rq = __builtin_amdgcn_make_buffer_rsrc(q, (short)0, (int)((uint32_t)T * H), 0x00020000);
  r.rs = __builtin_amdgcn_make_buffer_rsrc(qs, (short)0, (int)((uint32_t)T * (NB_H * 4)), 0x00020000);
  r.T = T; r.lane = threadIdx.x & 63; r.p = p;
  return r;
}
// Units of token groups tg .. tg + NU - 1 from this lane's token t0, block kb. Rows at or past T
// are out of the resources' ranges: zeros read, nothing written. The row is all in the vector
// offset, which alone decides the bounds check (the scalar offset stays inside a row).
template <int NU>
__device__ __forceinline__ void rq_load(const RQuant& r, int t0, int tg, int kb, v4i (&raw)[NU]) {
#pragma unroll
  for (int n = 0; n < NU; ++n)
    raw[n] = __builtin_bit_cast(
        v4i, __builtin_amdgcn_raw_buffer_load_b128(r.rx, (uint32_t)(t0 + 4 * (tg + n)) * (H * 2) + (r.lane & 15) * 16,
                                                   kb * (BLK * 2), 0));
}
template <int NU>
__device__ __forceinline__ void rq_store(const RQuant& r, int t0, int tg, int kb, const v4i (&raw)[NU]) {
  float v[NU][8], s[NU];
  uint32_t o[NU][2];
  bool finite = true;
#pragma unroll
  for (int n = 0; n < NU; ++n) {
    const uint32_t w[4] = {(uint32_t)raw[n][0], (uint32_t)raw[n][1], (uint32_t)raw[n][2], (uint32_t)raw[n][3]};
    bf16x8_to_f32(w, v[n]);
    const float m = __uint_as_float(row16_max_bf16(w) << 16);  // NaN if a value is
    s[n] = qblock_scale_finite(m);
    qblock_pack8_finite(w, v[n], QDiv{s[n], __builtin_amdgcn_rcpf(s[n])}, o[n]);
    finite = finite && m < __builtin_inff();
  }
  if (__builtin_expect(__builtin_amdgcn_ballot_w64(!finite) != 0, 0)) {
#pragma unroll
    for (int n = 0; n < NU; ++n) {
      float m = 0.f;  // (the maximum of the block skips NaNs)
#pragma unroll
      for (int i = 0; i < 8; ++i) m = fmaxf(m, fabsf(v[n][i]));
#pragma unroll
      for (int k = 1; k < 16; k <<= 1) m = fmaxf(m, __shfl_xor(m, k));
      s[n] = qblock_scale(m);
      const QDiv d = qblock_div(s[n]);
      o[n][0] = qblock_pack4(v[n][0], v[n][1], v[n][2], v[n][3], d);
      o[n][1] = qblock_pack4(v[n][4], v[n][5], v[n][6], v[n][7], d);
    }
  }
#pragma unroll
  for (int n = 0; n < NU; ++n) {
    const int t = t0 + 4 * (tg + n);
    __builtin_amdgcn_raw_buffer_store_b64(v2u{o[n][0], o[n][1]}, r.rq, (uint32_t)t * H + (r.lane & 15) * 8, kb * BLK, 0);
    const bool first = (r.lane & 15) == 0 && t < r.T;  // (t < T: a row of the transposed scales must not run on)
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(s[n]), r.rs, first ? (uint32_t)t * 4 : 0xF0000000u,
                                          (uint32_t)kb * r.T * 4, 0);
  }
}
// All items of a workgroup (first, first + gridDim.x, ...): at each of an item's first STEPS K
// blocks NU units a wave, token groups NU (k % TGS) .. of block k / TGS; EXTRA more
// barriers after each item's last K block.
template <int BM, int NU, int EXTRA>
__device__ __forceinline__ void rq_run(const RQuant& r, int first, int n_items) {
  constexpr int NT = E_GLOBAL / 64, TG = BM / 4 / RQ_WAVES, TGS = TG / NU, STEPS = TGS * RQ_KB;
  static_assert(TG % NU == 0 && STEPS <= NB_H && STEPS % RQ_D == 0 && NB_H % RQ_D == 0 && RQ_D % TGS == 0, "steps");
  auto token = [&](int i) {  // this lane's first token in item i (past the end: out of range)
    const int item = first + i * (int)gridDim.x;
    return (i < n_items ? item / NT * BM : r.T) + 4 * r.p * TG + (r.lane >> 4);
  };
  auto block = [&](int i) { return (first + i * (int)gridDim.x) % NT * RQ_KB; };
  v4i buf[RQ_D][NU];
  int t0 = token(0), kb0 = block(0);
#pragma unroll
  for (int d = 0; d < RQ_D; ++d) rq_load<NU>(r, t0, d % TGS * NU, kb0 + d / TGS, buf[d]);
#pragma unroll 1
  for (int i = 0; i < n_items; ++i) {
    const int t1 = token(i + 1), kb1 = block(i + 1);
#pragma unroll 1
    for (int k = 0; k < NB_H; k += RQ_D) {
      const bool last = k + RQ_D >= STEPS;
      const int tn = last ? t1 : t0, kn = last ? kb1 : kb0 + (k + RQ_D) / TGS;
#pragma unroll
      for (int d = 0; d < RQ_D; ++d) {
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (STEPS == NB_H || k < STEPS) {  // uniform
          rq_store<NU>(r, t0, d % TGS * NU, kb0 + k / TGS + d / TGS, buf[d]);
          rq_load<NU>(r, tn, d % TGS * NU, kn + d / TGS, buf[d]);
        }
      }
    }
#pragma unroll
    for (int e = 0; e < EXTRA; ++e) __builtin_amdgcn_s_barrier();
    t0 = t1;
    kb0 = kb1;
  }
}

constexpr int RT2_BM = 128;                                  // tokens per item
constexpr int RT2_BN = 64;                                   // experts per item
constexpr int RT2_NT = E_GLOBAL / RT2_BN;                    // 4 expert tiles
constexpr int RT2_REG = 4096;                                // 32 rows x 128 B
constexpr int RT2_A_BYTES = RT2_BM * BLK * 2;                // 32 KB: 4 row blocks x 2 lines
constexpr int RT2_STAGE = RT2_A_BYTES + RT2_BN * BLK * 2;    // + 16 KB: 2 row blocks x 2 lines
constexpr int RT2_NSTAGE = 3;
constexpr int RT2_CWAVES = 8, RT2_PWAVES = 4;
constexpr int RT2_JOBS = RT2_STAGE / 1024 / RT2_PWAVES;      // 12 load instructions per loader wave per block
constexpr int RT2_MIN_T = 576;
static_assert(RT2_JOBS * RT2_PWAVES * 1024 == RT2_STAGE, "load split");

template <bool QUANT>
__global__ __launch_bounds__(64 * (RT2_CWAVES + RT2_PWAVES + (QUANT ? RQ_WAVES : 0)), 1) void router_tiled_kernel(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ g, int T, float* __restrict__ logits,
    uint8_t* __restrict__ q, float* __restrict__ qs) {
  extern __shared__ __attribute__((aligned(16))) uint8_t rt_lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int total = (T + RT2_BM - 1) / RT2_BM * RT2_NT;
  const int first = xcd_remap(blockIdx.x, gridDim.x);
  int n_items = 0;
  for (int item = first; item < total; item += gridDim.x) ++n_items;
  const int G = n_items * NB_H;

  if (QUANT && wave >= RT2_CWAVES + RT2_PWAVES) {
    rq_run<RT2_BM, 2, 0>(rq_make(x, T, q, qs, wave - RT2_CWAVES - RT2_PWAVES), first, n_items);
    return;
  }
  if (wave >= RT2_CWAVES) {
    // loader wave p: jobs 12 p .. 12 p + 11 of the 48 per block (0-31 hidden rows,
    // 32-47 gate rows); a job moves 8 rows x 128 B (one line of a K block)
    const int p = wave - RT2_CWAVES, ld_row = lane >> 3;
    const uint8_t* src[RT2_JOBS];
    int dst[RT2_JOBS];
    int item = first - (int)gridDim.x, kb = NB_H, slot = 0;
    auto next_item = [&]() {
      item += gridDim.x;
      const int mt = item / RT2_NT, nt = item % RT2_NT;
#pragma unroll
      for (int i = 0; i < RT2_JOBS; ++i) {
        const int job = p * RT2_JOBS + i, rg = job & 3, h = (job >> 2) & 1;
        const int chunk = (lane & 7) ^ ld_row ^ (rg & 1);
        if (job < 32) {
          const int ib = job >> 3;
          const int row = min(mt * RT2_BM + ib * 32 + rg * 8 + ld_row, T - 1);
          src[i] = reinterpret_cast<const uint8_t*>(x + (size_t)row * H) + h * 128 + chunk * 16;
          dst[i] = (ib * 2 + h) * RT2_REG + rg * 1024;
        } else {
          const int jb = (job - 32) >> 3;
          const int e = nt * RT2_BN + jb * 32 + rg * 8 + ld_row;
          src[i] = reinterpret_cast<const uint8_t*>(g + (size_t)e * H) + h * 128 + chunk * 16;
          dst[i] = RT2_A_BYTES + (jb * 2 + h) * RT2_REG + rg * 1024;
        }
      }
      kb = 0;
    };
    auto issue = [&]() {
      if (kb == NB_H) next_item();
      uint8_t* st = rt_lds + slot * RT2_STAGE;
#pragma unroll
      for (int i = 0; i < RT2_JOBS; ++i) lds_direct16(src[i] + kb * 2 * BLK, st + dst[i]);  // 256 B per K block
      slot = slot == RT2_NSTAGE - 1 ? 0 : slot + 1;
      ++kb;
    };
    if (G > 0) issue();
    if (G > 1) issue();
#pragma unroll 1
    for (int gi = 0; gi < G; ++gi) {
      if (gi + 1 < G) asm volatile("s_waitcnt vmcnt(12)" ::: "memory");  // 12 loads per block
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if (gi + 2 < G) issue();
    }
    return;
  }

  // compute wave: tokens 32 wm .. of the item, experts 32 wn ..; MFMA step t of a
  // block reads, from line t / 4 of the row, 16 B chunk 4 ((t / 2) % 2) + 2 lg + t % 2
  // (the same for both operands, so the K pairing holds)
  const int wm = wave & 3, wn = wave >> 2;
  const int lr = lane & 31, lg = lane >> 5;
  int off[2][2];
#pragma unroll
  for (int ph = 0; ph < 2; ++ph)
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) off[ph][tt] = sw32(lr, 4 * ph + 2 * lg + tt);
  int slot = 0;
  for (int item = first; item < total; item += gridDim.x) {
    const int mt = item / RT2_NT, nt = item % RT2_NT;
    v16f acc = v16f{};
#pragma unroll 1
    for (int kb = 0; kb < NB_H; ++kb) {
      __builtin_amdgcn_s_barrier();  // block kb is in its slot; the slot before it is free
      asm volatile("" ::: "memory");
      const uint8_t* st = rt_lds + slot * RT2_STAGE;
      slot = slot == RT2_NSTAGE - 1 ? 0 : slot + 1;
      const uint8_t* sa = st + (wm * 2) * RT2_REG;
      const uint8_t* sb = st + RT2_A_BYTES + (wn * 2) * RT2_REG;
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        const int line = t >> 2, ph = (t >> 1) & 1, tt = t & 1;
        const v8bf a = *reinterpret_cast<const v8bf*>(sa + line * RT2_REG + off[ph][tt]);
        const v8bf b = *reinterpret_cast<const v8bf*>(sb + line * RT2_REG + off[ph][tt]);
        acc = mfma_bf16_32x32x16(a, b, acc);
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this block's LDS reads are done
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int t = mt * RT2_BM + wm * 32 + 8 * (i >> 2) + 4 * lg + (i & 3);
      if (t < T) logits[(size_t)t * E_GLOBAL + nt * RT2_BN + wn * 32 + lr] = acc[i];
    }
  }
}

// Middle T (from RT2_MIN_T tokens while its items fit on the CUs: 2,048 tokens on
// 256 CUs): the tiled kernel has fewer items than CUs there, and each item's 56 K
// blocks pass a 3-slot ring one memory latency per two blocks (33-36 us whatever
// T; 19-21 us here). Here an item is 32 tokens x 64 experts,
// so four times as many workgroups take part, and its stage (24 KB: one 32-row
// block of hidden rows, two of gate rows) fits a 5-slot ring, four blocks ahead.
// The 8 compute waves split each K block: wave (wn, kq) takes MFMA steps 2 kq and
// 2 kq + 1 of expert half wn, so every wave keeps one 32 x 32 accumulator; after
// the last block the four K quarters are added through LDS in kq order (a fixed
// order; no atomics).
constexpr int RT3_BM = 32;
constexpr int RT3_A_BYTES = RT3_BM * BLK * 2;                // 8 KB: 2 lines
constexpr int RT3_STAGE = RT3_A_BYTES + RT2_BN * BLK * 2;    // + 16 KB: 2 row blocks x 2 lines
constexpr int RT3_NSTAGE = 5;
constexpr int RT3_JOBS = RT3_STAGE / 1024 / RT2_PWAVES;      // 6 load instructions per loader wave per block
constexpr int RT3_RED = 8 * 16 * 64 * 4;                     // 8 waves x 16 values x 64 lanes
constexpr int RT3_LDS = RT3_NSTAGE * RT3_STAGE + RT3_RED;
static_assert(RT3_JOBS * RT2_PWAVES * 1024 == RT3_STAGE && RT3_LDS <= 160 * 1024, "stage");

// s_waitcnt vmcnt for n of the loader's blocks still in flight (n <= 3)
__device__ __forceinline__ void rt3_wait_blocks(int n) {
  switch (n) {
    case 3: asm volatile("s_waitcnt vmcnt(18)" ::: "memory"); break;
    case 2: asm volatile("s_waitcnt vmcnt(12)" ::: "memory"); break;
    case 1: asm volatile("s_waitcnt vmcnt(6)" ::: "memory"); break;
    default: asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); break;
  }
}

template <bool QUANT>
__global__ __launch_bounds__(64 * (RT2_CWAVES + RT2_PWAVES + (QUANT ? RQ_WAVES : 0)), 1) void router_ksplit_kernel(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ g, int T, float* __restrict__ logits,
    uint8_t* __restrict__ q, float* __restrict__ qs) {
  extern __shared__ __attribute__((aligned(16))) uint8_t rt_lds[];
  float* red = reinterpret_cast<float*>(rt_lds + RT3_NSTAGE * RT3_STAGE);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int total = (T + RT3_BM - 1) / RT3_BM * RT2_NT;
  const int first = xcd_remap(blockIdx.x, gridDim.x);
  int n_items = 0;
  for (int item = first; item < total; item += gridDim.x) ++n_items;
  const int G = n_items * NB_H;

  if (QUANT && wave >= RT2_CWAVES + RT2_PWAVES) {
    // (28 units a wave and item: one at each of the first 28 K blocks)
    rq_run<RT3_BM, 1, 1>(rq_make(x, T, q, qs, wave - RT2_CWAVES - RT2_PWAVES), first, n_items);
    return;
  }
  if (wave >= RT2_CWAVES) {
    // loader wave p: jobs 6 p .. 6 p + 5 of the 24 per block (0-7 hidden rows,
    // 8-23 gate rows); a job moves 8 rows x 128 B (one line of a K block)
    const int p = wave - RT2_CWAVES, ld_row = lane >> 3;
    const uint8_t* src[RT3_JOBS];
    int dst[RT3_JOBS];
    int item = first - (int)gridDim.x, kb = NB_H, slot = 0;
    auto next_item = [&]() {
      item += gridDim.x;
      const int mt = item / RT2_NT, nt = item % RT2_NT;
#pragma unroll
      for (int i = 0; i < RT3_JOBS; ++i) {
        const int job = p * RT3_JOBS + i;
        const int chunk_row = ld_row;
        if (job < 8) {
          const int rg = job & 3, h = job >> 2;
          const int row = min(mt * RT3_BM + rg * 8 + ld_row, T - 1);
          src[i] = reinterpret_cast<const uint8_t*>(x + (size_t)row * H) + h * 128 +
                   ((lane & 7) ^ chunk_row ^ (rg & 1)) * 16;
          dst[i] = h * RT2_REG + rg * 1024;
        } else {
          const int jj = job - 8, rg = jj & 3, h = (jj >> 2) & 1, jb = jj >> 3;
          const int e = nt * RT2_BN + jb * 32 + rg * 8 + ld_row;
          src[i] = reinterpret_cast<const uint8_t*>(g + (size_t)e * H) + h * 128 +
                   ((lane & 7) ^ chunk_row ^ (rg & 1)) * 16;
          dst[i] = RT3_A_BYTES + (jb * 2 + h) * RT2_REG + rg * 1024;
        }
      }
      kb = 0;
    };
    auto issue = [&]() {
      if (kb == NB_H) next_item();
      uint8_t* st = rt_lds + slot * RT3_STAGE;
#pragma unroll
      for (int i = 0; i < RT3_JOBS; ++i) lds_direct16(src[i] + kb * 2 * BLK, st + dst[i]);  // 256 B per K block
      slot = slot == RT3_NSTAGE - 1 ? 0 : slot + 1;
      ++kb;
    };
    for (int b = 0; b < RT3_NSTAGE - 1 && b < G; ++b) issue();
#pragma unroll 1
    for (int gi = 0; gi < G; ++gi) {
      rt3_wait_blocks(min(RT3_NSTAGE - 2, G - 1 - gi));  // block gi is in
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if (gi + RT3_NSTAGE - 1 < G) issue();
      if (gi % NB_H == NB_H - 1) __builtin_amdgcn_s_barrier();  // the compute waves' K-quarter sum
    }
    return;
  }

  // compute wave (wn, kq): experts 32 wn .. of the item, MFMA steps 2 kq, 2 kq + 1
  // of every K block; step t reads, from line t / 4 of the row, 16 B chunk
  // 4 ((t / 2) % 2) + 2 lg + t % 2 (the same for both operands)
  const int wn = wave & 1, kq = wave >> 1;
  const int lr = lane & 31, lg = lane >> 5;
  int off[2];
#pragma unroll
  for (int tt = 0; tt < 2; ++tt) off[tt] = sw32(lr, 4 * (kq & 1) + 2 * lg + tt);
  const int line = kq >> 1;
  int slot = 0;
  for (int item = first; item < total; item += gridDim.x) {
    const int mt = item / RT2_NT, nt = item % RT2_NT;
    v16f acc = v16f{};
#pragma unroll 1
    for (int kb = 0; kb < NB_H; ++kb) {
      __builtin_amdgcn_s_barrier();  // block kb is in its slot; the slot before it is free
      asm volatile("" ::: "memory");
      const uint8_t* st = rt_lds + slot * RT3_STAGE;
      slot = slot == RT3_NSTAGE - 1 ? 0 : slot + 1;
      const uint8_t* sa = st + line * RT2_REG;
      const uint8_t* sb = st + RT3_A_BYTES + (wn * 2 + line) * RT2_REG;
#pragma unroll
      for (int tt = 0; tt < 2; ++tt) {
        const v8bf a = *reinterpret_cast<const v8bf*>(sa + off[tt]);
        const v8bf b = *reinterpret_cast<const v8bf*>(sb + off[tt]);
        acc = mfma_bf16_32x32x16(a, b, acc);
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this block's LDS reads are done
    }
    // the K quarters: wave w's 16 values per lane to LDS, then wave w takes expert
    // half w % 2, values 4 (w / 2) .. + 3, and adds the quarters in kq order
#pragma unroll
    for (int i = 0; i < 16; ++i) red[(wave * 16 + i) * 64 + lane] = acc[i];
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int ii = 0; ii < 4; ++ii) {
      const int i = 4 * kq + ii;  // this wave's value index (kq doubles as the value group)
      float v = red[((0 * 2 + wn) * 16 + i) * 64 + lane];
#pragma unroll
      for (int q = 1; q < 4; ++q) v += red[((q * 2 + wn) * 16 + i) * 64 + lane];
      const int t = mt * RT3_BM + 8 * (i >> 2) + 4 * lg + (i & 3);
      if (t < T) logits[(size_t)t * E_GLOBAL + nt * RT2_BN + wn * 32 + lr] = v;
    }
  }
}

hipError_t launch_quantize_1x128(const uint16_t* x, int T, uint8_t* q, float* scale, hipStream_t stream);

// Whether the quantiser waves pay from RT2_MIN_T tokens on: the tiled kernel's first few
// token counts leave a quarter of the CUs busy, whose quantiser waves then take longer than
// the quantiser kernel on all of them. Both steps, us, in turn / together, calls back to back
// on the same buffers: T=1,024 25.9 / 23.2, 2,048 29.0 / 25.6 | 2,049 42.8 / 46.6, 2,304
// 43.2 / 46.4, 2,816 45.5 / 46.8 | 3,000 46.3 / 45.7, 4,100 51.1 / 48.4, 8,192 68.8 / 54.2,
// 14,107 138 / 128 (one call with the caches full of other data: 2,304 68.3 / 74.4, 3,000
// 73.4 / 69.9, 8,192 103 / 99).
constexpr int RQ_MIN_TILED_T = 3000;
static bool rq_fused(int T, int cu) {
  return T >= RQ_MIN_TILED_T || (T + RT3_BM - 1) / RT3_BM * RT2_NT <= cu;
}

// (q, qs null: the logits alone)
static hipError_t launch_router_tiled(const uint16_t* x, const uint16_t* g, int T, float* logits, uint8_t* q, float* qs,
                                      int cu, hipStream_t stream) {
  static PerDeviceOnce<hipError_t> once;
  hipError_t e = hipErrorInvalidDevice;
  once.get([] {
    const hipError_t r = hipFuncSetAttribute(reinterpret_cast<const void*>(router_tiled_kernel<false>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, RT2_NSTAGE * RT2_STAGE);
    return r != hipSuccess ? r
                           : hipFuncSetAttribute(reinterpret_cast<const void*>(router_tiled_kernel<true>),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, RT2_NSTAGE * RT2_STAGE);
  }, e);
  if (e != hipSuccess) return e;
  const int items = (T + RT2_BM - 1) / RT2_BM * RT2_NT;
  const int grid = min((items + 7) / 8 * 8, (cu + 7) / 8 * 8);
  const int threads = 64 * (RT2_CWAVES + RT2_PWAVES + (q ? RQ_WAVES : 0));
  if (q) hipLaunchKernelGGL(router_tiled_kernel<true>, dim3(grid), dim3(threads), RT2_NSTAGE * RT2_STAGE, stream, x, g, T,
                            logits, q, qs);
  else hipLaunchKernelGGL(router_tiled_kernel<false>, dim3(grid), dim3(threads), RT2_NSTAGE * RT2_STAGE, stream, x, g, T,
                          logits, q, qs);
  return hipGetLastError();
}

static hipError_t launch_router_ksplit(const uint16_t* x, const uint16_t* g, int T, float* logits, uint8_t* q, float* qs,
                                       int cu, hipStream_t stream) {
  static PerDeviceOnce<hipError_t> once;
  hipError_t e = hipErrorInvalidDevice;
  once.get([] {
    const hipError_t r = hipFuncSetAttribute(reinterpret_cast<const void*>(router_ksplit_kernel<false>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, RT3_LDS);
    return r != hipSuccess ? r
                           : hipFuncSetAttribute(reinterpret_cast<const void*>(router_ksplit_kernel<true>),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, RT3_LDS);
  }, e);
  if (e != hipSuccess) return e;
  const int items = (T + RT3_BM - 1) / RT3_BM * RT2_NT;
  const int grid = min((items + 7) / 8 * 8, (cu + 7) / 8 * 8);
  const int threads = 64 * (RT2_CWAVES + RT2_PWAVES + (q ? RQ_WAVES : 0));
  if (q) hipLaunchKernelGGL(router_ksplit_kernel<true>, dim3(grid), dim3(threads), RT3_LDS, stream, x, g, T, logits, q, qs);
  else hipLaunchKernelGGL(router_ksplit_kernel<false>, dim3(grid), dim3(threads), RT3_LDS, stream, x, g, T, logits, q, qs);
  return hipGetLastError();
}

// the tiled GEMM by token count: 32-token items with the K steps split over the
// waves while they fit on the CUs in one round, 128-token items beyond
static hipError_t launch_router_gemm(const uint16_t* x, const uint16_t* g, int T, float* logits, uint8_t* q, float* qs,
                                     int cu, hipStream_t stream) {
  return (T + RT3_BM - 1) / RT3_BM * RT2_NT <= cu ? launch_router_ksplit(x, g, T, logits, q, qs, cu, stream)
                                                  : launch_router_tiled(x, g, T, logits, q, qs, cu, stream);
}

hipError_t launch_router_logits(const uint16_t* x, const uint16_t* g, int T, float* logits, int cu,
                                hipStream_t stream) {
  if (T <= 0) return hipSuccess;
  if (T >= RT2_MIN_T) return launch_router_gemm(x, g, T, logits, nullptr, nullptr, cu, stream);
  hipLaunchKernelGGL(router_small_kernel<false>, dim3((T + RT_M - 1) / RT_M, E_GLOBAL / 16), dim3(64 * RS_WAVES), 0,
                     stream, x, g, T, logits, nullptr, nullptr);
  return hipGetLastError();
}

hipError_t launch_router_quantize(const uint16_t* x, const uint16_t* g, int T, float* logits, uint8_t* q, float* qs,
                                  int cu, hipStream_t stream) {
  if (T <= 0) return hipSuccess;
  if (T >= RT2_MIN_T) {
    if (!rq_fused(T, cu)) {
      const hipError_t e = launch_router_gemm(x, g, T, logits, nullptr, nullptr, cu, stream);
      return e != hipSuccess ? e : launch_quantize_1x128(x, T, q, qs, stream);
    }
    return launch_router_gemm(x, g, T, logits, q, qs, cu, stream);
  }
  hipLaunchKernelGGL(router_small_kernel<true>, dim3((T + RT_M - 1) / RT_M, E_GLOBAL / 16), dim3(64 * RS_WAVES), 0,
                     stream, x, g, T, logits, q, qs);
  return hipGetLastError();
}

}  // namespace moe
