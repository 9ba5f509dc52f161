// The SSD core of f32 inputs at d_state 64 / 128 as a walk along each (batch,
// head) chain, 64 tokens a step, with the state [P, N] in registers
// (workloads/mamba/model_ref.py:139-162 at a 64-token block; every chunking
// evaluates the same recurrence):
//   y[l, p]  = sum_{s<=l} exp(Acs[l]-Acs[s]) (C_l . B_s) dt[s] x[s, p]
//              + exp(Acs[l]) sum_n C[l, n] S[p, n]
//   S[p, n] <- exp(Acs[63]) S[p, n] + sum_l exp(Acs[63]-Acs[l]) dt[l] x[l, p] B[l, n]
// x is read once and y written once; no per-chunk state reaches memory.
//
// A workgroup takes two heads of one (batch, group), two waves per head; wave w
// owns p rows 32 w .. 32 w + 31 of the state and of y.  Every product is a
// 32x32x2 f32 MFMA on f32 values, and each result is the next one's operand in
// the registers it already lies in: an accumulator's register 4 k + jj holds
// row 8 k + 4 (lane / 32) + jj and column lane % 32, an operand's lane row (or
// column) lane % 32 and K slot lane / 32, so with the K slots of a product
// dealt out in accumulator row order
//   * S^T (rows n, columns p) is the A operand of the off-diagonal product,
//   * W = decay . C.B^T (rows s, columns l) the B operand of the diagonal one,
//   * x^T, loaded from memory straight into 32 registers per lane, its A
//     operand and, weighted, the B operand of the state update.
// Only B and C pass through LDS, each in one buffer: C is read in a step's
// first phase while B is copied, B in the second while the next C is.
//
// Bound: the f32 MFMAs (1/16 of the 16-bit rate).  At 64 x 512 tokens, 64 heads,
// d_state 64 they keep the matrix cores busy for 79% of the scan's 425 us (three
// workgroups per CU; two: 540 us) and the VALU adds 16%.  Measured (us per call,
// stage kernels -> walk): that shape 714 -> 501, 32 x 1024, 32 heads, d_state 128
// 541 -> 370, 16 x 512, 64 heads, d_state 64 189 -> 137.  No gain: wave
// priorities by phase, a fixed interleaving of MFMA, VALU and LDS instructions.
// W in registers for the whole step (formed between the off-diagonal products)
// does not fit beside x, S and y; so each wave forms it four values at a time.
#include "ssd_chain_step.h"
#include "../../include/ssd.h"

namespace ssd {

namespace {

constexpr int kP = 64;
constexpr int kHeads = 2;             // heads per workgroup
constexpr int kWaves = 2 * kHeads;

typedef float f32x16 __attribute__((ext_vector_type(16)));
__device__ __forceinline__ f32x16 mma2(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

template <int N, bool HAS_DT>
__global__ __launch_bounds__(64 * kWaves, N == 64 ? 3 : 2) void chain_scan_f32_kernel(ChainScanArgs p) {
  constexpr int NT = N / 32;
  constexpr int PPR = N / 4, RPB = 64 / PPR;        // 16-byte pieces per row of B / C, rows per 1 KB copy
  constexpr int DPW = kStep * N / 256 / kWaves;     // copies per wave
  constexpr int NY = 8 + 32;                        // y stores and x loads left in flight at the second barrier
  __shared__ __attribute__((aligned(1024))) float bs[kStep * N];
  __shared__ __attribute__((aligned(1024))) float cl[kStep * N];
  __shared__ __attribute__((aligned(256))) float al[2][kHeads][kStep];
  __shared__ __attribute__((aligned(256))) float dl[HAS_DT ? 2 : 1][HAS_DT ? kHeads : 1][HAS_DT ? kStep : 4];
  __shared__ __attribute__((aligned(256))) float wt[kWaves][kStep];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hh = wave >> 1, w = wave & 1;
  const int hl = lane >> 5, r = lane & 31, g = lane >> 4, i = lane & 15;

  // ---- unit: (batch, two heads of one group), heads fastest ----
  const int hb = p.nheads / kHeads;
  const int u = xcd_remap(blockIdx.x, gridDim.x);
  const int h0 = (u % hb) * kHeads, b = u / hb;
  const int h = h0 + hh, grp = h0 / (p.nheads / p.ngroups);
  const int last = p.nsteps - 1;

  // ---- copies of B and C rows: block wave + 4 m, rows RPB (wave + 4 m) + lane / PPR.
  // C: piece k of row l at slot k ^ (l & 15) (operand reads take one piece of 32
  // rows); B: at slot k ^ 8 ((l >> 2) & 1) (one column of rows l and l + 4).
  const char* bg = (const char*)uni(reinterpret_cast<const float*>(p.bm) + (int64_t)b * p.sbb + (int64_t)grp * p.sbg);
  const char* cg = (const char*)uni(reinterpret_cast<const float*>(p.cm) + (int64_t)b * p.scb + (int64_t)grp * p.scg);
  const char* cbg = (const char*)uni(reinterpret_cast<const f32x4*>(p.cb) + ((int64_t)b * p.nsteps * p.ngroups + grp) * kTiles * 64);
  const char* ag = (const char*)uni(p.acs + ((int64_t)b * p.nheads + h) * p.nsteps * kStep);
  const char* dg = HAS_DT ? (const char*)uni(p.dt + (int64_t)b * p.sdb + (int64_t)h * p.sdh) : nullptr;
  const float* xg = uni(reinterpret_cast<const float*>(p.x) + (int64_t)b * p.sxb + (int64_t)h * p.sxh + 32 * w);
  const int64_t bst = (int64_t)kStep * p.sbl * 4, cst = (int64_t)kStep * p.scl * 4, dst = (int64_t)kStep * p.sdl * 4;
  const int64_t cbst = (int64_t)p.ngroups * kTiles * 1024;
  const int64_t brow = (int64_t)RPB * kWaves * p.sbl * 4, crow = (int64_t)RPB * kWaves * p.scl * 4;
  const int row0 = RPB * wave + lane / PPR, slot = lane % PPR;
  const uint32_t bv = (uint32_t)(row0 * (int)p.sbl + 4 * (slot ^ (8 * ((row0 >> 2) & 1)))) * 4;
  // rows 8 further on (N = 128, odd m) have the other half's swizzle
  const uint32_t cv0 = (uint32_t)(row0 * (int)p.scl + 4 * (slot ^ (row0 & 15))) * 4;
  const uint32_t cv1 = (uint32_t)(row0 * (int)p.scl + 4 * (slot ^ ((row0 + RPB * kWaves) & 15))) * 4;
  const uint32_t bs_o = uni(lds_offset(bs)) + wave * 1024, cl_o = uni(lds_offset(cl)) + wave * 1024;
  const uint32_t al_o = uni(lds_offset(al)) + hh * 256, dl_o = uni(lds_offset(dl)) + hh * 256;
  const uint32_t dv = HAS_DT ? (uint32_t)(lane * (int)p.sdl) * 4 : 0;
  auto issue_b = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int m = 0; m < DPW; ++m) dma16_s(bg + m * brow, bv, bs_o + m * (kWaves * 1024));
  };
  auto issue_c = [&](int bf) __attribute__((always_inline)) {
#pragma unroll
    for (int m = 0; m < DPW; ++m) dma16_s(cg + m * crow, m & 1 ? cv1 : cv0, cl_o + m * (kWaves * 1024));
    if (w == 0) dma4_s(ag, lane * 4, al_o + (uint32_t)(bf * kHeads * 256));
    else if constexpr (HAS_DT) dma4_s(dg, dv, dl_o + (uint32_t)(bf * kHeads * 256));
  };

  // C.B^T in the diagonal product's order: groups of four s, k of block q (tokens
  // l 32 (q > 0) .., s 32 (q > 1) ..): s = 8 k + 4 hl + jj, l = r, from the 16 x 16
  // tile (t, s tile) = (2 (q > 0) + r / 16, 2 (q > 1) + k / 2) in chain_prep's
  // numbering; above the diagonal (masked below) the diagonal tile.  The groups
  // go blocks 0 and 1 in turn, then block 2; each is loaded three groups early.
  constexpr int kBlk[12] = {0, 1, 0, 1, 0, 1, 0, 1, 2, 2, 2, 2}, kGrp[12] = {0, 0, 1, 1, 2, 2, 3, 3, 0, 1, 2, 3};
  f32x4 cb[4];
  uint32_t cbv[3][2];
  {
    const uint32_t lo = (uint32_t)(hl * 16 + i) * 16;
    const bool t1 = (r >> 4) != 0;
    cbv[0][0] = lo + (t1 ? 4 : 0) * 1024, cbv[0][1] = lo + (t1 ? 1 : 0) * 1024;
    cbv[1][0] = lo + (t1 ? 9 : 6) * 1024, cbv[1][1] = lo + (t1 ? 7 : 8) * 1024;
    cbv[2][0] = lo + (t1 ? 5 : 2) * 1024, cbv[2][1] = lo + (t1 ? 3 : 2) * 1024;
  }
  auto load_cb = [&](int e) __attribute__((always_inline)) {
    const int q = kBlk[e], k = kGrp[e];
    cb[e & 3] = load16_b(cbg, cbv[q][k >> 1] + 512 * (k & 1));
  };
  // x: register 4 k + jj of block q: token 32 q + 8 k + 4 hl + jj, p = 32 w + r
  float xr[2][16];
  const uint32_t xv = (uint32_t)(4 * hl * (int)p.sxl + r) * 4;
  auto load_x = [&](__amdgpu_buffer_rsrc_t rs, int q, int j) __attribute__((always_inline)) {
    const uint32_t row = (uint32_t)(32 * q + 8 * (j >> 2) + (j & 3)) * (uint32_t)p.sxl * 4;
    xr[q][j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, xv, row, 0));
  };

  issue_c(0);
#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int j = 0; j < 16; ++j) load_x(rsrc(xg), q, j);

  // S^T tiles: st[nt][4 k + jj] = S[p = 32 w + r][n = 32 nt + 8 k + 4 hl + jj]
  f32x16 st[NT];
  const int64_t so = ((int64_t)b * p.nheads + h) * (kP * N) + (32 * w + r) * N + 4 * hl;
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const f32x4 v = p.init ? *reinterpret_cast<const f32x4*>(p.init + so + 32 * nt + 8 * k) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) st[nt][4 * k + jj] = v[jj];
    }
  // y: 16 rows of 64 bytes per instruction
  float* yg = const_cast<float*>(uni(reinterpret_cast<const float*>(p.y) + (int64_t)b * p.syb + (int64_t)h * p.syh + 32 * w));
  const uint32_t yv = (uint32_t)(i * (int)p.syl + 4 * (2 * (g & 1) + hl)) * 4;
  const int coff = r * PPR + (hl ^ (r & 15));  // C: piece 2 kk + hl, group kk by ^ 2 kk
  const int boff[2] = {4 * hl * N + r + 32 * hl, 4 * hl * N + r - 32 * hl};

  dma_wait();
  __syncthreads();

  for (int c = 0; c <= last; ++c) {
    // ---- first phase: weights, W, the off-diagonal product ----
    const int bf = c & 1;
    issue_b();
#pragma unroll
    for (int e = 0; e < 3; ++e) load_cb(e);
    const float* ab = al[bf][hh];
    const float a_own = ab[lane];
    const float aq = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(a_own), 63));
    const float dec = __builtin_amdgcn_exp2f(aq * kLog2e);
    {
      float wv = __builtin_amdgcn_exp2f((aq - a_own) * kLog2e);
      if constexpr (HAS_DT) wv *= dl[bf][hh][lane];
      wt[wave][lane] = wv;
    }
    float al2[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) al2[t] = ab[32 * t + r] * kLog2e;
    f32x16 acc[2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int j = 0; j < 16; ++j) acc[t][j] = 0.f;
    int co = coff;
    asm volatile("" : "+v"(co));  // (the groups' addresses are formed in the step: kept, they would not fit the registers)
    auto read_c = [&](f32x4 (&cf)[2], int kk) __attribute__((always_inline)) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
        cf[t] = reinterpret_cast<const f32x4*>(cl)[(co ^ (2 * kk)) + 32 * t * PPR];
    };
    f32x4 cf[2][2];
    read_c(cf[0], 0);
#pragma unroll
    for (int kk = 0; kk < 4 * NT; ++kk) {
      if (kk + 1 < 4 * NT) read_c(cf[(kk + 1) & 1], kk + 1);
#pragma unroll
      for (int jj = 0; jj < 4; ++jj)
#pragma unroll
        for (int t = 0; t < 2; ++t) acc[t] = mma2(st[kk >> 2][4 * (kk & 3) + jj], cf[kk & 1][t][jj], acc[t]);
      // the state's decay, its value entering the step being taken
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) st[kk >> 2][4 * (kk & 3) + jj] *= dec;
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) acc[t] *= __builtin_amdgcn_exp2f(al2[t]);
    dma_wait();
    __syncthreads();

    // ---- second phase: the diagonal product, y, the state update ----
    auto form_w = [&](int e) __attribute__((always_inline)) {
      const int q = kBlk[e], k = kGrp[e], s0 = 32 * (q > 1) + 8 * k + 4 * hl;
      const f32x4 as = *reinterpret_cast<const f32x4*>(ab + s0);
      f32x4 v;
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) v[jj] = cb[e & 3][jj] * __builtin_amdgcn_exp2f(__builtin_fmaf(as[jj], -kLog2e, al2[q > 0]));
      if constexpr (HAS_DT) v *= *reinterpret_cast<const f32x4*>(&dl[bf][hh][s0]);
      if (q != 1) {
        // the diagonal blocks; selection, not a product with the mask: exp2 above the diagonal may be inf
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) v[jj] = 8 * k + 4 * hl + jj <= r ? v[jj] : 0.f;
      }
      return v;
    };
    f32x4 wv4[2];
    wv4[0] = form_w(0);
    load_cb(3);
#pragma unroll
    for (int e = 0; e < 12; ++e) {
      const int q = kBlk[e], k = kGrp[e];
      if (e + 1 < 12) wv4[(e + 1) & 1] = form_w(e + 1);
      if (e + 4 < 12) load_cb(e + 4);
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) acc[q > 0] = mma2(xr[q > 1][4 * k + jj], wv4[e & 1][jj], acc[q > 0]);
      __builtin_amdgcn_sched_barrier(0);
    }
    const int64_t nx = c < last ? 1 : 0;  // (the last step copies itself again)
    bg += nx * bst;
    cg += nx * cst;
    cbg += nx * cbst;
    ag += nx * (kStep * 4);
    if constexpr (HAS_DT) dg += nx * dst;
    xg += nx * kStep * p.sxl;
    issue_c(bf ^ 1);
    auto store_y = [&](int t) __attribute__((always_inline)) {
#pragma unroll
      for (int k = 0; k < 4; k += 2) {
        f32x4 oa, ob;
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
          const auto q2 = __builtin_amdgcn_permlane16_swap(__float_as_uint(acc[t][4 * k + jj]), __float_as_uint(acc[t][4 * k + 4 + jj]), false, false);
          oa[jj] = __uint_as_float(q2[0]);
          ob[jj] = __uint_as_float(q2[1]);
        }
        typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
        // (the rows' offsets in the base: with one in a scalar register the compiler
        // does not keep a write to the data registers off the store's heels)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, oa), rsrc(yg + (int64_t)(32 * t) * p.syl), yv + 32 * k, 0, 0);
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, ob), rsrc(yg + (int64_t)(32 * t + 16) * p.syl), yv + 32 * k, 0, 0);
      }
    };
    // four tokens of B: columns 32 nt + r of rows 32 q + 8 k + 4 hl + jj
    auto read_b = [&](float (&bq)[NT][4], int kk) __attribute__((always_inline)) {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) bq[nt][jj] = bs[boff[nt & 1] + (8 * kk + jj) * N + 32 * nt];
    };
    auto read_wt = [&](int kk) __attribute__((always_inline)) { return *reinterpret_cast<const f32x4*>(&wt[wave][8 * kk + 4 * hl]); };
    float bq[2][NT][4];
    f32x4 wx[2], w4 = read_wt(0);
    read_b(bq[0], 0);
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) wx[0][jj] = xr[0][jj] * w4[jj];
    w4 = read_wt(1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) {
      // this group's products; the next one's operands between them
      if (kk < 7) {
        read_b(bq[(kk + 1) & 1], kk + 1);
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) wx[(kk + 1) & 1][jj] = xr[(kk + 1) >> 2][4 * ((kk + 1) & 3) + jj] * w4[jj];
      }
      if (kk < 6) w4 = read_wt(kk + 2);
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) load_x(rsrc(xg), kk >> 2, 4 * (kk & 3) + jj);
#pragma unroll
      for (int jj = 0; jj < 4; ++jj)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) st[nt] = mma2(bq[kk & 1][nt][jj], wx[kk & 1][jj], st[nt]);
      if (kk == 1) store_y(0);
      if (kk == 3) store_y(1);
      __builtin_amdgcn_sched_barrier(0);
    }
    yg += (int64_t)kStep * p.syl;
    accesses_before_wait();
    vm_wait<NY>();
    __syncthreads();
  }
  // the copies past the last step land before this workgroup's LDS is given away
  dma_wait();
  if (p.final_state) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int k = 0; k < 4; ++k)
        *reinterpret_cast<f32x4*>(p.final_state + so + 32 * nt + 8 * k) = f32x4{st[nt][4 * k], st[nt][4 * k + 1], st[nt][4 * k + 2], st[nt][4 * k + 3]};
  }
}

template <int N>
hipError_t launch_n(const ChainScanArgs& a, hipStream_t stream) {
  const int64_t grid = (int64_t)a.batch * (a.nheads / kHeads);
  if (grid > INT32_MAX) return hipErrorInvalidValue;
  auto kern = a.dt ? chain_scan_f32_kernel<N, true> : chain_scan_f32_kernel<N, false>;
  kern<<<dim3((unsigned)grid), dim3(64 * kWaves), 0, stream>>>(a);
  return hipGetLastError();
}

}  // namespace

// Whole chains, where there is more than one workgroup (two chains) per CU.
// Measured (us, stage kernels / walk; L 1024, 64 heads): 288 workgroups on 256 CUs
// 309 / 220 at d_state 64 and 430 / 332 at 128; 480 402 / 240 and 1227 / 351.  With fewer
// than one per CU, one wave per SIMD leaves the matrix cores idle for half a step:
// 96 workgroups (8 x 2048, 24 heads, d_state 128) 210 / 349, 128 267 / 358, 192
// (d_state 64) 136 / 123.  With exactly one per CU the walk would win (277 / 190 at
// d_state 128, 190 / 137 at 64); the line leaves it to the stage kernels, whose own
// entry points give the forward's bits.
ChainScanPlan chain_scan_f32_plan(int64_t batch, int64_t steps, int64_t nheads, int64_t ngroups, int64_t dstate) {
  const ChainScanPlan none{0, 0, false};
  if ((dstate != 64 && dstate != 128) || (nheads / ngroups) % kHeads != 0) return none;
  const int64_t cus = device_cu_count() > 0 ? device_cu_count() : 256;
  if (batch * nheads / kHeads <= cus) return none;
  return ChainScanPlan{1, (int)steps, false};
}

hipError_t launch_chain_prep_f32(const ChainScanArgs& a, const CumsumArgs& ca, int dstate, hipStream_t stream) {
  if (ca.chunk != kStep || ca.dt_raw) return hipErrorInvalidValue;
  return dstate == 64 ? launch_chain_prep_t<float, 2, float, false>(a, ca, stream) : launch_chain_prep_t<float, 4, float, false>(a, ca, stream);
}

hipError_t launch_chain_scan_f32(const ChainScanArgs& a, int dstate, hipStream_t stream) {
  return dstate == 64 ? launch_n<64>(a, stream) : launch_n<128>(a, stream);
}

}  // namespace ssd
