// The SSD core of 16-bit inputs at d_state 128 as a walk along each (batch,
// head) chain, 64 tokens a step, with the state [P, N] in f32 registers
// (workloads/mamba/model_ref.py:139-162 at a 64-token block; every chunking
// evaluates the same recurrence):
//   y[l, p]  = sum_{s<=l} exp(Acs[l]-Acs[s]) (C_l . B_s) dt[s] x[s, p]
//              + exp(Acs[l]) sum_n C[l, n] S[p, n]
//   S[p, n] <- exp(Acs[63]) S[p, n] + sum_l exp(Acs[63]-Acs[l]) dt[l] x[l, p] B[l, n]
// x is read once and y written once; no per-chunk state reaches memory, where
// the stage kernels write and read one per 256 (or 64) tokens and read x twice.
//
// Launches: chain_prep_kernel (64-token cumsums; C.B^T per (batch, step,
// group), and for bf16 inputs C as f16 rows with a power-of-two scale each),
// then chain_scan_kernel.  Chains too few to fill the GPU are cut into
// segments: chain_state_kernel first finds each segment's own end state, from
// which the state entering each segment follows.
//
// A scan workgroup takes HPW heads of one (batch, group), two waves per head;
// wave w owns p rows 32 w .. 32 w + 31 of the state and of y.  All products
// are 32x32x16 MFMAs arranged so that each result is the next one's operand
// without leaving its lane:
//   * S^T tiles (rows n, columns p) are accumulators; the n rows of a tile are
//     dealt out (by the addresses of the transposing B reads) so that a lane's
//     values are 8 consecutive n, the A operand of the off-diagonal product.
//     They are rounded to f16 there, as SSD_STATE_F16S rounds states: with a
//     power-of-two scale per row p, the row's largest magnitude in [2^14, 2^15).
//   * y^T tiles (rows p, columns l) start as the off-diagonal product, are
//     scaled by exp(Acs[l]), and take the diagonal product on top.
//   * W = decay . C.B^T is formed once per head, its ten causal 16 x 16 tiles
//     shared out over the two waves, and handed round through LDS in operand
//     order.
//   * x^T (from row-major x through ds_read_b64_tr_b16) is the A operand of
//     the diagonal product and, weighted, the B operand of the state update.
//     The weights go onto x (32 values per lane and step), as a hi + lo pair
//     of the input type, rather than onto B^T, which every wave needs whole.
//
// Bound: issue.  At batch 4 x 4096, 80 heads the MFMAs are busy for 36% and the
// VALU for 59% of the busy CUs' cycles (1 x 65536 the same, 8 x 2048 of 128 heads
// 38% and 57%, gated 25% and 61%; counters), and the two do not overlap on one
// SIMD.  Measured (us per call, stage kernels -> walk): batch 8 x 2048 tokens, 128
// heads, 8 groups, f16: 365 -> 201, the layer span there 567 -> 365; batch 4 x
// 4096, 80 heads, bf16: 197 -> 171 (3 segments); 1 x 65536, 80 heads: 800 -> 711
// (38 segments); with S as a hi + lo pair, layer span 2 x 1216 of 128 heads: 250
// -> 100 (one f16 there: 98).  The scale of every row costs 1-2% of a call: with rows
// inside [2^-9, 2^15) left as they were, 4 x 4096 took 166.0 us instead of 167.5,
// 1 x 65536 683 instead of 698 (f16 then loses bits below 2^-14).
// Slower: two 16-row halves per wave on 16x16x32 MFMAs (twice the LDS reads: 437
// against 387 us for the layer span), the MFMAs of a step behind all its copies
// (a copy stalls its wave while others queue: 6% of a step).
#include "ssd_chain_step.h"
#include "../../include/ssd.h"

namespace ssd {

namespace {

constexpr int kQ = kStep;    // tokens per step
constexpr int kP = 64;       // head dim
constexpr int kN = 128;      // d_state
constexpr int kWBlocks = 6;  // 32 (s) x 16 (l) blocks of W

typedef float f32x16 __attribute__((ext_vector_type(16)));
__device__ __forceinline__ f32x16 mma32(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x16 mma32(f16x8 a, f16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// HILO: S goes into the off-diagonal product as a hi + lo pair of the input type,
// one product each (f16 pairs of the scaled rows; bf16, whose exponents are f32's,
// of the values as they are, with C as it lies).
template <typename T, int HPW, bool HAS_DT, bool EPI, bool HILO>
__global__ __launch_bounds__(128 * HPW, 2) void chain_scan_kernel(ChainScanArgs p) {
  constexpr int NW = 2 * HPW;
  constexpr bool kF16 = std::is_same<T, f16>::value;
  constexpr bool kCT = !kF16 && !HILO;   // C from chain_prep's f16 rows
  constexpr bool kRows = kF16 || !HILO;  // S as f16 rows with a scale each
  typedef typename std::conditional<HILO, T, f16>::type E;  // of the off-diagonal operands
  constexpr int NX = 4 + (EPI ? 4 : 0);  // x copies and z loads left in flight at the first barrier
  constexpr int NY = 5 + 4;              // C.B^T loads and y stores left in flight at the second
  constexpr int DPW = 16 / NW;         // B (C) copies per wave
  __shared__ __attribute__((aligned(1024))) T bs[kQ * kN];
  __shared__ __attribute__((aligned(1024))) E cl[kQ * kN];
  __shared__ __attribute__((aligned(1024))) T xs[HPW * 2][kQ * kP];
  __shared__ __attribute__((aligned(1024))) T wl[HPW][kWBlocks * 64 * 8];
  // per head: Acs, dt and C row scales of the step's tokens; per wave: their
  // weights and the row scales of S
  __shared__ __attribute__((aligned(256))) float al[HPW][kQ];
  __shared__ __attribute__((aligned(256))) float dl[HAS_DT ? HPW : 1][HAS_DT ? kQ : 4];
  __shared__ __attribute__((aligned(256))) float csl[kCT ? HPW : 1][kCT ? kQ : 4];
  __shared__ __attribute__((aligned(256))) float wt[NW][kQ];
  __shared__ __attribute__((aligned(128))) float rsl[kRows ? NW : 1][32];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hh = wave >> 1, w = wave & 1;
  const int hl = lane >> 5, r = lane & 31;   // MFMA half and row / column
  const int g = lane >> 4, i = lane & 15;

  // ---- unit: (batch, segment, HPW heads of one group), heads fastest ----
  const int hb = p.nheads / HPW;
  const int u = xcd_remap(blockIdx.x, gridDim.x);
  const int h0 = (u % hb) * HPW, bseg = u / hb;
  const int seg = bseg % p.nseg, b = bseg / p.nseg;
  const int h = h0 + hh, grp = h0 / (p.nheads / p.ngroups);
  const int c0 = seg * p.seg_len, c1 = min(c0 + p.seg_len, p.nsteps), last = c1 - 1;

  // ---- copies: wave-uniform bases that step with c, and lane offsets ----
  // B and C rows: 256 bytes, piece k of row r at slot k ^ bsw(r) / k ^ (r & 15);
  // copy block d holds rows 4 d .. 4 d + 3.  (The transposing reads of B take 4
  // pieces of 8 consecutive rows at a time, the reads of C one piece of 16.)
  auto bsw = [](int row) __attribute__((always_inline)) { return (2 * row) & 14; };
  const int crow = lane >> 4, cslot = lane & 15;
  const int64_t bcg0 = ((int64_t)b * p.nsteps + c0) * p.ngroups + grp;
  const char* xg = (const char*)uni(reinterpret_cast<const T*>(p.x) + (int64_t)b * p.sxb + (int64_t)h * p.sxh + (int64_t)c0 * kQ * p.sxl);
  const char* bg = (const char*)uni(reinterpret_cast<const T*>(p.bm) + (int64_t)b * p.sbb + (int64_t)grp * p.sbg + (int64_t)c0 * kQ * p.sbl);
  const char* cg = kCT ? (const char*)uni(reinterpret_cast<const f16*>(p.ct) + bcg0 * kQ * kN)
                       : (const char*)uni(reinterpret_cast<const T*>(p.cm) + (int64_t)b * p.scb + (int64_t)grp * p.scg + (int64_t)c0 * kQ * p.scl);
  const char* cbg = (const char*)uni(reinterpret_cast<const f32x4*>(p.cb) + (bcg0 * kTiles + w) * 64);
  const char* ag = (const char*)uni(p.acs + (((int64_t)b * p.nheads + h) * p.nsteps + c0) * kQ);
  const char* dg = HAS_DT ? (const char*)uni(p.dt + (int64_t)b * p.sdb + (int64_t)h * p.sdh + (int64_t)c0 * kQ * p.sdl) : nullptr;
  const char* csg = kCT ? (const char*)uni(p.cscale + bcg0 * kQ) : nullptr;
  // bytes from one step to the next
  const int64_t xst = (int64_t)kQ * p.sxl * 2, bst = (int64_t)kQ * p.sbl * 2;
  const int64_t cst = kCT ? (int64_t)p.ngroups * kQ * kN * 2 : (int64_t)kQ * p.scl * 2;
  const int64_t cbst = (int64_t)p.ngroups * kTiles * 1024, dst = (int64_t)kQ * p.sdl * 4, csst = (int64_t)p.ngroups * kQ * 4;
  const uint32_t bs_o = uni(lds_offset(bs)) + DPW * wave * 1024, cl_o = uni(lds_offset(cl)) + DPW * wave * 1024;
  const uint32_t xs_o = uni(lds_offset(xs)) + (hh * 16 + w) * 1024;
  const uint32_t al_o = uni(lds_offset(al)) + hh * 256, dl_o = uni(lds_offset(dl)) + hh * 256;
  const uint32_t csl_o = uni(lds_offset(csl)) + hh * 256;
  // lane offsets: blocks d = DPW wave + m of B and C, blocks w + 2 m of x (B's
  // rows 8 further on lie in the same slots, so blocks m and m + 2 share one)
  uint32_t bv[2], cv[DPW];
#pragma unroll
  for (int m = 0; m < DPW; ++m) {
    const int row = 4 * (DPW * wave + m) + crow;
    if (m < 2) bv[m] = (uint32_t)(row * (int)p.sbl + 8 * (cslot ^ bsw(row & 15))) * 2;
    cv[m] = (uint32_t)(row * (kCT ? kN : (int)p.scl) + 8 * (cslot ^ (row & 15))) * 2;
  }
  const int64_t bst8 = (int64_t)8 * p.sbl * 2;
  const uint32_t xv = (uint32_t)((8 * w + (lane >> 3)) * (int)p.sxl + 8 * ((lane & 7) ^ (lane >> 3))) * 2;
  const int64_t xst16 = (int64_t)16 * p.sxl * 2;
  const uint32_t dv = HAS_DT ? (uint32_t)(lane * (int)p.sdl) * 4 : 0;

  // A copy stalls its wave while the copies before it, of all waves, pass the
  // CU's address path (16 cycles each), so they go out a few at a time between
  // the products: group C (C, C.B^T, Acs, dt, C scales) as parts 0 .. 3 of the
  // second phase, group B (B and x) as parts 0 .. 3 of the first.
  auto issue_c = [&](int part) __attribute__((always_inline)) {
#pragma unroll
    for (int m = 0; m < DPW; ++m)
      if (m % 2 == part) dma16_s(cg, cv[m], cl_o + m * 1024);
    if (part == 2) {
      if (w == 0) {
        dma4_s(ag, lane * 4, al_o);
      } else {
        if constexpr (HAS_DT) dma4_s(dg, dv, dl_o);
        if constexpr (kCT) dma4_s(csg, lane * 4, csl_o);
      }
    }
  };
  // x rows: 128 bytes, piece k of row s at slot k ^ (s & 7); this wave's blocks w, w + 2, .. of its head
  auto issue_b = [&](int part) __attribute__((always_inline)) {
#pragma unroll
    for (int m = 0; m < DPW; ++m)
      if ((2 * m) / DPW == part) dma16_s(bg + (m >> 1) * bst8, bv[m & 1], bs_o + m * 1024);
  };
  auto issue_x = [&](int part, int bf) __attribute__((always_inline)) {
#pragma unroll
    for (int m = 2 * part; m < 2 * part + 2; ++m) dma16_s(xg + m * xst16, xv, xs_o + (uint32_t)((bf * 8 + 2 * m) * 1024));
  };
  // C.B^T: this wave's five tiles go straight to registers, as buffer loads.  Never
  // as flat ones (what a load through a pointer that went through uni() becomes):
  // those may retire ahead of older accesses, and vm_wait<NY> counts on the order.
  f32x4 cbv[5];
  auto load_cb = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < 5; ++k) cbv[k] = load16_b(cbg, lane * 16 + k * 2048);
  };

#pragma unroll
  for (int part = 0; part < 3; ++part) issue_c(part);
  issue_x(0, 0);  // the first step's x; the rest of x, and B, come ahead of their use in the loop
  issue_x(1, 0);
  if (c0 < last) xg += xst;
  load_cb();

  // S^T tiles: st[nt][4 k + jj] = S[p = 32 w + r][n = 32 nt + 16 (k >> 1) + 8 hl + 4 (k & 1) + jj]
  f32x16 st[4];
  {
    const int64_t so = (32 * w + r) * kN + 8 * hl;
    auto load_s = [&](const float* sp, f32x16 (&v)[4]) __attribute__((always_inline)) {
#pragma unroll
      for (int nt = 0; nt < 4; ++nt)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const f32x4 q4 = *reinterpret_cast<const f32x4*>(sp + so + 32 * nt + 16 * (k >> 1) + 4 * (k & 1));
#pragma unroll
          for (int jj = 0; jj < 4; ++jj) v[nt][4 * k + jj] = q4[jj];
        }
    };
#pragma unroll
    for (int nt = 0; nt < 4; ++nt)
#pragma unroll
      for (int j = 0; j < 16; ++j) st[nt][j] = 0.f;
    const int64_t bh = (int64_t)b * p.nheads + h;
    if (p.linked) {
      load_s(p.seg_states + (((int64_t)b * p.nseg + seg) * p.nheads + h) * (kP * kN), st);
    } else {
      // the state entering the segment, from the end states of those before it
      if (p.init) load_s(p.init + bh * (kP * kN), st);
      for (int j = 0; j < seg; ++j) {
        f32x16 lo[4];
        load_s(p.seg_states + (((int64_t)b * p.nseg + j) * p.nheads + h) * (kP * kN), lo);
        const float dj = p.seg_decay[bh * p.nseg + j];
#pragma unroll
        for (int nt = 0; nt < 4; ++nt)
#pragma unroll
          for (int k = 0; k < 16; ++k) st[nt][k] = __builtin_fmaf(st[nt][k] * dj, dj, lo[nt][k]);
      }
    }
  }
  // the tiles above the diagonal inside W's blocks, (0, 1) and (2, 3), stay zero: block 2 (t >> 1) .. + s
  {
    vec4<T> z0;
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) z0[jj] = (T)0.f;
    store4<T>(&wl[hh][(w == 0 ? 1 : 5) * 512 + ((g & 1) * 32 + i) * 8 + 4 * (g >> 1)], z0);
  }
  const float dskip = EPI && p.dskip ? p.dskip[h] : 0.f;
  // y (and z): 16 rows of 64 bytes per instruction, 16-byte piece 2 (g & 1) + hl of the row in lane group g
  const int ypiece = 2 * (g & 1) + hl;
  // (a wave-uniform base and the lane's 32-bit offset: one register less than a
  // pointer per lane, and no vector arithmetic per step)
  T* yg = reinterpret_cast<T*>(p.y) + (int64_t)b * p.syb + (int64_t)h * p.syh + 32 * w;
  const uint32_t yv = (uint32_t)(i * (int)p.syl + 8 * ypiece) * 2;
  const T* zg = nullptr;
  uint32_t zo = 0;
  if constexpr (EPI) {
    zg = reinterpret_cast<const T*>(p.z) + (int64_t)b * p.szb + (int64_t)h * p.szh + 32 * w;
    zo = (uint32_t)(i * (int)p.szl + 8 * ypiece) * 2;
  }

  // operand addresses (elements)
  const int q = i & 3, trow = 4 * hl + (i >> 2);  // transposing reads: rows 16 kb + trow (+ 8)
  int boff[4];
#pragma unroll
  for (int nt = 0; nt < 4; ++nt)
    boff[nt] = trow * kN + 8 * ((4 * nt + 2 * (g & 1) + (q & 1)) ^ bsw(trow)) + 4 * (q >> 1);
  // C: piece 2 kb + hl, block kb by ^ 16 kb
  const int coff = r * kN + 8 * (hl ^ (r & 15));
  // W tiles: Acs (and dt) of the tile's tokens, and its place in W
  int asoff[3], aloff[2], woff[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    constexpr int dS[3] = {1, 2, -1}, dW[3] = {512 + 128, 2048, -512 + 128};
    asoff[k] = 16 * dS[k] * w + 4 * g;
    woff[k] = dW[k] * w + ((g & 1) * 32 + i) * 8 + 4 * (g >> 1);
    if (k < 2) aloff[k] = 16 * dS[k] * w + i;
  }
  const int xoff = trow * kP + 8 * ((4 * w + 2 * (g & 1) + (q >> 1)) ^ (trow & 7)) + 4 * (q & 1);

  dma_wait();
  __syncthreads();

  for (int c = c0; c < c1; ++c) {
    const int bf = (c - c0) & 1;
    const T* xb = xs[hh * 2 + bf];
    // the C.B^T loads end here, before this phase's copies queue up behind them
#pragma unroll
    for (int k = 0; k < 5; ++k) asm volatile("" : "+v"(cbv[k]));
    frag8<T> zv[EPI ? 4 : 1];
    // ---- first phase: weights, W, the off-diagonal product ----
    // (the workgroup in its second phase goes first where two share a CU: they
    // then finish together; 206 -> 198 us at 2 x 4 heads per CU)
    __builtin_amdgcn_s_setprio(0);
    const float* ab = al[hh];
    const float a_own = ab[lane];
    int co = coff;
    if constexpr (EPI) asm volatile("" : "+v"(co));  // (the eight addresses, kept over the steps, would not fit the registers)
    auto read_c = [&, coff = co](frag8<E> (&cf)[2], int kb) __attribute__((always_inline)) {
#pragma unroll
      for (int t = 0; t < 2; ++t) cf[t] = *reinterpret_cast<const frag8<E>*>(cl + (coff ^ (16 * kb)) + 32 * t * kN);
    };
    frag8<E> cf[2][2];
    read_c(cf[0], 0);
    // operands of this wave's five W tiles
    constexpr int kDI[5] = {0, 0, 1, 0, 2}, kTI[5] = {0, 0, 1, 0, 0};
    f32x4 as[2];
    float alv[2], el[2];
    auto read_tile = [&](int k) __attribute__((always_inline)) {
      as[k & 1] = *reinterpret_cast<const f32x4*>(ab + asoff[kDI[k]] + 16 * kS[k]);
      alv[k & 1] = ab[aloff[kTI[k]] + 16 * kT[k]];
    };
    read_tile(0);
#pragma unroll
    for (int t = 0; t < 2; ++t) el[t] = ab[32 * t + r];
    __builtin_amdgcn_sched_barrier(0);
    // S as f16 rows: the row's largest magnitude over the tiles, then over the two halves
    // (four independent chains, two values an instruction)
    float m = 0.f;
    if constexpr (kRows) {
      float mx[4];
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) mx[nt] = __builtin_elementwise_maximum(fabsf(st[nt][0]), fabsf(st[nt][1]));
#pragma unroll
      for (int j = 2; j < 16; j += 2)
#pragma unroll
        for (int nt = 0; nt < 4; ++nt)
          mx[nt] = __builtin_elementwise_maximum(__builtin_elementwise_maximum(fabsf(st[nt][j]), fabsf(st[nt][j + 1])), mx[nt]);
      m = __builtin_elementwise_maximum(__builtin_elementwise_maximum(mx[0], mx[1]), __builtin_elementwise_maximum(mx[2], mx[3]));
      const auto r32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(m), __float_as_uint(m), false, false);
      m = nn_max(__uint_as_float(r32[0]), __uint_as_float(r32[1]));
    }
    const float aq = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(a_own), 63));
    const float dec = __builtin_amdgcn_exp2f(aq * kLog2e);
    {
      float wv = __builtin_amdgcn_exp2f((aq - a_own) * kLog2e);
      if constexpr (HAS_DT) wv *= dl[hh][lane];
      wt[wave][lane] = wv;
    }
    f32x16 acc[2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int j = 0; j < 16; ++j) acc[t][j] = 0.f;
    float sc = 1.f, nz = -0.f;
    if constexpr (kRows) {
      const int e = m > 0.f ? min(max(__builtin_amdgcn_frexp_expf(m) - 15, -100), 100) : 0;
      sc = __builtin_ldexpf(1.f, -e);
      if (hl == 0) rsl[wave][r] = __builtin_ldexpf(1.f, e);
      // (scaled and rounded by one v_fma_mixlo / mixhi per value: the opaque -0
      // addend keeps the compiler from making it a product and a conversion)
      asm("" : "+v"(nz));
    }
    frag8<E> sf[2], sl[2];
    auto operand_s = [&](int kb) __attribute__((always_inline)) {
      const f32x16& v = st[kb >> 1];
      const int j0 = 8 * (kb & 1);
      if constexpr (kRows) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          sf[kb & 1][j] = (f16)__builtin_fmaf(v[j0 + j], sc, nz);
          if constexpr (HILO) sl[kb & 1][j] = (f16)__builtin_fmaf(v[j0 + j], sc, -(float)sf[kb & 1][j]);
        }
      } else {
        f32x4 a, b2;
#pragma unroll
        for (int j = 0; j < 4; ++j) a[j] = v[j0 + j], b2[j] = v[j0 + 4 + j];
        split_f32<T>(a, b2, sf[kb & 1], sl[kb & 1]);
      }
    };
    operand_s(0);
#pragma unroll
    for (int kb = 0; kb < 8; ++kb) {
      if (kb < 7) read_c(cf[(kb + 1) & 1], kb + 1);
      if (kb < 4) read_tile(kb + 1);
      // this step's B, the next step's x, then the gate's operands
      if (kb < 2) issue_b(kb);
      else if (kb < 4) issue_x(kb - 2, bf ^ 1);
      if (EPI && kb == 5) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int k = 0; k < 2; ++k) zv[EPI ? 2 * t + k : 0] = __builtin_bit_cast(frag8<T>, load16_g(zg + ((int64_t)c * kQ + 32 * t + 16 * k) * p.szl, zo));
      }
#pragma unroll
      for (int t = 0; t < 2; ++t) acc[t] = mma32(sf[kb & 1], cf[kb & 1][t], acc[t]);
      if constexpr (HILO) {
#pragma unroll
        for (int t = 0; t < 2; ++t) acc[t] = mma32(sl[kb & 1], cf[kb & 1][t], acc[t]);
      }
      if (kb < 7) operand_s(kb + 1);
      // the state's decay, its value entering the step being taken
#pragma unroll
      for (int j = 0; j < 8; ++j) st[kb >> 1][8 * (kb & 1) + j] *= dec;
      // between the products: this wave's five W tiles
      if (kb < 5) {
        const int s0 = kS[kb], t0 = kT[kb];
        const float al2 = alv[kb & 1] * kLog2e;
        f32x4 v;
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) v[jj] = cbv[kb][jj] * __builtin_amdgcn_exp2f(__builtin_fmaf(as[kb & 1][jj], -kLog2e, al2));
        if constexpr (HAS_DT) v *= *reinterpret_cast<const f32x4*>(&dl[hh][asoff[kDI[kb]] + 16 * s0]);
        if (kb < 2) {
          // the diagonal tiles; selection, not a product with the mask: exp2 above the diagonal may be inf
#pragma unroll
          for (int jj = 0; jj < 4; ++jj) v[jj] = 4 * g + jj <= i ? v[jj] : 0.f;
        }
        store4<T>(&wl[hh][woff[kDI[kb]] + ((t0 >> 1) * 2 + s0) * 512 + (t0 & 1) * 128], __builtin_convertvector(v, vec4<T>));
      }
    }
    // rows p carry their scale, columns l exp(Acs[l]) and C's scale
    float ev[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      ev[t] = __builtin_amdgcn_exp2f(el[t] * kLog2e);
      if constexpr (kCT) ev[t] *= csl[hh][32 * t + r];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      f32x4 rs = f32x4{1.f, 1.f, 1.f, 1.f};
      if constexpr (kRows) rs = *reinterpret_cast<const f32x4*>(&rsl[wave][8 * k + 4 * hl]);
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) acc[t][4 * k + jj] *= kRows ? rs[jj] * ev[t] : ev[t];
    }
    if (c < last) bg += bst;
    if (c + 1 < last) xg += xst;
    accesses_before_wait();
    vm_wait<NX>();
    __syncthreads();

    // ---- second phase: the diagonal product, the state update, y ----
    __builtin_amdgcn_s_setprio(1);
    // group C of the next step (the last step copies itself again)
    if (c < last) {
      cg += cst;
      cbg += cbst;
      ag += kQ * 4;
      if constexpr (HAS_DT) dg += dst;
      if constexpr (kCT) csg += csst;
    }
    auto read_b = [&](frag8<T> (&bq)[4], int kb) __attribute__((always_inline)) {
#pragma unroll
      for (int nt = 0; nt < 4; ++nt)
        bq[nt] = join<T>(lds_read_tr(bs + boff[nt] + 16 * kb * kN), lds_read_tr(bs + boff[nt] + (16 * kb + 8) * kN));
    };
    auto read_x = [&](int kb) __attribute__((always_inline)) {
      return join<T>(lds_read_tr(xb + xoff + 16 * kb * kP), lds_read_tr(xb + xoff + (16 * kb + 8) * kP));
    };
    auto read_w = [&](int k) __attribute__((always_inline)) {
      return *reinterpret_cast<const frag8<T>*>(&wl[hh][k * 512 + lane * 8]);
    };
    auto read_wt = [&](int k) __attribute__((always_inline)) { return *reinterpret_cast<const f32x4*>(&wt[wave][8 * k + 4 * hl]); };
    frag8<T> xf[2], xh[2], xl[2], bq[2][4];
    xf[0] = read_x(0);
    f32x4 w0 = read_wt(0), w1 = read_wt(1);
    read_b(bq[0], 0);
    xf[1] = read_x(1);
    split_weighted<T, true>(xf[0], w0, w1, xh[0], xl[0]);
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      // this block's products, the next block's operands and weighting between them
      const frag8<T> x0 = xf[kb & 1], wb = read_w(2 + kb);
      frag8<T> wa;
      if (kb < 2) wa = read_w(kb);
      if (kb < 3) {
        w0 = read_wt(2 * kb + 2);
        w1 = read_wt(2 * kb + 3);
        read_b(bq[(kb + 1) & 1], kb + 1);
        issue_c(kb);
      } else if (!EPI) {
        load_cb();
      }
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) st[nt] = mma32(bq[kb & 1][nt], xh[kb & 1], st[nt]);
      if (kb < 2) acc[0] = mma32(x0, wa, acc[0]);
      acc[1] = mma32(x0, wb, acc[1]);
      if (kb < 2) xf[kb & 1] = read_x(kb + 2);
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) st[nt] = mma32(bq[kb & 1][nt], xl[kb & 1], st[nt]);
      if (kb < 3) {
        split_weighted<T, true>(xf[(kb + 1) & 1], w0, w1, xh[(kb + 1) & 1], xl[(kb + 1) & 1]);
#pragma unroll
        for (int q2 = 0; q2 < 8; ++q2) {
          __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x2, std::is_same<T, f16>::value ? 4 : 5, 0);
        }
      }
    }
    if constexpr (EPI) load_cb();
    // y: rows p 8 k + 4 hl .. + 3 per lane.  The halves swap, so that a lane
    // holds 8 consecutive p, 8 (k + hl) .., of token 32 t + r; then tokens
    // r < 16 and r >= 16 swap, so that one store writes 64 bytes of 16 rows
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
      typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
      u32x4 zz[2], o[2];
      if constexpr (EPI) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const u32x4 za = __builtin_bit_cast(u32x4, zv[2 * t]), zb = __builtin_bit_cast(u32x4, zv[2 * t + 1]);
          const auto q2 = __builtin_amdgcn_permlane16_swap(za[j], zb[j], false, false);
          zz[0][j] = q2[0];
          zz[1][j] = q2[1];
        }
      }
#pragma unroll
      for (int k = 0; k < 4; k += 2) {
        f32x4 v[2];
#pragma unroll
        for (int e2 = 0; e2 < 2; ++e2)
#pragma unroll
          for (int jj = 0; jj < 4; ++jj) v[e2][jj] = acc[t][4 * (k + e2) + jj];
        if constexpr (EPI) {
          const auto z0 = __builtin_amdgcn_permlane32_swap(zz[k / 2][0], zz[k / 2][2], false, false);
          const auto z1 = __builtin_amdgcn_permlane32_swap(zz[k / 2][1], zz[k / 2][3], false, false);
#pragma unroll
          for (int e2 = 0; e2 < 2; ++e2) {
            const vec4<T> z4 = __builtin_bit_cast(vec4<T>, (u32x2{z0[e2], z1[e2]}));
            const vec4<T> x4 = load4<T>(xb + (32 * t + r) * kP + 8 * ((4 * w + k + e2) ^ (r & 7)) + 4 * hl);
#pragma unroll
            for (int jj = 0; jj < 4; ++jj) {
              const float zf = to_f32<T>(z4[jj]);
              v[e2][jj] = __builtin_fmaf(dskip, to_f32<T>(x4[jj]), v[e2][jj]) * zf *
                          __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-kLog2e * zf));
            }
          }
        }
        const u32x2 a = __builtin_bit_cast(u32x2, __builtin_convertvector(v[0], vec4<T>));
        const u32x2 d = __builtin_bit_cast(u32x2, __builtin_convertvector(v[1], vec4<T>));
        const auto w0 = __builtin_amdgcn_permlane32_swap(a[0], d[0], false, false);
        const auto w1 = __builtin_amdgcn_permlane32_swap(a[1], d[1], false, false);
        o[k / 2] = u32x4{w0[0], w1[0], w0[1], w1[1]};
      }
      u32x4 oa, ob;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const auto q2 = __builtin_amdgcn_permlane16_swap(o[0][j], o[1][j], false, false);
        oa[j] = q2[0];
        ob[j] = q2[1];
      }
      T* yr = yg + ((int64_t)c * kQ + 32 * t) * p.syl;
      store16_g(yr, yv, __builtin_bit_cast(f32x4, oa));
      store16_g(yr + 16 * p.syl, yv, __builtin_bit_cast(f32x4, ob));
    }
    accesses_before_wait();
    vm_wait<NY>();
    __syncthreads();
  }
  // the copies past the last step land before this workgroup's LDS is given away
  dma_wait();
  if (p.final_state && c1 == p.nsteps) {
    float* fp = p.final_state + ((int64_t)b * p.nheads + h) * (kP * kN) + (32 * w + r) * kN + 8 * hl;
#pragma unroll
    for (int nt = 0; nt < 4; ++nt)
#pragma unroll
      for (int k = 0; k < 4; ++k)
        *reinterpret_cast<f32x4*>(fp + 32 * nt + 16 * (k >> 1) + 4 * (k & 1)) = f32x4{st[nt][4 * k], st[nt][4 * k + 1], st[nt][4 * k + 2], st[nt][4 * k + 3]};
  }
}

// The state at the end of every segment but the last, from a zero state, and
// the square root of the segment's decay (of many tokens: where their log-decays
// are positive the decay itself may lie beyond f32, and a state that is still
// zero has to stay so): the scan's state update alone, for chains too few to fill the GPU as one segment each.  A step here is
// shorter than the latency of HBM, so B and x are copied two steps ahead, into
// a ring of three buffers; one barrier per step.
template <typename T, int HPW, bool HAS_DT>
__global__ __launch_bounds__(128 * HPW, HPW == 4 ? 2 : 1) void chain_state_kernel(ChainScanArgs p) {
  constexpr int NW = 2 * HPW, DPW = 16 / NW;
  constexpr int kStages = 3;
  constexpr int kPer = DPW + 4 + 1 + (HAS_DT ? 1 : 0);  // copies per wave and step
  __shared__ __attribute__((aligned(1024))) T bs[kStages][kQ * kN];
  __shared__ __attribute__((aligned(1024))) T xs[kStages][HPW][kQ * kP];
  __shared__ __attribute__((aligned(256))) float al[kStages][NW][kQ];
  __shared__ __attribute__((aligned(256))) float dl[kStages][HAS_DT ? NW : 1][HAS_DT ? kQ : 4];
  __shared__ __attribute__((aligned(256))) float wt[NW][kQ];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hh = wave >> 1, w = wave & 1;
  const int hl = lane >> 5, r = lane & 31, g = lane >> 4, i = lane & 15;

  const int hb = p.nheads / HPW, ns = p.nseg - 1;
  const int u = xcd_remap(blockIdx.x, gridDim.x);
  const int h0 = (u % hb) * HPW, bseg = u / hb;
  const int seg = bseg % ns, b = bseg / ns;
  const int h = h0 + hh, grp = h0 / (p.nheads / p.ngroups);
  const int c0 = seg * p.seg_len, c1 = c0 + p.seg_len, last = c1 - 1;

  auto bsw = [](int row) __attribute__((always_inline)) { return (2 * row) & 14; };
  const int crow = lane >> 4, cslot = lane & 15;
  const char* xg = (const char*)uni(reinterpret_cast<const T*>(p.x) + (int64_t)b * p.sxb + (int64_t)h * p.sxh + (int64_t)c0 * kQ * p.sxl);
  const char* bg = (const char*)uni(reinterpret_cast<const T*>(p.bm) + (int64_t)b * p.sbb + (int64_t)grp * p.sbg + (int64_t)c0 * kQ * p.sbl);
  const char* ag = (const char*)uni(p.acs + (((int64_t)b * p.nheads + h) * p.nsteps + c0) * kQ);
  const char* dg = HAS_DT ? (const char*)uni(p.dt + (int64_t)b * p.sdb + (int64_t)h * p.sdh + (int64_t)c0 * kQ * p.sdl) : nullptr;
  const int64_t xst = (int64_t)kQ * p.sxl * 2, bst = (int64_t)kQ * p.sbl * 2, dst = (int64_t)kQ * p.sdl * 4;
  const uint32_t bs_o = uni(lds_offset(bs)) + DPW * wave * 1024;
  const uint32_t xs_o = uni(lds_offset(xs)) + (hh * 8 + w) * 1024;
  const uint32_t al_o = uni(lds_offset(al)) + wave * 256, dl_o = uni(lds_offset(dl)) + wave * 256;
  uint32_t bv[DPW], xv[4];
#pragma unroll
  for (int m = 0; m < DPW; ++m) {
    const int row = 4 * (DPW * wave + m) + crow;
    bv[m] = (uint32_t)(row * (int)p.sbl + 8 * (cslot ^ bsw(row & 15))) * 2;
  }
#pragma unroll
  for (int m = 0; m < 4; ++m)
    xv[m] = (uint32_t)((8 * (w + 2 * m) + (lane >> 3)) * (int)p.sxl + 8 * ((lane & 7) ^ (lane >> 3))) * 2;
  const uint32_t dv = HAS_DT ? (uint32_t)(lane * (int)p.sdl) * 4 : 0;

  // a quarter of a step's copies into buffer bf
  auto issue = [&](int part, int bf) __attribute__((always_inline)) {
#pragma unroll
    for (int m = 0; m < DPW; ++m)
      if (m % 4 == part) dma16_s(bg, bv[m], bs_o + (uint32_t)(bf * 16384 + m * 1024));
    dma16_s(xg, xv[part], xs_o + (uint32_t)((bf * HPW * 8 + 2 * part) * 1024));
    if (part == 0) {
      dma4_s(ag, lane * 4, al_o + (uint32_t)(bf * NW * 256));
      if constexpr (HAS_DT) dma4_s(dg, dv, dl_o + (uint32_t)(bf * NW * 256));
    }
  };
  auto advance = [&]() __attribute__((always_inline)) {
    xg += xst;
    bg += bst;
    ag += kQ * 4;
    if constexpr (HAS_DT) dg += dst;
  };
#pragma unroll
  for (int k = 0; k < kStages - 1; ++k) {
#pragma unroll
    for (int part = 0; part < 4; ++part) issue(part, k);
    if (c0 + k < last) advance();
  }

  f32x16 st[4];
#pragma unroll
  for (int nt = 0; nt < 4; ++nt)
#pragma unroll
    for (int j = 0; j < 16; ++j) st[nt][j] = 0.f;
  float atot = 0.f;
  int bf = 0;
  const int q = i & 3, trow = 4 * hl + (i >> 2);
  int boff[4];
#pragma unroll
  for (int nt = 0; nt < 4; ++nt)
    boff[nt] = trow * kN + 8 * ((4 * nt + 2 * (g & 1) + (q & 1)) ^ bsw(trow)) + 4 * (q >> 1);
  const int xoff = trow * kP + 8 * ((4 * w + 2 * (g & 1) + (q >> 1)) ^ (trow & 7)) + 4 * (q & 1);

  for (int c = c0; c < c1; ++c) {
    vm_wait<(kStages - 2) * kPer>();  // this step's copies
    __syncthreads();
    const int nbf = bf == 0 ? kStages - 1 : bf - 1;  // the buffer of the step before
    const T* xb = xs[bf][hh];
    const T* bb = bs[bf];
    auto read_b = [&](frag8<T> (&bq)[4], int kb) __attribute__((always_inline)) {
#pragma unroll
      for (int nt = 0; nt < 4; ++nt)
        bq[nt] = join<T>(lds_read_tr(bb + boff[nt] + 16 * kb * kN), lds_read_tr(bb + boff[nt] + (16 * kb + 8) * kN));
    };
    auto read_x = [&](int kb) __attribute__((always_inline)) {
      return join<T>(lds_read_tr(xb + xoff + 16 * kb * kP), lds_read_tr(xb + xoff + (16 * kb + 8) * kP));
    };
    auto read_wt = [&](int k) __attribute__((always_inline)) { return *reinterpret_cast<const f32x4*>(&wt[wave][8 * k + 4 * hl]); };
    const float a_own = al[bf][wave][lane];
    frag8<T> xf[2], xh[2], xl[2], bq[2][4];
    xf[0] = read_x(0);
    read_b(bq[0], 0);
    xf[1] = read_x(1);
    const float aq = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(a_own), 63));
    const float dec = __builtin_amdgcn_exp2f(aq * kLog2e);
    float wv = __builtin_amdgcn_exp2f((aq - a_own) * kLog2e);
    if constexpr (HAS_DT) wv *= dl[bf][wave][lane];
    wt[wave][lane] = wv;
    atot += aq;
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) st[nt] *= dec;
    f32x4 w0 = read_wt(0), w1 = read_wt(1);
    split_weighted<T, true>(xf[0], w0, w1, xh[0], xl[0]);
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      if (kb < 3) {
        w0 = read_wt(2 * kb + 2);
        w1 = read_wt(2 * kb + 3);
        read_b(bq[(kb + 1) & 1], kb + 1);
      }
      if (kb < 2) xf[kb & 1] = read_x(kb + 2);
      issue(kb, nbf);  // two steps ahead (the last steps copy the last one again)
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) st[nt] = mma32(bq[kb & 1][nt], xh[kb & 1], st[nt]);
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) st[nt] = mma32(bq[kb & 1][nt], xl[kb & 1], st[nt]);
      if (kb < 3) {
        split_weighted<T, true>(xf[(kb + 1) & 1], w0, w1, xh[(kb + 1) & 1], xl[(kb + 1) & 1]);
#pragma unroll
        for (int q2 = 0; q2 < 8; ++q2) {
          __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x2, std::is_same<T, f16>::value ? 4 : 5, 0);
        }
      }
    }
    if (c + kStages - 1 < last) advance();
    bf = bf == kStages - 1 ? 0 : bf + 1;
  }
  dma_wait();
  float* fp = p.seg_states + (((int64_t)b * p.nseg + seg) * p.nheads + h) * (kP * kN) + (32 * w + r) * kN + 8 * hl;
#pragma unroll
  for (int nt = 0; nt < 4; ++nt)
#pragma unroll
    for (int k = 0; k < 4; ++k)
      *reinterpret_cast<f32x4*>(fp + 32 * nt + 16 * (k >> 1) + 4 * (k & 1)) = f32x4{st[nt][4 * k], st[nt][4 * k + 1], st[nt][4 * k + 2], st[nt][4 * k + 3]};
  if (w == 0 && lane == 0) p.seg_decay[((int64_t)b * p.nheads + h) * p.nseg + seg] = __builtin_amdgcn_exp2f(atot * (0.5f * kLog2e));
}

template <typename T, int HPW>
hipError_t launch_state_t(const ChainScanArgs& a, hipStream_t stream) {
  const int64_t grid = (int64_t)a.batch * (a.nseg - 1) * (a.nheads / HPW);
  if (grid > INT32_MAX) return hipErrorInvalidValue;
  auto kern = a.dt ? chain_state_kernel<T, HPW, true> : chain_state_kernel<T, HPW, false>;
  kern<<<dim3((unsigned)grid), dim3(128 * HPW), 0, stream>>>(a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || !a.linked) return e;
  // the state entering each segment
  StatePassingArgs sp;
  sp.states = a.seg_states;
  sp.decay = a.seg_decay;
  sp.root_decay = true;
  sp.init = a.init;
  sp.final_state = nullptr;
  sp.batch = a.batch;
  sp.nchunks = a.nseg;
  sp.nheads = a.nheads;
  sp.headdim = kP;
  sp.dstate = kN;
  return launch_state_passing(sp, SSD_DTYPE_F32, stream);
}

template <typename T, int HPW, bool HAS_DT, bool EPI, bool HILO>
hipError_t launch_scan_t(const ChainScanArgs& a, hipStream_t stream) {
  const int64_t grid = (int64_t)a.batch * a.nseg * (a.nheads / HPW);
  if (grid > INT32_MAX) return hipErrorInvalidValue;
  auto kern = chain_scan_kernel<T, HPW, HAS_DT, EPI, HILO>;
  kern<<<dim3((unsigned)grid), dim3(128 * HPW), 0, stream>>>(a);
  return hipGetLastError();
}

template <typename T, bool HILO>
hipError_t launch_t(const ChainScanArgs& a, hipStream_t stream) {
  const int hpg = a.nheads / a.ngroups;
  if (hpg % 2 != 0) return hipErrorInvalidValue;
  hipError_t e = hipSuccess;
  if (a.nseg > 1) e = hpg % 4 == 0 ? launch_state_t<T, 4>(a, stream) : launch_state_t<T, 2>(a, stream);
  if (e != hipSuccess) return e;
  if (!a.z) return a.dt ? launch_scan_t<T, 2, true, false, HILO>(a, stream) : launch_scan_t<T, 2, false, false, HILO>(a, stream);
  if (!a.dt) return hipErrorInvalidValue;  // (the gate belongs to the layer, whose dt is always there)
  return a.wide ? launch_scan_t<T, 4, true, true, HILO>(a, stream) : launch_scan_t<T, 2, true, true, HILO>(a, stream);
}

}  // namespace

size_t chain_scan_cb_bytes(int64_t steps) { return (size_t)steps * kTiles * 64 * sizeof(f32x4); }
size_t chain_scan_ct_bytes(int64_t steps) { return (size_t)steps * kQ * kN * 2; }
size_t chain_scan_cscale_bytes(int64_t steps) { return (size_t)steps * kQ * sizeof(float); }

// The plan with the least expected time, and whether that is clearly (10%)
// below the stage kernels'.  Times in us, from runs on 256 CUs: a step of the
// scan takes `one` with at most one workgroup (two heads) on a CU, `two` with
// two; a step of the state kernel 2.05 with up to one workgroup (four heads, or
// two of a group that four does not divide) per CU.  Stage kernels: 27 + 9.4 per
// 1000 (chain, 64 token step) pairs, or where 256 does not divide the sequence
// 52 + 22 per 1000; with the layer's gate 35 + 13.1 and 40 + 38.
// Measured with forced segment counts on 18 shapes (us, stage kernels / chosen
// count / fastest count): 4 x 4096, 80 heads 209 / 178 / 174; 3 x 3072, 80 heads
// 117 / 104 / 104; 16 x 512, 64 heads 89 / 53 / 53; 1 x 2880, 80 heads 125 / 63 /
// 63; 3 x 2368, 24 heads in groups of six 96 / 58 / 58; span 2 x 1216, 128 heads
// 243 / 91 / 91, 1 x 2048 98 / 95 / 89.  Where the model is off: it knows no cost
// per workgroup, so that 1 x 65536, 80 heads runs in 38 segments (735 us) where 12
// take 711; and it is up to 18% high for few workgroups, so that 1 x 16384, 80
// heads stays on the stage kernels (228; 190 in 12 segments).
ChainScanPlan chain_scan_plan(int64_t batch, int64_t steps, int64_t nheads, int64_t ngroups, bool epi) {
  ChainScanPlan best{0, 0, false};
  const int64_t hpg = nheads / ngroups, chains = batch * nheads;
  if (hpg % 2 != 0) return best;
  const int64_t cus = device_cu_count() > 0 ? device_cu_count() : 256;
  // Under ten steps per CU the stage kernels stay although the walk is faster (2 x
  // 2112 tokens of 24 heads: 86 us, 44 as a walk): calls of that size are compared
  // bit for bit with the stage kernels' own entry points.
  const int64_t pairs = chains * steps;
  if (pairs < 10 * cus) return best;
  const float one = epi ? 3.7f : 3.f, two = epi ? 6.7f : 5.3f;
  float best_us = 0.f;
  for (int64_t want = 1; want <= 64 && want <= steps; ++want) {
    const int64_t len = (steps + want - 1) / want, nseg = (steps + len - 1) / len;
    if (nseg != want) continue;
    const int64_t units = chains / 2 * nseg, rest = units % (2 * cus);
    float t = (float)len * ((float)(units / (2 * cus)) * two + (rest > cus ? two : rest ? one : 0.f));
    if (nseg > 1) {
      const int64_t su = chains / (hpg % 4 == 0 ? 4 : 2) * (nseg - 1);
      t += 5.f + (float)len * 2.05f * (float)((su + cus - 1) / cus);
      t += nseg > kFoldSegs ? 8.f + 0.006f * (float)(chains * nseg) : 3.f * (float)nseg;
    }
    if (best.nseg == 0 || t < best_us) {
      best = ChainScanPlan{(int)nseg, (int)len, false};
      best_us = t;
    }
  }
  const float kpairs = 1e-3f * (float)pairs;
  const float prep = 10.f + 0.37f * kpairs + 0.008f * (float)(batch * steps * ngroups);
  const bool whole = steps % 4 == 0;
  const float stages = epi ? (whole ? 35.f + 13.1f * kpairs : 40.f + 38.f * kpairs)
                           : (whole ? 27.f + 9.4f * kpairs : 52.f + 22.f * kpairs);
  if (prep + best_us > 0.9f * stages) return ChainScanPlan{0, 0, false};
  // the gated variant with four heads per workgroup where that fills every CU
  // alike: B, C and C.B^T are copied once per four heads (batch 8 x 2048 of 128
  // heads: 368 against 380 us; 2 x 1216 in its four segments 91 against 92; where
  // it leaves CUs idle, 4 x 2048, 256 against 205)
  const int64_t u4 = chains / 4 * best.nseg;
  best.wide = epi && hpg % 4 == 0 && u4 * 8 >= ((u4 + cus - 1) / cus) * cus * 7;
  return best;
}

hipError_t launch_chain_prep(const ChainScanArgs& a, const CumsumArgs& ca, int dtype, hipStream_t stream) {
  if (ca.chunk != kQ || (ca.dt_raw && ca.raw_dtype != dtype)) return hipErrorInvalidValue;
  if (dtype == SSD_DTYPE_BF16)
    return ca.dt_raw ? launch_chain_prep_t<bf16, 4, bf16, true>(a, ca, stream) : launch_chain_prep_t<bf16, 4, float, false>(a, ca, stream);
  if (dtype == SSD_DTYPE_F16)
    return ca.dt_raw ? launch_chain_prep_t<f16, 4, f16, true>(a, ca, stream) : launch_chain_prep_t<f16, 4, float, false>(a, ca, stream);
  return hipErrorInvalidValue;
}

hipError_t launch_chain_scan(const ChainScanArgs& a, int dtype, hipStream_t stream) {
  if (dtype == SSD_DTYPE_BF16) return a.hilo ? launch_t<bf16, true>(a, stream) : launch_t<bf16, false>(a, stream);
  if (dtype == SSD_DTYPE_F16) return a.hilo ? launch_t<f16, true>(a, stream) : launch_t<f16, false>(a, stream);
  return hipErrorInvalidValue;
}

}  // namespace ssd
