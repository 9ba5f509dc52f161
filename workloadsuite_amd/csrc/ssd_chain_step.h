// Building blocks of the chain walks (ssd_chain_scan.hip for 16-bit inputs,
// ssd_chain_scan_f32.hip): copies, the causal tiles of C.B^T and the launch
// that forms them together with K1's 64-token cumsums.
#pragma once

#include "ssd_cumsum_body.h"
#include "ssd_device.h"
#include "ssd_launch.h"

namespace ssd {

constexpr int kStep = 64;    // tokens per step
constexpr int kTiles = 10;   // causal 16 x 16 tiles of C.B^T

// Global -> LDS copies of 16 (4) bytes per lane from the wave-uniform base s
// plus the lane's byte offset v: no vector address arithmetic per copy.  M0
// holds the LDS destination; nothing else in these kernels uses it.
__device__ __forceinline__ void dma16_s(const void* s, uint32_t v, uint32_t lds_off) {
  asm volatile(
      "s_mov_b32 m0, %2\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %0, %1"
      :
      : "v"(v), "s"(s), "s"(lds_off)
      : "memory");
}
__device__ __forceinline__ void dma4_s(const void* s, uint32_t v, uint32_t lds_off) {
  asm volatile(
      "s_mov_b32 m0, %2\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dword %0, %1"
      :
      : "v"(v), "s"(s), "s"(lds_off)
      : "memory");
}
__device__ __forceinline__ uint32_t uni(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }
template <typename U> __device__ __forceinline__ const U* uni(const U* q) {
  const uint64_t v = (uint64_t)q;
  return (const U*)(((uint64_t)uni((uint32_t)(v >> 32)) << 32) | uni((uint32_t)v));
}
// Buffer accesses from a wave-uniform base on: the lane's byte offset in one
// register, a row's in a scalar one (and no flat access, as through a pointer
// that went through uni(), which would also hold up the LDS counter).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* base) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, -1, 0x00020000);
}
__device__ __forceinline__ f32x4 load16_b(const void* base, uint32_t v) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc(base), v, 0, 0));
}
// The same as a global access (a generic pointer would make it a flat one, which
// a counted wait on other accesses cannot hold apart from them).
__device__ __forceinline__ f32x4 load16_g(const void* base, uint32_t v) {
  typedef const f32x4 __attribute__((address_space(1))) * gptr;
  return *(gptr)((const char __attribute__((address_space(1)))*)base + v);
}
__device__ __forceinline__ void store16_g(void* base, uint32_t v, f32x4 d) {
  typedef f32x4 __attribute__((address_space(1))) * gptr;
  *(gptr)((char __attribute__((address_space(1)))*)base + v) = d;
}

// In front of a counted wait (vm_wait) that relies on loads the compiler issued
// before it: without a store or an access it knows nothing of in between, they may
// end up behind the wait and its barrier, next to their use.
__device__ __forceinline__ void accesses_before_wait() { asm volatile("" ::: "memory"); }

// The causal tiles (row tile t of l, column tile s of s, s <= t) in pairs 2 m +
// w, one for each wave of a head: (t, s) = (kT[m] + kDT[m] w, kS[m] + kDS[m] w).
// Pairs 0 and 1 are the diagonal ones.
constexpr int kT[5] = {0, 2, 1, 2, 2}, kDT[5] = {1, 1, 2, 1, 1};
constexpr int kS[5] = {0, 2, 0, 0, 1}, kDS[5] = {1, 1, 2, 1, -1};

namespace {

// C.B^T tiles and, for bf16, the f16 C rows of (batch, step, group) bcg; 4 waves, wave t = row tile t.
template <typename T, int NK>
__device__ __forceinline__ void chain_prep_body(const ChainScanArgs& p, int bcg, int tid) {
  const int lane = tid & 63, t = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, i = lane & 15;
  const int grp = bcg % p.ngroups, bc = bcg / p.ngroups;
  const int c = bc % p.nsteps, b = bc / p.nsteps;
  const T* bg = reinterpret_cast<const T*>(p.bm) + (int64_t)b * p.sbb + (int64_t)c * kStep * p.sbl + (int64_t)grp * p.sbg;
  const T* cg = reinterpret_cast<const T*>(p.cm) + (int64_t)b * p.scb + (int64_t)c * kStep * p.scl + (int64_t)grp * p.scg;
  frag8<T> cf[NK];
#pragma unroll
  for (int kc = 0; kc < NK; ++kc) cf[kc] = load8<T>(cg + (int64_t)(16 * t + i) * p.scl + 32 * kc + 8 * g);
  f32x4* cb = reinterpret_cast<f32x4*>(p.cb) + (int64_t)bcg * kTiles * 64 + lane;
#pragma unroll
  for (int k = 0; k < kTiles; ++k) {
    const int m = k >> 1, wk = k & 1, s = kS[m] + kDS[m] * wk;
    if (kT[m] + kDT[m] * wk != t) continue;  // wave-uniform
    f32x4 d = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kc = 0; kc < NK; ++kc) d = mma(load8<T>(bg + (int64_t)(16 * s + i) * p.sbl + 32 * kc + 8 * g), cf[kc], d);
    cb[k * 64] = d;
  }
  if constexpr (std::is_same<T, bf16>::value) {
    if (!p.ct) return;  // (S as a hi + lo pair: the walk takes C as it lies)
    // each row as f16 times 2^-e, its largest element in [2^14, 2^15) (bf16
    // values then convert exactly down to 2^-31 of it)
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    uint32_t mb = 0;
#pragma unroll
    for (int kc = 0; kc < NK; ++kc) {
      const auto w = __builtin_bit_cast(u32x4, cf[kc]);
#pragma unroll
      for (int j = 0; j < 4; ++j) mb = max(mb, max(w[j] & 0x7fffu, (w[j] >> 16) & 0x7fffu));
    }
    float m = __uint_as_float(min(mb, 0x7f80u) << 16);  // a NaN counts as inf, as in every lane
    m = nn_max(m, __shfl_xor(m, 16));
    m = nn_max(m, __shfl_xor(m, 32));
    const int e = m > 0.f ? min(max(__builtin_amdgcn_frexp_expf(m) - 15, -100), 100) : 0;
    f16* row = reinterpret_cast<f16*>(p.ct) + ((int64_t)bcg * kStep + 16 * t + i) * (32 * NK);
#pragma unroll
    for (int kc = 0; kc < NK; ++kc) {
      f16x8 hv;
#pragma unroll
      for (int j = 0; j < 8; ++j) hv[j] = (f16)__builtin_ldexpf(to_f32<T>(cf[kc][j]), -e);
      store8<f16>(row + 32 * kc + 8 * g, hv);
    }
    if (g == 0) p.cscale[(int64_t)bcg * kStep + 16 * t + i] = __builtin_ldexpf(1.f, e);
  }
}

// K1's blocks (64-token cumsums, 256 threads each) and the prep blocks in one launch.
template <typename T, int NK, typename R, bool RAW>
__global__ __launch_bounds__(256) void chain_prep_kernel(ChainScanArgs p, CumsumArgs ca, int nk1) {
  __shared__ CumsumTile<kStep> tile;
  if ((int)blockIdx.x >= nk1) {
    chain_prep_body<T, NK>(p, (int)blockIdx.x - nk1, threadIdx.x);
    return;
  }
  cumsum_load<kStep, R, RAW>(ca, blockIdx.x, threadIdx.x, tile);
  __syncthreads();
  cumsum_scan<kStep>(ca, blockIdx.x, threadIdx.x / kWave, threadIdx.x % kWave, tile);
}

template <typename T, int NK, typename R, bool RAW>
hipError_t launch_chain_prep_t(const ChainScanArgs& a, const CumsumArgs& ca, hipStream_t stream) {
  const int64_t nk1 = cumsum_blocks(ca), nprep = (int64_t)a.batch * a.nsteps * a.ngroups;
  if (nk1 + nprep > INT32_MAX) return hipErrorInvalidValue;
  chain_prep_kernel<T, NK, R, RAW><<<dim3((unsigned)(nk1 + nprep)), 256, 0, stream>>>(a, ca, (int)nk1);
  return hipGetLastError();
}

}  // namespace

}  // namespace ssd
