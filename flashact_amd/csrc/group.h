// Building blocks of the kernels that run small batches on groups of XCDs (pi05_group.hip, ma2_group.hip):
// per-wave epoch flags inside an XCD and across the XCDs of a group, the LDS ring through which two loader
// waves stream a CU's weights (and K/V), and the token-tile GEMM that reads it.
//
// A workgroup is one CU: waves 0-3 compute, waves 4-5 load. Every compute wave is an independent agent with
// its own flags; no workgroup barrier runs after the prologue. Workgroup b runs on XCD b % 8 as rank b / 8
// (checked by each kernel against HW_REG_XCC_ID).
//
// The kernel's configuration K provides G (XCDs per group) and L_CTL (byte offset of the LDS control words:
// u32 ready[2], consumed[4], abort, then the kernel's own).
#pragma once
#include "fa_device.h"

namespace fa {
namespace grp {

constexpr int NX = 8, NR = 32, NWG = 256;
constexpr int NCW = 4, NLW = 2, NTH = 64 * (NCW + NLW);  // compute waves, loader waves
constexpr int PAGE = 16384;                             // ring page bytes: 16 fragments of 16 rows x 32 k
constexpr int MAXF = 2;                                 // pages in flight per loader wave (1: 3-9 % slower)
constexpr uint32_t OOB = 0x80000000u;                   // buffer offset past every resource
constexpr uint32_t OFF_CTRL = 0, OFF_XFLAG = 1024;
constexpr uint32_t OFF_DONE = 24;  // u32: groups of this launch that have finished
static_assert(OFF_XFLAG + NX * NR * NCW * 8 <= kWsCounters, "flags stay below the fixup counters");
static_assert(kWsGroupFlags + NX * NR * NCW * 8 <= kWsDataBase, "group flags stay below the data");

extern __shared__ __attribute__((aligned(16))) unsigned char fg_lds[];

struct Ctx {
  int x, j, grp, r, wave, lane, lr, lq;  // XCD, its index in the group, group, rank
  int ns;                 // samples of this group
  rsrc_t ws;
  unsigned char* wsp;
  uint32_t xb, part;      // byte offsets of this XCD's block and this group's partial sums
  uint32_t lds_addr;
  unsigned* err;
  uint64_t e, eg;         // epochs of this wave's latest XCD / group signal
};

// Recompute lane-derived addresses per stage instead of keeping them live across the layer.
__device__ __forceinline__ void launder(Ctx& c) { asm volatile("" : "+v"(c.lane), "+v"(c.lr), "+v"(c.lq)); }

template <class K>
__device__ __forceinline__ unsigned ctl_ld(int i) {
  return __hip_atomic_load(reinterpret_cast<unsigned*>(fg_lds + K::L_CTL) + i, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_WORKGROUP);
}
template <class K>
__device__ __forceinline__ void ctl_st(int i, unsigned v) {
  __hip_atomic_store(reinterpret_cast<unsigned*>(fg_lds + K::L_CTL) + i, v, __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ bool aborted(const Ctx& c) {
  return __hip_atomic_load(c.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & kErrSpin;
}

// ---------------------------------------------------------------- synchronisation
// Signal: the wave drains its stores and publishes its epoch to its own flag (plain store, read by its
// XCD). Waits are capped and set the sticky error bit, which makes every later wait return at once.
__device__ __forceinline__ void xcd_signal(Ctx& c) {
  __builtin_amdgcn_s_waitcnt(0);
  c.e += 1;
  if (c.lane == 0)
    __hip_atomic_store(reinterpret_cast<uint64_t*>(c.wsp + OFF_XFLAG) + (c.x * NR + c.r) * NCW + c.wave, c.e,
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// Waits until ready(lane) holds in every lane of the wave; `load` returns whether the lane's flags are.
template <class F>
__device__ __forceinline__ void poll(const Ctx& c, const F& ok) {
  if (aborted(c)) return;
  for (unsigned it = 0;; ++it) {
    if (__builtin_amdgcn_ballot_w64(!ok()) == 0) break;
    if (it > kSpinCap) {
      if (c.lane == 0) atomicOr(c.err, kErrSpin);
      break;
    }
    __builtin_amdgcn_s_sleep(1);
  }
  asm volatile("" ::: "memory");  // loads after the wait stay after it
}
__device__ __forceinline__ bool flag_ge(u32x2 v, uint64_t e) { return (((uint64_t)v[1] << 32) | v[0]) >= e; }

__device__ __forceinline__ void xcd_sync(Ctx& c) {
  xcd_signal(c);
  const uint32_t off = OFF_XFLAG + c.x * (NR * NCW * 8) + c.lane * 16;
  poll(c, [&] {
    const u32x4 v = ldb128<kCpSc1>(c.ws, off);
    return flag_ge(u32x2{v[0], v[1]}, c.e) && flag_ge(u32x2{v[2], v[3]}, c.e);
  });
}
// Wait until wave `wv` (waves w0 and w1) of the ranks in `mask` has passed the sync point this wave passed
// last; xcd_wait: this wave's own index.
__device__ __forceinline__ void xcd_wait_w(const Ctx& c, uint32_t mask, int wv) {
  const bool mine = c.lane < NR && ((mask >> (c.lane & 31)) & 1u);
  const uint32_t off = mine ? OFF_XFLAG + ((c.x * NR + c.lane) * NCW + wv) * 8 : OOB;
  poll(c, [&] { return !mine || flag_ge(ldb64<kCpSc1>(c.ws, off), c.e); });
}
__device__ __forceinline__ void xcd_wait_w2(const Ctx& c, uint32_t mask, int w0, int w1) {
  const bool mine = (mask >> (c.lane & 31)) & 1u;
  const uint32_t off = mine ? OFF_XFLAG + ((c.x * NR + (c.lane & 31)) * NCW + (c.lane < 32 ? w0 : w1)) * 8 : OOB;
  poll(c, [&] { return !mine || flag_ge(ldb64<kCpSc1>(c.ws, off), c.e); });
}
__device__ __forceinline__ void xcd_wait(const Ctx& c, uint32_t mask) { xcd_wait_w(c, mask, c.wave); }

// Partial sums: published to the whole group. With G = 1 that is the XCD; otherwise the stores went out
// with sc1 and so does the flag (its own array, read across XCDs).
template <class K>
__device__ __forceinline__ void part_signal(Ctx& c) {
  if constexpr (K::G == 1) {
    xcd_signal(c);
  } else {
    __builtin_amdgcn_s_waitcnt(0);
    c.eg += 1;
    if (c.lane == 0)
      __hip_atomic_store(reinterpret_cast<uint64_t*>(c.wsp + kWsGroupFlags) + (c.x * NR + c.r) * NCW + c.wave, c.eg,
                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}
template <class K>
__device__ __forceinline__ void part_wait(const Ctx& c) {
  if constexpr (K::G == 1) {
    xcd_wait(c, 0xffffffffu);
  } else {
    const uint32_t off = kWsGroupFlags + ((c.grp * K::G * NR + c.lane) * NCW + c.wave) * 8;
    poll(c, [&] {
      u32x2 v[K::G / 2];
#pragma unroll
      for (int i = 0; i < K::G / 2; i++) v[i] = ldb64<kCpSc1>(c.ws, off + i * 64 * NCW * 8);
      bool ok = true;
#pragma unroll
      for (int i = 0; i < K::G / 2; i++) ok = ok && flag_ge(v[i], c.eg);
      return ok;
    });
  }
}
// cache policy of partial-sum stores: they leave the XCD only with G > 1
template <class K>
constexpr int kCpPart = K::G == 1 ? kCpPlain : kCpSc1;

// ---------------------------------------------------------------- weight ring
template <class K>
__device__ __forceinline__ void page_wait(const Ctx& c, int pg) {
  for (unsigned it = 0;; ++it) {
    const unsigned r0 = ctl_ld<K>(0), r1 = ctl_ld<K>(1);
    if ((int)min(r0, r1) > pg || ctl_ld<K>(6)) break;
    if (it > kSpinCap) {
      ctl_st<K>(6, 1u);
      if (c.lane == 0) atomicOr(c.err, kErrSpin);
      break;
    }
    __builtin_amdgcn_s_sleep(1);
  }
  asm volatile("" ::: "memory");
}
template <class K>
__device__ __forceinline__ void page_release(const Ctx& c, int upto) {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this wave's LDS reads have returned
  if (c.lane == 0) ctl_st<K>(2 + c.wave, (unsigned)upto);
}

// global_load_lds_dwordx4 with a wave-uniform base and a 32-bit lane offset: lane i copies 16 bytes to
// LDS m0 + 16 i (fragments in the order of copy_row / copy_chunk).
__device__ __forceinline__ void dma16(const unsigned char* base, uint32_t voff, uint32_t lds) {
  unsigned saved;
  // (each half is cast to uint32_t before widening: readfirstlane returns int)
  const uint64_t a = reinterpret_cast<uint64_t>(base);
  const uint64_t u = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(a >> 32)) << 32 |
                     (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)a);
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0"
               : "=&s"(saved)
               : "v"(voff), "s"(u), "s"(__builtin_amdgcn_readfirstlane(lds))
               : "memory");
}

#define FA_PG_VMCNT(n) (((n) & 15) | (((n) >> 4) << 14) | (7 << 4) | (15 << 8))

// Loader wave lw copies fragments 8 lw .. 8 lw + 7 of every page, in the order the compute waves read them.
// A page needs its ring slot released by the four compute waves and at most MAXF of this wave's pages in
// flight; every page is eight copies per wave, so the waits count them.
template <class K>
struct LoaderBase {
  const Ctx& c;
  int lw, pg = 0, done = 0;
  bool ok = true;
  __device__ LoaderBase(const Ctx& c_, int lw_) : c(c_), lw(lw_) {}

  __device__ __forceinline__ void complete_oldest() {
    if (pg - done > 1)  // another page is in flight behind the oldest
      __builtin_amdgcn_s_waitcnt(FA_PG_VMCNT(8));
    else
      __builtin_amdgcn_s_waitcnt(FA_PG_VMCNT(0));
    static_assert(MAXF <= 2, "waits cover two pages in flight");
    asm volatile("" ::: "memory");
    ++done;
    if (c.lane == 0) ctl_st<K>(lw, (unsigned)done);
  }
  __device__ __forceinline__ bool room() {
    for (unsigned idle = 0;;) {
      if (pg - done < MAXF) {
        if (pg < K::RING) return true;
        const unsigned m = min(min(ctl_ld<K>(2), ctl_ld<K>(3)), min(ctl_ld<K>(4), ctl_ld<K>(5)));
        if ((int)m >= pg - K::RING + 1) return true;
      }
      if (done < pg) {
        complete_oldest();
        idle = 0;
        continue;
      }
      if (ctl_ld<K>(6) || ++idle > kSpinCap) {
        if (!ctl_ld<K>(6)) {
          ctl_st<K>(6, 1u);
          if (c.lane == 0) atomicOr(c.err, kErrSpin);
        }
        ok = false;
        return false;
      }
      __builtin_amdgcn_s_sleep(1);
    }
  }
  __device__ __forceinline__ uint32_t dst() const { return c.lds_addr + (uint32_t)(pg % K::RING) * PAGE + lw * 8192; }

  // NFR fragments of a GEMM stage with R row tiles, fragment F = (k-step F / R, row tile F % R): base(rt) = the tile's first row at the stage's first k
  template <int R, int NFR, class Base>
  __device__ __forceinline__ void stage(uint32_t voff, const Base& base) {
#pragma unroll 1
    for (int i = 0; i < (NFR + 15) / 16 && ok; i++) {
      if (!room()) return;
      const uint32_t d = dst();
#pragma unroll
      for (int f = 0; f < 8; f++) {
        const int F = min(16 * i + 8 * lw + f, NFR - 1), ks = F / R, rt = F - ks * R;  // past the last: repeated
        dma16(base(rt) + ks * 64, voff, d + f * 1024);
      }
      pg++;
    }
  }

  __device__ __forceinline__ void drain() {
    if (ok)
      while (done < pg) complete_oldest();
    __builtin_amdgcn_s_waitcnt(0);
  }
};

// ---------------------------------------------------------------- GEMM (NB token tiles per wave)
// acc[n][rt] = W[row tile rt][k] X[token][k] over KS k-steps, weights from ring pages pg0.. (fragment
// F = ks R + rt), tokens from the workspace at xoff[n] + 1 KB per k-step (OOB: zeros). The operand
// loads run two chunks of KC k-steps ahead (one chunk's MFMAs take 0.3-0.4 us, less than a loaded L2
// round trip); A fragments are read from LDS in batches ahead of their MFMAs, each feeding NB of them;
// pages are released as their last fragment is read.
template <class K, int R, int KS, int NB>
__device__ __forceinline__ void gemm(f32x4 (&acc)[NB][R], const Ctx& c, int pg0, const uint32_t (&xoff)[NB]) {
  constexpr int KC = KS % (8 / NB) == 0 ? 8 / NB : KS % (6 / NB) == 0 ? 6 / NB : 1, NCK = KS / KC, NA = KC * R;
  constexpr int AB = NA % 8 == 0 ? 8 : (NA % 5 == 0 ? 5 : (NA % 6 == 0 ? 6 : (NA % 4 == 0 ? 4 : 3)));
  static_assert(NA % AB == 0, "whole batches");
  constexpr int CH = R * NB >= 4 ? 1 : 2;  // accumulator chains per row tile
  f32x4 ac[CH][NB][R];
#pragma unroll
  for (int h = 0; h < CH; h++)
#pragma unroll
    for (int n = 0; n < NB; n++)
#pragma unroll
      for (int rt = 0; rt < R; rt++) ac[h][n][rt] = f32x4{0.f, 0.f, 0.f, 0.f};
  const uint32_t fo = frag_slot(c.lr, c.lq);
  u32x4 xf[3][NB][KC];
  auto load = [&](int ck) __attribute__((always_inline)) {
#pragma unroll
    for (int n = 0; n < NB; n++)
#pragma unroll
      for (int k = 0; k < KC; k++) xf[ck % 3][n][k] = ldb128<kCpSc1>(c.ws, xoff[n] + (ck * KC + k) * 1024);
  };
  load(0);
  if (NCK > 1) load(1);
#pragma unroll
  for (int ck = 0; ck < NCK; ck++) {
    if (ck + 2 < NCK) load(ck + 2);
    page_wait<K>(c, pg0 + ((ck + 1) * NA - 1) / 16);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int h = 0; h < NA; h += AB) {
      u32x4 af[AB];
#pragma unroll
      for (int q = 0; q < AB; q++) {
        const int F = ck * NA + h + q;
        af[q] = *reinterpret_cast<const u32x4*>(fg_lds + ((pg0 + F / 16) % K::RING) * PAGE + fo + (F % 16) * 1024);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < AB; q++) {
        const int k = (h + q) / R, rt = (h + q) % R;
#pragma unroll
        for (int n = 0; n < NB; n++) ac[k % CH][n][rt] = mfma16(af[q], xf[ck % 3][n][k], ac[k % CH][n][rt]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    // whole pages, and with the last chunk a page that its fragments only began
    constexpr int last = (KS * R + 15) / 16;
    const int upto = ck + 1 == NCK ? last : (ck + 1) * NA / 16;
    if (upto > ck * NA / 16) page_release<K>(c, pg0 + upto);
  }
#pragma unroll
  for (int n = 0; n < NB; n++)
#pragma unroll
    for (int rt = 0; rt < R; rt++) acc[n][rt] = CH == 2 ? ac[0][n][rt] + ac[CH - 1][n][rt] : ac[0][n][rt];
}

// The launch sequence advances when the last of `groups` groups is done: the groups do not wait for one
// another, and a workgroup that starts late must still read this launch's number. Run by one lane of a
// group, whose wave has seen every wave of the group past the prologue.
__device__ __forceinline__ void finish_group(unsigned char* ws, uint64_t seq, unsigned groups, unsigned owner) {
  unsigned* done = reinterpret_cast<unsigned*>(ws + OFF_DONE);
  if (__hip_atomic_fetch_add(done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != groups - 1) return;
  __hip_atomic_store(done, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(reinterpret_cast<unsigned*>(ws + kWsOwner), owner, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(reinterpret_cast<uint64_t*>(ws + OFF_CTRL), seq + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace grp
}  // namespace fa
