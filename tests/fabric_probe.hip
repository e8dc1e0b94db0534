// Latency and bandwidth probe of the MI355X fabric (gfx950), the measurements behind the per-phase
// latency budget of the batch-1 kernels:
//   handoff: one wave of workgroup 0 and one wave of a partner workgroup pass a round number back and
//            forth ROUNDS times. Workgroup 0 stores 1 KB of data, waits for the stores (timed: the
//            store acknowledgement), stores a flag; the partner polls the flag (sc1 loads), reads and
//            checks the data (sc1), stores its own flag; workgroup 0 polls that (the whole round trip is
//            timed). Partner 8 (rank 1 of XCD 0) is on workgroup 0's XCD: data and flags as plain stores,
//            which stay in the XCD's L2, or as sc1 stores. Partner 1 is on XCD 1: sc1 stores (plain
//            stores would stay in XCD 0's L2 and never reach it).
//   stream : 256 workgroups read a 1 GiB buffer in 32 MiB chunks (each XCD's 32 CUs split a chunk), in
//            three modes: every XCD reads the same chunk sequence; every XCD reads its own chunks; XCD 0
//            alone. Bandwidth per XCD and over the active XCDs.
//   copy   : 256 workgroups, two waves each, copy fragments of 16 rows x 64 bytes (rows 512 bytes apart, as K and
//            V of a prefix) into an LDS ring of 8 pages of 16 KB, two pages in flight per wave, with a lane's
//            row and 16-byte chunk in MFMA order (row lane % 16, chunk lane / 16) or four neighbouring
//            lanes to a row (copy_row and copy_chunk of fa_device.h). From the L2 (1 MiB per XCD, over and over)
//            and from memory (32 MiB that eight workgroups of an XCD share, as the heads of a sample its K
//            and V). The last page is compared with its source.
//   lds    : 4 waves of one workgroup per CU read whole fragments back, 16 bytes per lane: in MFMA order, in
//            the order of frag_slot (fa_device.h), and in that order without its rotation.
// Every index is in bounds, every wait is capped (a side whose wait hits the cap stops), and only
// workgroups 0 and the partner take part in a hand-off (the others return at once); the stream kernel
// stores one word per workgroup at most.
// usage: fabric_probe      prints one line per measurement, then "FABRIC OK" when no read was stale,
//                          no wait hit its cap and every workgroup ran on the XCD its index implies.
#include <hip/hip_runtime.h>

#include <cstdio>

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

constexpr int ROUNDS = 400;
constexpr unsigned CAP = 1u << 20;                 // polls per wait
constexpr unsigned DATA = 64 * 1024;               // data ring: 64 slots of 1 KB
constexpr unsigned F0 = DATA, F1 = DATA + 4096;    // flags, one per side, 4 KB apart
constexpr unsigned BUF = DATA + 8192;

__device__ __forceinline__ unsigned xcc() { return __builtin_amdgcn_s_getreg((3 << 11) | (0 << 6) | 20) & 7u; }

// out[0] store-ack ticks, [1] round-trip ticks (100 MHz ticks, summed over rounds), [3] stale reads,
// [4] / [7] capped waits of workgroup 0 / the partner, [5] XCD of workgroup 0, [6] XCD of the partner
template <int CP>
__global__ void __launch_bounds__(64) handoff(unsigned char* buf, int partner, unsigned long long* out) {
  const int me = blockIdx.x, lane = threadIdx.x;
  if (me != 0 && me != partner) return;
  const auto r = __builtin_amdgcn_make_buffer_rsrc(buf, (short)0, (int)BUF, 0x00020000);
  unsigned long long ack = 0, rt = 0, bad = 0, capped = 0;
  if (lane == 0) out[me == 0 ? 5 : 6] = xcc();
  for (unsigned i = 1; i <= ROUNDS; i++) {
    const unsigned doff = (i % 64) * 1024 + lane * 16;
    if (me == 0) {
      const unsigned long long t0 = __builtin_amdgcn_s_memrealtime();
      __builtin_amdgcn_raw_buffer_store_b128(u32x4{i, i, i, i}, r, doff, 0, CP);
      __builtin_amdgcn_s_waitcnt(0);
      const unsigned long long t1 = __builtin_amdgcn_s_memrealtime();
      if (lane == 0) __builtin_amdgcn_raw_buffer_store_b32(i, r, F0, 0, CP);
      unsigned it = 0;
      for (; it < CAP; it++) {
        if (__builtin_amdgcn_readfirstlane(__builtin_amdgcn_raw_buffer_load_b32(r, F1, 0, 16)) == i) break;
        __builtin_amdgcn_s_sleep(1);
      }
      const unsigned long long t2 = __builtin_amdgcn_s_memrealtime();
      ack += t1 - t0;
      rt += t2 - t0;
      if (it >= CAP) {  // the partner is gone: stop (it stops at its own next capped wait)
        capped++;
        break;
      }
    } else {
      unsigned it = 0;
      for (; it < CAP; it++) {
        if (__builtin_amdgcn_readfirstlane(__builtin_amdgcn_raw_buffer_load_b32(r, F0, 0, 16)) == i) break;
        __builtin_amdgcn_s_sleep(1);
      }
      if (it >= CAP) {
        capped++;
        break;
      }
      const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, doff, 0, 16);
      bad += (v[0] != i) | (v[3] != i);
      if (lane == 0) __builtin_amdgcn_raw_buffer_store_b32(i, r, F1, 0, CP);
      __builtin_amdgcn_s_waitcnt(0);
    }
  }
  // stale reads and capped waits of any lane; timings of lane 0
  bad = __builtin_amdgcn_ballot_w64(bad != 0) != 0;
  if (lane == 0) {
    if (me == 0) {
      out[0] = ack;
      out[1] = rt;
      out[4] = capped;
    } else {
      out[3] = bad;
      out[7] = capped;
    }
  }
}

// Workgroup b runs on XCD b % 8 as rank b / 8 (recorded in xccs). mode 0: every XCD reads the same
// chunk sequence; mode 1: each XCD its own chunks; mode 2: XCD 0 alone.
__global__ void __launch_bounds__(256) stream(const unsigned char* W, unsigned long long size, int mode, int chunks,
                                              unsigned long long cb, unsigned* sink, unsigned* xccs) {
  const int x = blockIdx.x & 7, rk = blockIdx.x >> 3;
  if (threadIdx.x == 0) xccs[blockIdx.x] = xcc();
  if (mode == 2 && x != 0) return;
  u32x4 acc = {0, 0, 0, 0};
  const unsigned long long per_cu = cb / 32;  // bytes of a chunk per CU
  for (int c = 0; c < chunks; c++) {
    const unsigned long long base =
        mode == 1 ? ((unsigned long long)(c * 8 + x) * cb) % size : ((unsigned long long)c * cb) % size;
    const unsigned char* p = W + base + rk * per_cu;
    for (unsigned long long o = threadIdx.x * 16; o < per_cu; o += 256 * 16 * 8) {
      u32x4 v[8];
#pragma unroll
      for (int k = 0; k < 8; k++) {
        const unsigned long long oo = o + k * 256 * 16;
        v[k] = oo < per_cu ? *reinterpret_cast<const u32x4*>(p + oo) : u32x4{0, 0, 0, 0};
      }
#pragma unroll
      for (int k = 0; k < 8; k++) acc ^= v[k];
    }
  }
  const unsigned s = acc[0] ^ acc[1] ^ acc[2] ^ acc[3];
  if (s == 0x12345678u) sink[blockIdx.x] = s;  // keeps the loads live
}

__device__ __forceinline__ int quad_row(int lane) { return lane >> 2; }
__device__ __forceinline__ int quad_chunk(int lane) { return (lane ^ -(lane >> 4)) & 3; }
__device__ __forceinline__ unsigned quad_slot(int lr, int lq) { return lr * 64 + ((lq ^ -(lr >> 2)) & 3) * 16; }

constexpr int PAGE = 16384, RING = 8;
extern __shared__ __attribute__((aligned(16))) unsigned char ring[];

__global__ void fill(unsigned* W, unsigned long long n) {
  for (unsigned long long i = blockIdx.x * (unsigned long long)blockDim.x + threadIdx.x; i < n;
       i += (unsigned long long)gridDim.x * blockDim.x)
    W[i] = (unsigned)i;
}

// W: 1 GiB of words that hold their index. L2: 256 pages of the XCD's own MiB, else 2048 of the eight workgroups'.
template <bool L2>
constexpr int kPages = L2 ? 256 : 2048;
template <bool QUAD, bool L2>
__global__ void __launch_bounds__(128) copy_order(const unsigned char* W, unsigned* bad) {
  constexpr int PAGES = kPages<L2>;
  const int x = blockIdx.x & 7, rk = blockIdx.x >> 3, lane = threadIdx.x & 63, lw = threadIdx.x >> 6;
  const int row = QUAD ? quad_row(lane) : lane & 15, chunk = QUAD ? quad_chunk(lane) : lane >> 4;
  auto src = [&](int pg) {  // of this wave: 16 rows x 512 bytes
    const unsigned long long page = L2 ? x * 64ull + (pg + 2 * rk) % 64 : (x * 4ull + rk / 8) * PAGES + pg;
    return W + page * PAGE + lw * 8192;
  };
  for (int pg = 0; pg < PAGES; pg++) {
    const unsigned char* s = src(pg) + row * 512 + chunk * 16;
    unsigned char* d = ring + (pg % RING) * PAGE + lw * 8192;
#pragma unroll
    for (int f = 0; f < 8; f++)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(s + f * 64),
                                       (__attribute__((address_space(3))) void*)(d + f * 1024), 16, 0, 0);
    __builtin_amdgcn_s_waitcnt(8 | (7 << 4) | (15 << 8));  // vmcnt(8): the page before has landed
  }
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  // MFMA lane (lr, lq) of every fragment of the last page: row lr, chunk lq
  const int lr = lane & 15, lq = lane >> 4;
  const unsigned first = (unsigned)((src(PAGES - 1) - W) / 4);
  unsigned wrong = 0;
  for (int f = 0; f < 8; f++) {
    const u32x4 v = *reinterpret_cast<const u32x4*>(ring + ((PAGES - 1) % RING) * PAGE + lw * 8192 + f * 1024 +
                                                    (QUAD ? quad_slot(lr, lq) : lane * 16));
    const unsigned want = first + lr * 128 + f * 16 + lq * 4;
    wrong |= (v[0] != want) | (v[3] != want + 3);
  }
  if (wrong) atomicOr(bad, 1u);
}

// MODE 0 MFMA order, 1 frag_slot, 2 frag_slot without the rotation. 16 fragments per pass and wave.
template <int MODE>
__global__ void __launch_bounds__(256) lds_read(int passes, unsigned* sink) {
  const int lane = threadIdx.x & 63, lr = lane & 15, lq = lane >> 4;
  for (int i = threadIdx.x; i < RING * PAGE / 4; i += 256) reinterpret_cast<unsigned*>(ring)[i] = i;
  __syncthreads();
  const unsigned at = (threadIdx.x >> 6) * 2 * PAGE + (MODE == 0 ? lane * 16 : MODE == 1 ? quad_slot(lr, lq) : lr * 64 + lq * 16);
  u32x4 acc = {0, 0, 0, 0};
  for (int p = 0; p < passes; p++) {
    unsigned a = at + (p & 1) * PAGE;
    asm volatile("" : "+v"(a));  // read anew in every pass
    u32x4 v[16];
#pragma unroll
    for (int f = 0; f < 16; f++) v[f] = *reinterpret_cast<const u32x4*>(ring + a + f * 1024);
#pragma unroll
    for (int f = 0; f < 16; f++) acc ^= v[f];
  }
  const unsigned s = acc[0] ^ acc[1] ^ acc[2] ^ acc[3];
  if (s == 0x12345678u) sink[blockIdx.x] = s;
}

int main() {
  unsigned char* buf = nullptr;
  unsigned long long* out = nullptr;
  if (hipMalloc(&buf, BUF) != hipSuccess || hipMalloc(&out, 8 * 8) != hipSuccess) return 2;
  int bad = 0;
  const int cases[3][2] = {{8, 0}, {8, 1}, {1, 1}};  // (partner, sc1 stores)
  for (const auto& cs : cases) {
    const int partner = cs[0], sc1 = cs[1];
    {
      if (hipMemset(buf, 0, BUF) != hipSuccess || hipMemset(out, 0, 64) != hipSuccess) return 2;
      if (sc1)
        hipLaunchKernelGGL(handoff<16>, dim3(256), dim3(64), 0, 0, buf, partner, out);
      else
        hipLaunchKernelGGL(handoff<0>, dim3(256), dim3(64), 0, 0, buf, partner, out);
      if (hipDeviceSynchronize() != hipSuccess) return 3;
      unsigned long long t[8];
      if (hipMemcpy(t, out, sizeof(t), hipMemcpyDeviceToHost) != hipSuccess) return 3;
      const bool same = t[5] == t[6];
      if (t[5] != 0 || t[6] != (unsigned long long)(partner % 8)) bad = 1;
      if (t[3] || t[4] || t[7]) bad = 1;
      printf("handoff %s %s: store_ack_ns %.0f round_trip_ns %.0f stale %llu capped %llu\n", same ? "same-xcd" : "cross-xcd",
             sc1 ? "sc1" : "plain", t[0] * 10.0 / ROUNDS, t[1] * 10.0 / ROUNDS, t[3], t[4] + t[7]);
    }
  }
  (void)hipFree(buf);
  (void)hipFree(out);

  const unsigned long long size = 1ull << 30, cb = 32ull << 20;
  unsigned char* W = nullptr;
  unsigned *sink = nullptr, *xccs = nullptr;
  if (hipMalloc(&W, size) != hipSuccess || hipMalloc(&sink, 4096) != hipSuccess || hipMalloc(&xccs, 4096) != hipSuccess)
    return 2;
  if (hipMemset(W, 7, size) != hipSuccess) return 2;
  hipEvent_t a, b;
  if (hipEventCreate(&a) != hipSuccess || hipEventCreate(&b) != hipSuccess) return 2;
  const int chunks = (int)((2ull << 30) / cb / 8);  // 256 MiB per XCD
  const char* names[3] = {"same-data", "own-data", "xcd0-alone"};
  for (int mode = 0; mode < 3; mode++) {
    float ms = 0.f;
    for (int rep = 0; rep < 2; rep++) {  // the second launch is reported
      (void)hipEventRecord(a);
      hipLaunchKernelGGL(stream, dim3(256), dim3(256), 0, 0, W, size, mode, chunks, cb, sink, xccs);
      (void)hipEventRecord(b);
      if (hipEventSynchronize(b) != hipSuccess) return 3;
      (void)hipEventElapsedTime(&ms, a, b);
    }
    const double per_xcd = (double)chunks * cb;
    const int nx = mode == 2 ? 1 : 8;
    printf("stream %s: per_xcd_GBs %.0f total_GBs %.0f ms %.3f\n", names[mode], per_xcd / ms / 1e6,
           nx * per_xcd / ms / 1e6, ms);
  }
  auto timed = [&](auto launch) {  // ms of the second launch, negative on an error
    float ms = -1.f;
    for (int rep = 0; rep < 2; rep++) {
      (void)hipEventRecord(a);
      launch();
      (void)hipEventRecord(b);
      if (hipEventSynchronize(b) != hipSuccess || hipEventElapsedTime(&ms, a, b) != hipSuccess) return -1.f;
    }
    return ms;
  };
  static_assert(32ull * kPages<false> * PAGE == 1ull << 30, "the copies' pages are the buffer");
  hipLaunchKernelGGL(fill, dim3(2048), dim3(256), 0, 0, reinterpret_cast<unsigned*>(W), size / 4);
  unsigned wrong = 1;
  if (hipMemset(sink, 0, 4) != hipSuccess) return 2;
  const auto copies = {(const void*)copy_order<false, true>, (const void*)copy_order<true, true>,
                       (const void*)copy_order<false, false>, (const void*)copy_order<true, false>};
  const auto reads = {(const void*)lds_read<0>, (const void*)lds_read<1>, (const void*)lds_read<2>};
  for (const void* k : copies)
    if (hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, RING * PAGE) != hipSuccess) return 2;
  for (const void* k : reads)
    if (hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, RING * PAGE) != hipSuccess) return 2;
  const char* cn[4] = {"l2 mfma-order", "l2 quad-order", "memory mfma-order", "memory quad-order"};
  int i = 0;
  for (const void* k : copies) {
    const float ms = timed([&] {
      const unsigned char* w = W;
      void* args[] = {&w, &sink};
      (void)hipLaunchKernel(k, dim3(256), dim3(128), args, RING * PAGE, 0);
    });
    if (ms <= 0.f) return 3;
    printf("copy %s: per_cu_GBs %.1f\n", cn[i], (double)(i < 2 ? kPages<true> : kPages<false>) * PAGE / ms / 1e6);
    i++;
  }
  if (hipMemcpy(&wrong, sink, 4, hipMemcpyDeviceToHost) != hipSuccess) return 3;
  if (wrong) bad = 1;
  const char* rn[3] = {"mfma-order", "rotated", "unrotated"};
  i = 0;
  for (const void* k : reads) {
    int passes = 4000;
    const float ms = timed([&] {
      void* args[] = {&passes, &sink};
      (void)hipLaunchKernel(k, dim3(256), dim3(256), args, RING * PAGE, 0);
    });
    if (ms <= 0.f) return 3;
    printf("lds %s: per_cu_GBs %.0f\n", rn[i++], 4.0 * passes * PAGE / ms / 1e6);
  }
  unsigned h[256];
  if (hipMemcpy(h, xccs, sizeof(h), hipMemcpyDeviceToHost) != hipSuccess) return 3;
  for (int i = 0; i < 256; i++)
    if (h[i] != (unsigned)(i % 8)) bad = 1;
  (void)hipFree(W);
  (void)hipFree(sink);
  (void)hipFree(xccs);
  printf(bad ? "FABRIC FAILED\n" : "FABRIC OK\n");
  return bad;
}
