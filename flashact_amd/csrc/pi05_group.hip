// pi0.5 action-expert denoise loop for 2 to 16 samples: groups of XCDs, each group running its own
// samples through the whole S-step Euler loop with no grid-wide barrier. ONE cooperative launch of 256
// workgroups (one per CU) of 6 waves.
//
// G XCDs form a group (G = 4: 2 groups, G = 2: 4, G = 1: 8) of up to NB samples (NB = 1 or 2).
// XCD j of a group owns query heads [8/G j, 8/G (j + 1)), MLP columns [4096/G j, ..) and those K windows
// of the O and down projections, so everything but the projections' partial sums stays in its L2.
// Within the XCD, rank r = blockIdx / 8 owns output rows of every GEMM; the O and down projections are
// also split over C = 4/G K windows of 512 / 1024, so a rank reads a quarter of the token operand instead
// of all of it, and every group ends with 4 partial sums per residual update (the K split of the
// stage-engine kernel, pi05_batched.hip).
// Waves 0-3 compute: wave w owns tokens 16w..16w+15 of each of the group's samples in every stage (NB
// token tiles) and signals its own flags, so no workgroup barrier runs after the prologue. Waves 4-5
// load: they stream the CU's weight rows and its chunk's prefix K/V from HBM into an 8-page LDS ring
// (16 KB pages), free-running ahead of the compute waves.
//
// Per layer ([W] = waits for the waves that wrote the operand, [X] = XCD barrier, {E} = waits for the
// group's partial sums):
//   N1   x += gate * sum of the 4 down partials (layer 0: x = embed(x_t)); xn = adaRMS(x)   (x in LDS)
//   [W] QKV   2048/G + 512 rows (heads of the XCD, all k and v), RoPE
//   [X] ATT   item = (sample, head, key chunk), 32 items: prefix keys from the ring, this step's keys
//             spread over the chunks
//   [W] COMB  key chunks combined, one operand fragment at a time
//   [W] O     partial sums {E} N2 [W] GU [W] DN partial sums {E}
//
// What bounds it: each group streams all 34.6 MB of a layer's weights, 34.6/G MB per XCD. The fabric
// feeds one XCD at 0.80-0.97 TB/s while all eight read, 1.3 alone (tests/fabric_probe.hip): about 40 us per
// layer with G = 1, 20 with G = 2, 10 with G = 4. The stage engine at these batches had 40 to 180 GEMM items for the 256
// CUs in every stage but gate/up, and eight grid barriers of about 2 us per layer. At 16 samples a layer takes
// 88 us: gate/up 20.7, attention 17.5 (its 512 KB of K/V per CU arrive at 44 GB/s; without softmax and P V it
// takes as long), down 11.1, QKV 8.6, the norms 14.5 with the waits for the partial sums, barriers 5.7.
#include "group.h"
#include "../../include/flashact_mi355x.h"
#include "fa_host.h"

namespace fa {
namespace pg {
using namespace fa::grp;

constexpr int D = 1024, HD = 256, AD = 32, FF = 4096, QD = 2048;
constexpr int TP = 64;   // token slots of a sample
constexpr int RING = 8;  // ring pages

// Shape of one configuration: G XCDs per group, NB samples per group.
template <int G_, int NB_>
struct Cfg {
  static constexpr int G = G_, NB = NB_, RING = pg::RING;
  static constexpr int NGRP = NX / G;
  static constexpr int HX = 8 / G;             // heads per XCD
  static constexpr int C = 4 / G;              // K windows of the O and down projections per XCD
  static constexpr int NKC = NR / (NB * HX);   // key chunks per (sample, head)
  static constexpr int SK = TP / NKC;          // this step's keys per chunk
  static constexpr int SKT = SK > 16 ? 2 : 1;  // their key tiles (tile kt holds keys 8 a + 4 kt + i, see below)
  static constexpr int SEGU = NKC >= 16 ? 1 : 2;  // 64-key units per attention segment
  static constexpr int RQ = (QD / G + 512) / (16 * NR);  // row tiles per rank: QKV
  static constexpr int RP = D * C / (16 * NR);           // O and down
  static constexpr int RG = 2 * FF / G / (16 * NR);      // gate/up, in PG passes of RGP
  static constexpr int PG = RG > 8 ? 2 : 1, RGP = RG / PG;
  static constexpr int KO = 16, KD = 32, KX = 32;  // k-steps: O window, down window, QKV and gate/up
  static constexpr int PQ = RQ * KX / 16, PO = RP * KO / 16, PGU = RG * KX / 16, PD = RP * KD / 16;  // pages
  static constexpr int FPR = NB * HX / 4;      // combine fragments per wave (0: ranks < 16 take one)
  // workspace of one XCD (bytes), operands in MFMA fragment order [tile (n, w)][k-step][1 KB]
  static constexpr uint32_t X_XN = 0;
  static constexpr uint32_t X_Q = X_XN + NB * TP * D * 2;             // [n][head][w][8 k-steps]
  static constexpr uint32_t X_ATTP = X_Q + NB * HX * TP * HD * 2;     // [rank][w][8 k-steps]
  static constexpr uint32_t X_ML = X_ATTP + NR * TP * HD * 2;         // [rank][64] (m, l)
  static constexpr uint32_t X_ATTN = X_ML + NR * TP * 8;              // [n, w][8 HX k-steps]
  static constexpr uint32_t X_H = X_ATTN + NB * TP * HX * HD * 2;     // [n, w][128 / G k-steps]
  static constexpr uint32_t X_KS = X_H + NB * TP * (FF / G) * 2;      // [layer parity][n][64][256]
  static constexpr uint32_t X_VS = X_KS + 2 * NB * TP * HD * 2;       // [layer parity][n][256][64]
  static constexpr uint32_t XB = X_VS + 2 * NB * TP * HD * 2;
  static constexpr uint32_t OFF_XCD = kWsDataBase;
  // fp32 partial sums [O | down][4 windows][NB 64 tokens][1024] of one group; one buffer serves both with
  // G = 1, where the down projection starts only after every reader of the O partials is done
  static constexpr uint32_t PB1 = 4u * NB * TP * D * 4, PB = (G == 1 ? 1 : 2) * PB1;
  static constexpr uint32_t OFF_PART = OFF_XCD + NX * XB;
  static constexpr uint32_t WS = OFF_PART + NGRP * PB;
  // LDS (bytes)
  static constexpr uint32_t L_CTL = RING * PAGE;           // u32 ready[2], consumed[4], abort
  static constexpr uint32_t L_XRES = L_CTL + 64;           // f32 [2 NB][1024] residual rows
  static constexpr uint32_t L_XT = L_XRES + 2 * NB * D * 4;  // f32 [2 NB][32] x_t rows
  static constexpr uint32_t LDS = L_XT + 2 * NB * AD * 4;
  static_assert(LDS <= 160 * 1024, "LDS of one CU");
  static_assert(NB * HX * NKC == NR && NKC >= 2 && NB <= 2, "one attention item per rank");
};
__host__ __device__ constexpr uint32_t frag_off(int KS, int t, int k) {  // as in pi05_bs1.hip
  return (uint32_t)(((((t >> 4) * KS + (k >> 5)) * 4 + ((k >> 3) & 3)) * 16 + (t & 15)) * 16 + (k & 7) * 2);
}

struct Params {
  const bf16* w1;
  const bf16* wo;
  const bf16* w2;
  const bf16* w3;
  const float* mods;
  const float* mod_final;
  const float* rope_cos;
  const float* rope_sin;
  const float* w_ain;
  const float* b_ain;
  const float* w_aout;
  const float* b_aout;
  bf16* kcache;
  bf16* vtcache;
  float* x_t;
  unsigned long long* stage_cycles;
  unsigned char* ws;
  int NL, Lp, Lmax, S, Tv, B, xt_rows;
};

struct PCtx : Ctx {
  int an, ah, kbeg, kend, sbeg, nsfx, nun;  // attention item: slot, head, prefix keys, this step's keys, 64-key units
  rsrc_t rc, rs;
};

// Token t of a sample is normed by rank t % 32, wave t / 16: the norm waves of this wave's tile.
__device__ __forceinline__ void wait_norm_rows(const Ctx& c) { xcd_wait(c, c.wave & 1 ? 0xffff0000u : 0xffffu); }

// First row of QKV row tile rt of rank r (virtual rows: this XCD's heads, then k, then v).
template <class K>
__device__ __forceinline__ int qkv_row(int j, int vr) {
  return vr < 256 * K::HX ? 256 * K::HX * j + vr : QD + (vr - 256 * K::HX);
}

// The pages of a layer: QKV, the chunk's segments of K and V^T, O, gate/up (PG passes), down.
template <class K>
struct Loader : LoaderBase<K> {
  const Params& p;
  const PCtx& c;
  __device__ Loader(const Params& p_, const PCtx& c_, int lw_) : LoaderBase<K>(c_, lw_), p(p_), c(c_) {}

  __device__ void run() {
    const int NL = p.NL;
    const int cr = copy_row(c.lane), cq = copy_chunk(c.lane);
    const uint32_t vq = cr * (D * 2) + cq * 16, vo = cr * (QD * 2) + cq * 16, vd = cr * (FF * 2) + cq * 16;
    const int win = c.r / (NR / K::C), rg = c.r % (NR / K::C);  // K window and row group of O and down
    const int b = c.grp + c.an * K::NGRP;
    const uint32_t vstep = 16u * p.Lmax * 2;
    auto u8 = [](const bf16* q) { return reinterpret_cast<const unsigned char*>(q); };
#pragma unroll 1
    for (int li = 0; li < p.S * NL && this->ok; li++) {
      const int l = li % NL;
      const unsigned char* w1 = u8(p.w1) + (size_t)l * 2560 * D * 2;
      this->template stage<K::RQ, K::RQ * K::KX>(vq, [&](int rt) { return w1 + (size_t)qkv_row<K>(c.j, 16 * (K::RQ * c.r + rt)) * D * 2; });
      const unsigned char* kb = u8(p.kcache) + ((size_t)b * NL + l) * p.Lmax * HD * 2;
      const unsigned char* vb = u8(p.vtcache) + ((size_t)b * NL + l) * HD * p.Lmax * 2;
#pragma unroll 1
      for (int u0 = 0; u0 < c.nun && this->ok; u0 += K::SEGU) {  // a segment: its K pages, then its V^T pages
        const int np = 2 * min(K::SEGU, c.nun - u0);
#pragma unroll 1
        for (int i = 0; i < np; i++) {  // K: key tile this->lw, k-step f; keys past the chunk copy key 0 (masked later)
          if (!this->room()) break;
          int key = c.kbeg + 64 * u0 + 32 * i + 8 * (cr >> 2) + 4 * this->lw + (cr & 3);
          if (key >= c.kend) key = 0;
          const uint32_t d = this->dst();
#pragma unroll
          for (int f = 0; f < 8; f++) dma16(kb + f * 64, (uint32_t)key * (HD * 2) + cq * 16, d + f * 1024);
          this->pg++;
        }
#pragma unroll 1
        for (int i = 0; i < np; i++) {  // V^T: dim tile 8 this->lw + f; an 8-key group that starts in the chunk
          if (!this->room()) break;         // stays within the row (Lmax)
          int kv = c.kbeg + 64 * u0 + 32 * i + 8 * cq;
          if (kv >= c.kend) kv = 0;
          const uint32_t vv = (uint32_t)cr * p.Lmax * 2 + kv * 2;
          const uint32_t d = this->dst();
#pragma unroll
          for (int f = 0; f < 8; f++) dma16(vb + (size_t)(8 * this->lw + f) * vstep, vv, d + f * 1024);
          this->pg++;
        }
      }
      const unsigned char* wo = u8(p.wo) + ((size_t)l * D * QD + (size_t)16 * K::RP * rg * QD + 512 * (K::C * c.j + win)) * 2;
      this->template stage<K::RP, K::RP * K::KO>(vo, [&](int rt) { return wo + (size_t)rt * 16 * QD * 2; });
#pragma unroll 1
      for (int q = 0; q < K::PG; q++) {
        const unsigned char* w2 =
            u8(p.w2) + ((size_t)l * 2 * FF + (size_t)c.j * (2 * FF / K::G) + 16 * (K::RG * c.r + K::RGP * q)) * D * 2;
        this->template stage<K::RGP, K::RGP * K::KX>(vq, [&](int rt) { return w2 + (size_t)rt * 16 * D * 2; });
      }
      const unsigned char* w3 = u8(p.w3) + ((size_t)l * D * FF + (size_t)16 * K::RP * rg * FF + 1024 * (K::C * c.j + win)) * 2;
      this->template stage<K::RP, K::RP * K::KD>(vd, [&](int rt) { return w3 + (size_t)rt * 16 * FF * 2; });
    }
    this->drain();
  }
};

// Workspace offsets of the wave's token rows (tile (n, w)) of a fragment-ordered operand with KT k-steps,
// from k-step ks0; rows past Tv or of an absent sample read zeros.
template <class K>
__device__ __forceinline__ void tok_off(const Params& p, const PCtx& c, uint32_t base, int KT, int ks0, uint32_t (&o)[K::NB]) {
  const int t = 16 * c.wave + c.lr;
#pragma unroll
  for (int n = 0; n < K::NB; n++)
    o[n] = t < p.Tv && n < c.ns ? c.xb + base + (uint32_t)(((n * 4 + c.wave) * KT + ks0) * 1024 + c.lane * 16) : OOB;
}

// ---------------------------------------------------------------- norm stages
// MODE 0: x = embed(x_t). MODE 1: x += gate * sum of the 4 partials. MODE 2: as 1, then the final norm, the
// action projection and the Euler update. The wave norms token t = r + 32 (wave / 2) of every sample
// (LDS slot 2 n + wave / 2); lane holds columns 4 lane + 256 k + i.
template <class K, int MODE>
__device__ __forceinline__ void stage_norm(const Params& p, const PCtx& c, uint32_t part, const float* gate,
                                           const float* scale, const float* shift, float dt) {
  const int t = c.r + 32 * (c.wave >> 1);
  // the modulations do not depend on the wait; the partials of every sample are requested together
  f32x4 sc[4], sh[4], gt[4];
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const int d = 4 * c.lane + 256 * k;
    sc[k] = *reinterpret_cast<const f32x4*>(scale + d);
    sh[k] = *reinterpret_cast<const f32x4*>(shift + d);
    if (MODE != 0) gt[k] = *reinterpret_cast<const f32x4*>(gate + d);
  }
  u32x4 v[K::NB][4][4];
  if (MODE != 0) {
    part_wait<K>(c);
#pragma unroll
    for (int n = 0; n < K::NB; n++)
#pragma unroll
      for (int s = 0; s < 4; s++)
#pragma unroll
        for (int k = 0; k < 4; k++)
          v[n][s][k] = ldb128<kCpSc1>(c.ws, c.part + part + (uint32_t)(((n * TP + t) * D + 4 * c.lane) * 4) + s * (K::PB1 / 4) + k * 1024);
  }
#pragma unroll
  for (int n = 0; n < K::NB; n++) {
    if (n >= c.ns) continue;
    float* xres = reinterpret_cast<float*>(fg_lds + K::L_XRES) + (2 * n + (c.wave >> 1)) * D;
    float* xt = reinterpret_cast<float*>(fg_lds + K::L_XT) + (2 * n + (c.wave >> 1)) * AD;
    f32x4 x[4];
    if (MODE == 0) {
      // coalesced 1 KB reads of W_ain [1024][32]: read j covers rows 8j..8j+7 (lane L: row 8j + L/8,
      // inputs 4 (L%8)..+3), an 8-lane DPP sum finishes each row
      const f32x4 xa = *reinterpret_cast<const f32x4*>(xt + 4 * (c.lane & 7));
      const float* W = p.w_ain + 4 * c.lane;
#pragma unroll 1
      for (int j0 = 0; j0 < D / 8; j0 += 8) {
        f32x4 w[8];
#pragma unroll
        for (int q = 0; q < 8; q++) w[q] = *reinterpret_cast<const f32x4*>(W + (size_t)(j0 + q) * 8 * AD);
#pragma unroll
        for (int q = 0; q < 8; q++) {
          float s = w[q][0] * xa[0] + w[q][1] * xa[1] + w[q][2] * xa[2] + w[q][3] * xa[3];
          s = dpp_f32<0xB1>(s) + s;
          s = dpp_f32<0x4E>(s) + s;
          s = dpp_f32<0x141>(s) + s;
          if ((c.lane & 7) == 0) xres[8 * (j0 + q) + (c.lane >> 3)] = s;
        }
      }
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const int d = 4 * c.lane + 256 * k;
        x[k] = *reinterpret_cast<const f32x4*>(xres + d) + *reinterpret_cast<const f32x4*>(p.b_ain + d);
      }
    } else {
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const f32x4 s = as_f32x4(v[n][0][k]) + as_f32x4(v[n][1][k]) + as_f32x4(v[n][2][k]) + as_f32x4(v[n][3][k]);
        x[k] = *reinterpret_cast<const f32x4*>(xres + 4 * c.lane + 256 * k) + gt[k] * s;
      }
    }
    float ss = 0.f;
#pragma unroll
    for (int k = 0; k < 4; k++) ss += x[k][0] * x[k][0] + x[k][1] * x[k][1] + x[k][2] * x[k][2] + x[k][3] * x[k][3];
    const float rr = rsqrtf(wave_sum(ss) / (float)D + 1e-6f);
    f32x4 h[4];
#pragma unroll
    for (int k = 0; k < 4; k++)
#pragma unroll
      for (int i = 0; i < 4; i++) h[k][i] = x[k][i] * rr * (1.0f + sc[k][i]) + sh[k][i];
    if (MODE != 2) {
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const int d = 4 * c.lane + 256 * k;
        *reinterpret_cast<f32x4*>(xres + d) = x[k];
        // whole 16-byte slots: lanes (2i, 2i + 1) hold columns 8i .. 8i + 7 of this k; the even lane
        // stores the slot for even k, the odd lane for odd k
        const unsigned lo = pack_bf16x2(h[k][0], h[k][1]), hi = pack_bf16x2(h[k][2], h[k][3]);
        const unsigned plo = swap_adj(lo), phi = swap_adj(hi);
        if ((c.lane & 1) == (k & 1))
          *reinterpret_cast<u32x4*>(p.ws + c.xb + K::X_XN + n * (TP * D * 2) + frag_off(32, t, d & ~7)) =
              (c.lane & 1) ? u32x4{plo, phi, lo, hi} : u32x4{lo, hi, plo, phi};
      }
    } else {
#pragma unroll 1
      for (int a0 = 0; a0 < AD; a0 += 4) {
        f32x4 wv[4][4];
#pragma unroll
        for (int a = 0; a < 4; a++)
#pragma unroll
          for (int k = 0; k < 4; k++)
            wv[a][k] = *reinterpret_cast<const f32x4*>(p.w_aout + (a0 + a) * D + 4 * c.lane + 256 * k);
#pragma unroll
        for (int a = 0; a < 4; a++) {
          float s = 0.f;
#pragma unroll
          for (int k = 0; k < 4; k++)
            s += wv[a][k][0] * h[k][0] + wv[a][k][1] * h[k][1] + wv[a][k][2] * h[k][2] + wv[a][k][3] * h[k][3];
          s = wave_sum(s);
          if (c.lane == 0) xt[a0 + a] += dt * (s + p.b_aout[a0 + a]);
        }
      }
    }
  }
}

// ---------------------------------------------------------------- QKV
template <class K>
__device__ __forceinline__ void stage_qkv(const Params& p, const PCtx& c, int li, int l, int pg0, bool last) {
  constexpr int R = K::RQ;
  const int t = 16 * c.wave + c.lr;
  if (16 * c.wave >= p.Tv) {
    page_release<K>(c, pg0 + K::PQ);
    return;
  }
  const bool tv = t < p.Tv;
  wait_norm_rows(c);
  f32x4 acc[K::NB][R];
  uint32_t xo[K::NB];
  tok_off<K>(p, c, K::X_XN, 32, 0, xo);
  gemm<K, R, K::KX, K::NB>(acc, c, pg0, xo);
#pragma unroll
  for (int rt = 0; rt < R; rt++) {
    const int vr0 = 16 * (R * c.r + rt);  // wave-uniform: the tile lies within q, k or v
    if (vr0 >= 256 * K::HX + 256) {       // v dims d..d+3 of token t, transposed
      const int d = vr0 - (256 * K::HX + 256) + 4 * c.lq;
#pragma unroll
      for (int n = 0; n < K::NB; n++) {
        if (!tv || n >= c.ns) continue;
        unsigned short* vs = reinterpret_cast<unsigned short*>(p.ws + c.xb + K::X_VS) + ((li & 1) * K::NB + n) * TP * HD;
        unsigned short* vr =
            reinterpret_cast<unsigned short*>(p.vtcache) +
            (((size_t)(c.grp + n * K::NGRP) * p.NL + l) * HD + d) * p.Lmax + p.Lp + t;
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const unsigned short u = bf16_bits(acc[n][rt][i]);
          vs[(d + i) * TP + t] = u;
          if (last && c.j == l % K::G) vr[(size_t)i * p.Lmax] = u;
        }
      }
      continue;
    }
    const int p0 = (vr0 < 256 * K::HX ? vr0 & 255 : vr0 - 256 * K::HX) / 2 + 2 * c.lq;  // first of two RoPE pairs
    const uint32_t ro = tv ? (uint32_t)(t * 128 + p0) * 4 : OOB;
    const u32x2 cs = ldb64<kCpPlain>(c.rc, ro), sn = ldb64<kCpPlain>(c.rs, ro);
    const float c0 = as_f32(cs[0]), c1 = as_f32(cs[1]), s0 = as_f32(sn[0]), s1 = as_f32(sn[1]);
#pragma unroll
    for (int n = 0; n < K::NB; n++) {
      const f32x4 v = acc[n][rt];
      const unsigned plo = pack_bf16x2(v[0] * c0 - v[1] * s0, v[2] * c1 - v[3] * s1);
      const unsigned phi = pack_bf16x2(v[1] * c0 + v[0] * s0, v[3] * c1 + v[2] * s1);
      if (!tv || n >= c.ns) continue;
      if (vr0 < 256 * K::HX) {
        unsigned char* q = p.ws + c.xb + K::X_Q + (uint32_t)((n * K::HX + (vr0 >> 8)) * TP * HD * 2);
        *reinterpret_cast<unsigned*>(q + frag_off(8, t, p0)) = plo;
        *reinterpret_cast<unsigned*>(q + frag_off(8, t, p0 + 128)) = phi;
      } else {
        unsigned char* k = p.ws + c.xb + K::X_KS + (uint32_t)(((((li & 1) * K::NB + n) * TP + t) * HD + p0) * 2);
        *reinterpret_cast<unsigned*>(k) = plo;
        *reinterpret_cast<unsigned*>(k + 256) = phi;
        if (last && c.j == l % K::G) {  // the caller's caches keep the last step's rows
          bf16* kr = p.kcache + (((size_t)(c.grp + n * K::NGRP) * p.NL + l) * p.Lmax + p.Lp + t) * HD + p0;
          *reinterpret_cast<unsigned*>(kr) = plo;
          *reinterpret_cast<unsigned*>(kr + 128) = phi;
        }
      }
    }
  }
}

// ---------------------------------------------------------------- attention
// Item of rank r: slot an, head ah, prefix keys [kbeg, kend) in segments of up to SEGU 64-key units from
// the ring (a segment's K pages, then its V^T pages), after this step's keys [sbeg, sbeg + nsfx) of the
// XCD's copies, whose loads arrive with q. Wave w: query rows of tokens 16w..16w+15. Per segment: S^T = K Q^T of all
// its keys, one softmax (rescaling what earlier segments left), O^T += V^T P^T of all its keys: the two
// MFMA phases are free of the softmax's serial chain, which a loop over 32-key blocks paid per block
// (ATT 25 us per layer at 16 samples, 14 at 8).
// K rows are permuted inside each 32-key block: row 4a + i of tile kt is key 8a + 4kt + i, so a lane's S^T
// values of tiles (0, 1) are keys 8 lq .. 8 lq + 7, the P^T operand, and V^T fragments are read whole.
template <class K>
__device__ __forceinline__ void stage_att(const Params& p, const PCtx& c, int li, int pgk) {
  constexpr int NT = 4 * K::SEGU;  // key tiles of a segment
  if (16 * c.wave >= p.Tv || c.an >= c.ns) {
    page_release<K>(c, pgk + 4 * c.nun);
    return;
  }
  const int t = 16 * c.wave + c.lr;
  const bool tv = t < p.Tv;
  const float qscale = 1.4426950408889634f / 16.0f;  // log2(e) / sqrt(256)
  const uint32_t pbase = (uint32_t)(c.r * TP + t);
  if (c.nun == 0 && c.nsfx <= 0) {  // empty chunk: weight 0 in the combine
    if (tv && c.lq == 0) *reinterpret_cast<f32x2*>(p.ws + c.xb + K::X_ML + pbase * 8) = f32x2{-1e30f, 0.f};
    return;
  }
  u32x4 qf[8], skf[2][8], sv[16];
  {
    const uint32_t qb = tv ? c.xb + K::X_Q + (uint32_t)((c.an * K::HX + c.ah) * TP * HD * 2) + frag_off(8, t, 8 * c.lq) : OOB;
#pragma unroll
    for (int ks = 0; ks < 8; ks++) qf[ks] = ldb128<kCpSc1>(c.ws, qb + ks * 1024);
    // this step's keys (rows past nsfx: zeros) and the 16-byte groups of their V^T that start below nsfx
    const uint32_t kb = c.xb + K::X_KS + (uint32_t)((((li & 1) * K::NB + c.an) * TP + c.sbeg) * HD * 2);
#pragma unroll
    for (int kt = 0; kt < 2; kt++) {
      const int key = 8 * (c.lr >> 2) + 4 * kt + (c.lr & 3);
      const uint32_t a = key < c.nsfx ? kb + key * (HD * 2) + c.lq * 16 : OOB;
#pragma unroll
      for (int ks = 0; ks < 8; ks++) skf[kt][ks] = ldb128<kCpSc1>(c.ws, a + ks * 64);
    }
    const uint32_t vb = c.xb + K::X_VS + (uint32_t)((((li & 1) * K::NB + c.an) * TP * HD + c.lr * TP + c.sbeg + 8 * c.lq) * 2);
    const uint32_t va = 8 * c.lq < c.nsfx ? vb : OOB;
#pragma unroll
    for (int dt = 0; dt < 16; dt++) sv[dt] = ldb128<kCpSc1>(c.ws, va + dt * (16 * TP * 2));
  }
  // S^T of one key tile
  auto score = [&](const u32x4 (&kf)[8]) __attribute__((always_inline)) {
    f32x4 a = {0.f, 0.f, 0.f, 0.f}, b = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < 8; ks += 2) {
      a = mfma16(kf[ks], qf[ks], a);
      b = mfma16(kf[ks + 1], qf[ks + 1], b);
    }
    return a + b;
  };
  // keys 8 lq + 4 kt + i >= nv of a 32-key block: S = -inf, V = 0
  auto smask = [&](f32x4& s, int kt, int nv) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; i++)
      if (8 * c.lq + 4 * kt + i >= nv) s[i] = -1e30f;
  };
  auto vmask = [&](u32x4& v, int nv) __attribute__((always_inline)) {
    const int q = min(max(nv - 8 * c.lq, 0), 8);
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] &= q >= 2 * e + 2 ? 0xffffffffu : (q == 2 * e + 1 ? 0xffffu : 0u);
  };
  auto pack_p = [&](const f32x4& a, const f32x4& b) __attribute__((always_inline)) {
    return u32x4{pack_bf16x2(a[0], a[1]), pack_bf16x2(a[2], a[3]), pack_bf16x2(b[0], b[1]), pack_bf16x2(b[2], b[3])};
  };
  float m = -1e30f, lsum = 0.f;
  f32x4 o[16];
  // softmax of N key tiles (pairs = 32-key blocks) against the running (m, l) -> P^T operands; returns the
  // factor of what came before
  auto softmax = [&](auto& x, auto& pb) __attribute__((always_inline)) {
    constexpr int N = sizeof(x) / sizeof(f32x4);
    float bm = -1e30f;
#pragma unroll
    for (int q = 0; q < N; q++) bm = fmaxf(bm, fmaxf(fmaxf(x[q][0], x[q][1]), fmaxf(x[q][2], x[q][3])));
    const float mnew = fmaxf(m, cols_max(bm) * qscale);
    const float alpha = exp2_w(m - mnew);
    m = mnew;
    float ps = 0.f;
#pragma unroll
    for (int q = 0; q < N; q += 2) {
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          x[q + h][i] = exp2_w(fmaf(x[q + h][i], qscale, -m));
          ps += x[q + h][i];
        }
      pb[q / 2] = pack_p(x[q], x[q + 1]);
    }
    lsum = lsum * alpha + cols_sum(ps);
    return alpha;
  };
  {
    f32x4 s[2];
    u32x4 pb[1];
#pragma unroll
    for (int kt = 0; kt < 2; kt++) {
      s[kt] = score(skf[kt]);
      smask(s[kt], kt, c.nsfx);
    }
    if (c.nsfx > 0) softmax(s, pb);
    else pb[0] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
    for (int dt = 0; dt < 16; dt++) {
      vmask(sv[dt], c.nsfx);
      o[dt] = mfma16(sv[dt], pb[0], f32x4{0.f, 0.f, 0.f, 0.f});
    }
  }
#pragma unroll 1
  for (int u0 = 0; u0 < c.nun; u0 += K::SEGU) {
    const int nu = min(K::SEGU, c.nun - u0);       // units of this segment
    const int nv0 = c.kend - (c.kbeg + 64 * u0);    // its valid keys
    const int pk = pgk + 4 * u0, pv = pk + 2 * nu;  // its K and V^T pages
    f32x4 s[NT];
#pragma unroll
    for (int u = 0; u < K::SEGU; u++) {
#pragma unroll
      for (int q = 0; q < 4; q++) s[4 * u + q] = f32x4{-1e30f, -1e30f, -1e30f, -1e30f};
      if (u >= nu) continue;
      page_wait<K>(c, pk + 2 * u + 1);
      u32x4 kf[2][8];
      auto rd = [&](int q) {
        const uint32_t a = ((pk + 2 * u + (q >> 1)) % RING) * PAGE + frag_slot(c.lr, c.lq) + (q & 1) * 8192;
#pragma unroll
        for (int ks = 0; ks < 8; ks++) kf[q & 1][ks] = *reinterpret_cast<const u32x4*>(fg_lds + a + ks * 1024);
      };
      rd(0);
#pragma unroll
      for (int q = 0; q < 4; q++) {
        if (q + 1 < 4) rd(q + 1);
        __builtin_amdgcn_sched_barrier(0);
        s[4 * u + q] = score(kf[q & 1]);
        __builtin_amdgcn_sched_barrier(0);
      }
      page_release<K>(c, pk + 2 * u + 2);
      if (u == nu - 1 && nv0 < 64 * nu) {
#pragma unroll
        for (int q = 0; q < 4; q++) smask(s[4 * u + q], q & 1, nv0 - 64 * u - 32 * (q >> 1));
      }
    }
    u32x4 pb[NT / 2];
    const float alpha = softmax(s, pb);
#pragma unroll
    for (int dt = 0; dt < 16; dt++) o[dt] *= alpha;
#pragma unroll
    for (int u = 0; u < K::SEGU; u++) {
      if (u >= nu) continue;
      page_wait<K>(c, pv + 2 * u + 1);
      u32x4 vf[2][8];
      auto rd = [&](int q) {  // half q & 1 of the dims of block q / 2
        const uint32_t a = ((pv + 2 * u + (q >> 1)) % RING) * PAGE + frag_slot(c.lr, c.lq) + (q & 1) * 8192;
#pragma unroll
        for (int d8 = 0; d8 < 8; d8++) vf[q & 1][d8] = *reinterpret_cast<const u32x4*>(fg_lds + a + d8 * 1024);
      };
      const bool part = u == nu - 1 && nv0 < 64 * nu;
      rd(0);
#pragma unroll
      for (int q = 0; q < 4; q++) {
        if (q + 1 < 4) rd(q + 1);
        __builtin_amdgcn_sched_barrier(0);
        if (part) {
#pragma unroll
          for (int d8 = 0; d8 < 8; d8++) vmask(vf[q & 1][d8], nv0 - 64 * u - 32 * (q >> 1));
        }
#pragma unroll
        for (int d8 = 0; d8 < 8; d8++)
          o[8 * (q & 1) + d8] = mfma16(vf[q & 1][d8], pb[2 * u + (q >> 1)], o[8 * (q & 1) + d8]);
        __builtin_amdgcn_sched_barrier(0);
      }
      page_release<K>(c, pv + 2 * u + 2);
    }
  }
  // O^T / l in the O projection's operand order, whole 16-byte slots (see pi05_bs1.hip)
  const float inv = lsum > 0.f ? 1.0f / lsum : 0.f;
  const bool odd = c.lq & 1;
  const uint32_t ob = c.xb + K::X_ATTP + (uint32_t)((c.r * 4 + c.wave) * 8192 + (((c.lq >> 1) + 2 * (c.lq & 1)) * 16 + c.lr) * 16);
#pragma unroll
  for (int ks = 0; ks < 8; ks++) {
    const unsigned a0 = pack_bf16x2(o[2 * ks][0] * inv, o[2 * ks][1] * inv);
    const unsigned a1 = pack_bf16x2(o[2 * ks][2] * inv, o[2 * ks][3] * inv);
    const unsigned b0 = pack_bf16x2(o[2 * ks + 1][0] * inv, o[2 * ks + 1][1] * inv);
    const unsigned b1 = pack_bf16x2(o[2 * ks + 1][2] * inv, o[2 * ks + 1][3] * inv);
    const LanePair s0 = swap16(a0, b0), s1 = swap16(a1, b1);
    if (tv)  // rows past Tv are never read
      *reinterpret_cast<u32x4*>(p.ws + ob + ks * 1024) = odd ? u32x4{s0.lo, s1.lo, b0, b1} : u32x4{a0, a1, s0.hi, s1.hi};
  }
  if (tv && c.lq == 0) *reinterpret_cast<f32x2*>(p.ws + c.xb + K::X_ML + pbase * 8) = f32x2{m, lsum};
}

// ---------------------------------------------------------------- combine
// Fragment id = (slot, head, k-step) of token tile w: wave w of rank r takes ids FPR r .. + FPR - 1 (with
// G = 4: id r of ranks < 16). A lane owns one 16-byte slot (token 16 w + lane % 16, 8 dims).
template <class K>
__device__ __forceinline__ void stage_comb(const Params& p, const PCtx& c) {
  constexpr int NF = K::FPR > 0 ? K::FPR : 1;
  const int id0 = c.r * NF;
  if (16 * c.wave >= p.Tv || id0 >= K::NB * K::HX * 8) return;
  const int nh = id0 >> 3, n = nh / K::HX;  // a rank's ids share their (slot, head)
  if (n >= c.ns) return;
  xcd_wait(c, (K::NKC == 32 ? 0xffffffffu : ((1u << (K::NKC & 31)) - 1u)) << (nh * K::NKC));
  const int t = 16 * c.wave + c.lr;
  const bool tv = t < p.Tv;
  u32x2 ml[K::NKC];
  u32x4 v[NF][K::NKC];
#pragma unroll
  for (int k = 0; k < K::NKC; k++) {
    const int rr = nh * K::NKC + k;
    ml[k] = ldb64<kCpSc1>(c.ws, tv ? c.xb + K::X_ML + (uint32_t)(rr * TP + t) * 8 : OOB);
#pragma unroll
    for (int f = 0; f < NF; f++)
      v[f][k] = ldb128<kCpSc1>(c.ws, tv ? c.xb + K::X_ATTP + (uint32_t)((rr * 4 + c.wave) * 8192 + ((id0 + f) & 7) * 1024 + c.lane * 16) : OOB);
  }
  __builtin_amdgcn_sched_barrier(0);
  float M = -1e30f;
#pragma unroll
  for (int k = 0; k < K::NKC; k++) M = fmaxf(M, as_f32(ml[k][0]));
  float wt[K::NKC], L = 0.f;
#pragma unroll
  for (int k = 0; k < K::NKC; k++) {
    wt[k] = as_f32(ml[k][1]) * exp2_w(as_f32(ml[k][0]) - M);
    L += wt[k];
  }
  const float inv = L > 0.f ? 1.0f / L : 0.f;
#pragma unroll
  for (int f = 0; f < NF; f++) {
    float u[8];
#pragma unroll
    for (int e = 0; e < 8; e++) u[e] = 0.f;
#pragma unroll
    for (int k = 0; k < K::NKC; k++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const unsigned d = wt[k] != 0.f ? v[f][k][e] : 0u;  // empty chunks hold no partial
        u[2 * e] = fmaf(wt[k], bf_lo(d), u[2 * e]);
        u[2 * e + 1] = fmaf(wt[k], bf_hi(d), u[2 * e + 1]);
      }
    u32x4 out;
#pragma unroll
    for (int e = 0; e < 4; e++) out[e] = pack_bf16x2(u[2 * e] * inv, u[2 * e + 1] * inv);
    const int ks = (nh % K::HX) * 8 + ((id0 + f) & 7);
    *reinterpret_cast<u32x4*>(p.ws + c.xb + K::X_ATTN + (uint32_t)(((n * 4 + c.wave) * 8 * K::HX + ks) * 1024 + c.lane * 16)) = out;
  }
}

// Stores the fp32 partial sums of the rank's rows (row group rg, window index wd of the group).
template <class K>
__device__ __forceinline__ void store_part(const Params& p, const PCtx& c, uint32_t part, int wd, int rg,
                                           const f32x4 (&acc)[K::NB][K::RP]) {
  const int t = 16 * c.wave + c.lr;
  if (t >= p.Tv) return;
#pragma unroll
  for (int n = 0; n < K::NB; n++) {
    if (n >= c.ns) continue;
#pragma unroll
    for (int rt = 0; rt < K::RP; rt++)
      stb128<kCpPart<K>>(c.ws, c.part + part + wd * (K::PB1 / 4) +
                                  (uint32_t)(((n * TP + t) * D + 16 * (K::RP * rg + rt) + 4 * c.lq) * 4),
                         as_u32x4(acc[n][rt]));
  }
}

// Ranks whose combine wrote K window `win` (heads 2 win, 2 win + 1) of the attention output.
template <class K>
__device__ __forceinline__ uint32_t comb_ranks(int win) {
  if constexpr (K::FPR == 0) return 0xffffu;
  constexpr int NF = K::FPR > 0 ? K::FPR : 1, W = 16 / NF;  // ranks per window and slot
  uint32_t m = 0;
#pragma unroll
  for (int n = 0; n < K::NB; n++) m |= ((W >= 32 ? 0u : 1u << W) - 1u) << ((n * K::HX * 8 + 16 * win) / NF);
  return m;
}

template <class K>
__device__ __forceinline__ void stage_oproj(const Params& p, const PCtx& c, int pg0) {
  if (16 * c.wave >= p.Tv) {
    page_release<K>(c, pg0 + K::PO);
    return;
  }
  const int win = c.r / (NR / K::C), rg = c.r % (NR / K::C);
  xcd_wait(c, comb_ranks<K>(win));
  f32x4 acc[K::NB][K::RP];
  uint32_t xo[K::NB];
  tok_off<K>(p, c, K::X_ATTN, 8 * K::HX, 16 * win, xo);
  gemm<K, K::RP, K::KO, K::NB>(acc, c, pg0, xo);
  store_part<K>(p, c, 0, K::C * c.j + win, rg, acc);
}

template <class K>
__device__ __forceinline__ void stage_gu(const Params& p, const PCtx& c, int pg0) {
  if (16 * c.wave >= p.Tv) {
    page_release<K>(c, pg0 + K::PGU);
    return;
  }
  wait_norm_rows(c);
  uint32_t xo[K::NB];
  tok_off<K>(p, c, K::X_XN, 32, 0, xo);
#pragma unroll 1
  for (int q = 0; q < K::PG; q++) {
    f32x4 acc[K::NB][K::RGP];
    // operand offsets are derived in each pass (hoisted out of the loop they spilled)
#pragma unroll
    for (int n = 0; n < K::NB; n++) asm volatile("" : "+v"(xo[n]));
    gemm<K, K::RGP, K::KX, K::NB>(acc, c, pg0 + q * (K::PGU / K::PG), xo);
    int t = 16 * c.wave + c.lr;
    asm volatile("" : "+v"(t));  // the store addresses are derived here, not kept live over the GEMM
    if (t >= p.Tv) continue;
    // rows 2f, 2f + 1 = gate f, up f: the lane's columns f = 8 (row tile) + 2 lq + (0, 1) of the rank's slice.
    // One exchange with lane ^ 16 per pair of row tiles gives a lane 4 consecutive columns (8 bytes).
#pragma unroll
    for (int n = 0; n < K::NB; n++) {
      if (n >= c.ns) continue;
#pragma unroll
      for (int rt = 0; rt < K::RGP; rt += 2) {
        const f32x4 a = acc[n][rt], b = acc[n][rt + 1];
        const unsigned p0 = pack_bf16x2(gelu_tanh(a[0]) * a[1], gelu_tanh(a[2]) * a[3]);
        const unsigned p1 = pack_bf16x2(gelu_tanh(b[0]) * b[1], gelu_tanh(b[2]) * b[3]);
        const bool odd = c.lq & 1;
        const LanePair sw = swap16(p0, p1);
        const unsigned recv = odd ? sw.lo : sw.hi;
        const int f = 8 * (K::RG * c.r + K::RGP * q + rt) + (odd ? 8 + 2 * (c.lq - 1) : 2 * c.lq);
        *reinterpret_cast<u32x2*>(p.ws + c.xb + K::X_H + n * (TP * (FF / K::G) * 2) + frag_off(128 / K::G, t, f)) =
            odd ? u32x2{recv, p1} : u32x2{p0, recv};
      }
    }
  }
}

template <class K>
__device__ __forceinline__ void stage_dn(const Params& p, const PCtx& c, int pg0) {
  if (16 * c.wave >= p.Tv) {
    page_release<K>(c, pg0 + K::PD);
    return;
  }
  const int win = c.r / (NR / K::C), rg = c.r % (NR / K::C);
  constexpr int GW = 8 * K::G;  // gate/up ranks per 1024-column window
  xcd_wait(c, GW == 32 ? 0xffffffffu : ((1u << (GW & 31)) - 1u) << (GW * win));
  f32x4 acc[K::NB][K::RP];
  uint32_t xo[K::NB];
  tok_off<K>(p, c, K::X_H, 128 / K::G, 32 * win, xo);
  gemm<K, K::RP, K::KD, K::NB>(acc, c, pg0, xo);
  store_part<K>(p, c, K::PB - K::PB1, K::C * c.j + win, rg, acc);
}

// ---------------------------------------------------------------- instrumentation
__device__ __forceinline__ void mark(const Params& p, const PCtx& c, int idx, uint64_t& t0) {
  if (p.stage_cycles && blockIdx.x == 0 && c.wave == 0 && c.lane == 0) {
    const uint64_t now = __builtin_amdgcn_s_memrealtime();
    p.stage_cycles[idx] += now - t0;  // 0-7 stages N1 QKV ATT COMB O N2 GU DN, 8 final, 9 XCD barrier and signals
    t0 = now;
  }
}

// ---------------------------------------------------------------- kernel
template <int G, int NB>
__global__ void __launch_bounds__(NTH, 1) pi05_group_kernel(Params p) {
  using K = Cfg<G, NB>;
  PCtx c;
  const int tid = threadIdx.x;
  c.x = blockIdx.x & 7;
  c.grp = c.x / G;
  c.j = c.x % G;
  c.ns = min(NB, (p.B - c.grp + K::NGRP - 1) / K::NGRP);
  if (p.B <= c.grp) return;  // no sample for this group: the whole workgroup
  c.lane = tid & 63;
  c.wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  c.lr = c.lane & 15;
  c.lq = c.lane >> 4;
  c.r = blockIdx.x >> 3;
  c.ws = make_rsrc(p.ws, K::WS);
  c.wsp = p.ws;
  c.rc = make_rsrc(p.rope_cos, (uint32_t)(p.Tv * 128 * 4));
  c.rs = make_rsrc(p.rope_sin, (uint32_t)(p.Tv * 128 * 4));
  c.xb = K::OFF_XCD + (uint32_t)c.x * K::XB;
  c.part = K::OFF_PART + (uint32_t)c.grp * K::PB;
  c.lds_addr = (uint32_t)(uintptr_t)fg_lds;
  c.err = reinterpret_cast<unsigned*>(p.ws + OFF_CTRL + 8);
  {
    c.an = c.r / (K::HX * K::NKC);
    c.ah = (c.r / K::NKC) % K::HX;
    const int kc = c.r % K::NKC, chunk = 64 * ((p.Lp + 64 * K::NKC - 1) / (64 * K::NKC));
    c.kbeg = min(kc * chunk, p.Lp);
    c.kend = min(c.kbeg + chunk, p.Lp);
    c.nun = c.an < c.ns ? (c.kend - c.kbeg + 63) / 64 : 0;
    c.sbeg = kc * K::SK;
    c.nsfx = min(p.Tv - c.sbeg, K::SK);
  }
  if (tid < 16) ctl_st<K>(tid, 0u);
  if (tid == 0 && xcc_id() != (unsigned)c.x) atomicOr(c.err, kErrXcd);
  const uint64_t seq = ld_flag(reinterpret_cast<const uint64_t*>(p.ws + OFF_CTRL));
  __syncthreads();  // the only workgroup barrier: LDS control words are initialised
  if (c.wave >= NCW) {
    Loader<K> L(p, c, c.wave - NCW);
    L.run();
    return;
  }
  c.e = c.eg = seq << 32;
  const int NL = p.NL;
  const int t = c.r + 32 * (c.wave >> 1);
  const bool nw = (c.wave & 1) == (c.r >> 4) && t < p.Tv;  // this wave owns a token in the norm stages
  if (nw && c.lane < AD)
    for (int n = 0; n < c.ns; n++)
      reinterpret_cast<float*>(fg_lds + K::L_XT)[(2 * n + (c.wave >> 1)) * AD + c.lane] =
          p.x_t[((size_t)(c.grp + n * K::NGRP) * p.xt_rows + t) * AD + c.lane];
  const float dt = -1.0f / (float)p.S;
  const int ppl = K::PQ + 4 * c.nun + K::PO + K::PGU + K::PD;
  int pb = 0;  // first ring page of the layer
  uint64_t t0 = __builtin_amdgcn_s_memrealtime();
#pragma unroll 1
  for (int step = 0; step < p.S; step++) {
#pragma unroll 1
    for (int l = 0; l < NL; l++, pb += ppl) {
      launder(c);
      const int li = step * NL + l;
      const float* mod_in = p.mods + ((size_t)li * 2 + 0) * 3 * D;
      const float* mod_post = p.mods + ((size_t)li * 2 + 1) * 3 * D;
      if (nw) {
        if (l == 0)
          stage_norm<K, 0>(p, c, 0, nullptr, mod_in, mod_in + D, 0.f);
        else
          stage_norm<K, 1>(p, c, K::PB - K::PB1, mod_post - 6 * D + 2 * D, mod_in, mod_in + D, 0.f);
      }
      mark(p, c, 0, t0);
      xcd_signal(c);
      launder(c);
      mark(p, c, 9, t0);
      stage_qkv<K>(p, c, li, l, pb, step == p.S - 1);
      mark(p, c, 1, t0);
      xcd_sync(c);
      launder(c);
      mark(p, c, 9, t0);
      stage_att<K>(p, c, li, pb + K::PQ);
      mark(p, c, 2, t0);
      xcd_signal(c);
      launder(c);
      mark(p, c, 9, t0);
      stage_comb<K>(p, c);
      mark(p, c, 3, t0);
      xcd_signal(c);
      launder(c);
      mark(p, c, 9, t0);
      stage_oproj<K>(p, c, pb + K::PQ + 4 * c.nun);
      mark(p, c, 4, t0);
      part_signal<K>(c);
      launder(c);
      mark(p, c, 9, t0);
      if (nw) stage_norm<K, 1>(p, c, 0, mod_in + 2 * D, mod_post, mod_post + D, 0.f);
      mark(p, c, 5, t0);
      xcd_signal(c);
      launder(c);
      mark(p, c, 9, t0);
      stage_gu<K>(p, c, pb + K::PQ + 4 * c.nun + K::PO);
      mark(p, c, 6, t0);
      xcd_signal(c);
      launder(c);
      mark(p, c, 9, t0);
      stage_dn<K>(p, c, pb + K::PQ + 4 * c.nun + K::PO + K::PGU);
      mark(p, c, 7, t0);
      part_signal<K>(c);
    }
    if (nw) {
      const int li = step * NL + NL - 1;
      const float* gl = p.mods + ((size_t)li * 2 + 1) * 3 * D + 2 * D;
      const float* mf = p.mod_final + (size_t)step * 3 * D;
      stage_norm<K, 2>(p, c, K::PB - K::PB1, gl, mf, mf + D, dt);
    }
    mark(p, c, 8, t0);
  }
  if (c.j == 0 && nw && c.lane < AD)
    for (int n = 0; n < c.ns; n++)
      p.x_t[((size_t)(c.grp + n * K::NGRP) * p.xt_rows + t) * AD + c.lane] =
          reinterpret_cast<float*>(fg_lds + K::L_XT)[(2 * n + (c.wave >> 1)) * AD + c.lane];
  if (c.j == 0 && c.r == 0 && c.wave == 0 && c.lane == 0) finish_group(p.ws, seq, (unsigned)min(p.B, K::NGRP), kOwnerPi05Group);
}

struct Choice {
  const void* kernel;
  unsigned lds;
  size_t ws;
};
template <int G, int NB>
Choice choice() {
  return {(const void*)pi05_group_kernel<G, NB>, Cfg<G, NB>::LDS, Cfg<G, NB>::WS};
}
// Wider groups stream fewer weights per XCD but exchange partial sums between XCDs. Two samples per group
// share every weight fragment. ms per launch (Lp = 968, Tv = 50, 10 steps), against the stage engine's, all before
// the copies of copy_row, with which the shapes taken run 5.7, 7.8, 10.3 and 15.9:
//   batch 2   (4, 1) 6.2, (4, 2) 7.1               stage engine 16.7
//   batch 4   (4, 2) 8.4, (2, 1) 8.4 (Tv = 10: 6.0 against 6.4)      17.0
//   batch 8   (2, 2) 11.2, (1, 1) 12.8                               17.4
//   batch 16  (1, 2) 16.9, (2, 4) 17.6                               18.9
// Past 16 samples an XCD would hold more than two, whose tokens fill the stage engine's tiles.
Choice pick(int batch) {
  if (batch <= 2) return choice<4, 1>();
  if (batch <= 4) return choice<4, 2>();
  if (batch <= 8) return choice<2, 2>();
  return choice<1, 2>();
}

}  // namespace pg

// ---------------------------------------------------------------- host
bool pi05_group_eligible(int batch, int Tv) { return batch >= 2 && batch <= 16 && Tv >= 1 && Tv <= pg::TP; }
size_t pi05_group_workspace_bytes(int batch) { return pg::pick(batch).ws; }

// From 9 samples on a rank copies half of the prefix K and V of its (sample, head) by itself, so each key
// comes eight times, once per head: 1.8 us per layer and 128 keys. The stage engine's items hold a sample's
// 128 keys with up to 256 query rows of all heads and go out in rounds of 256. us per layer of both, fitted to
// 2048 <= Lp <= 8100, Tv 1 to 64, 9 to 16 samples. Groups against the stage engine, ms per step of 18 layers:
//   9 samples, Tv = 10   Lp 2048 1.48, 1.68   3072 1.73, 1.74   4096 1.99, 1.93   8100 2.99, 2.25
//  12 samples, Tv = 10   Lp 3072 1.74, 1.88   4096 2.01, 1.92   8100 3.00, 2.27
//  12 samples, Tv = 50   Lp 4096 2.27, 2.80                     8100 3.21, 3.85
// The rule lies within 5 % of the faster one everywhere. With up to 8 samples the groups stay ahead to the longest
// prefix (8 samples, Lp = 8100, Tv = 10: 1.65, 2.10).
bool pi05_group_faster(int batch, int Tv, int Lp) {
  if (batch <= 8) return true;
  auto up = [](int a, int b) { return (a + b - 1) / b; };
  const int rounds = up(batch * up(Lp + Tv, 128) * up(8 * Tv, 256), 256);
  const float stage = 82.f + 9.2f * rounds + 1.33e-5f * batch * (Lp + Tv) * Tv;
  return 52.f + 0.36f * Tv + 1.79f * up(Lp, 128) <= stage;
}

int pi05_denoise_group(const fa_pi05_args* a, fa_stream_t stream) {
  using namespace fa::pg;
  const Choice k = pick(a->batch);
  int rc = host::check_device(k.kernel, NTH, k.lds, NWG, "fa_pi05_denoise");
  if (rc != FA_OK) return rc;
  Params p;
  p.w1 = static_cast<const bf16*>(a->w1);
  p.wo = static_cast<const bf16*>(a->wo);
  p.w2 = static_cast<const bf16*>(a->w2);
  p.w3 = static_cast<const bf16*>(a->w3);
  p.mods = a->mods;
  p.mod_final = a->mod_final;
  p.rope_cos = a->rope_cos;
  p.rope_sin = a->rope_sin;
  p.w_ain = a->w_ain;
  p.b_ain = a->b_ain;
  p.w_aout = a->w_aout;
  p.b_aout = a->b_aout;
  p.kcache = static_cast<bf16*>(a->kcache);
  p.vtcache = static_cast<bf16*>(a->vtcache);
  p.x_t = a->x_t;
  p.stage_cycles = a->stage_cycles;
  p.ws = static_cast<unsigned char*>(a->workspace);
  p.NL = a->num_layers;
  p.Lp = a->Lp;
  p.Lmax = a->Lmax;
  p.S = a->num_steps;
  p.Tv = a->Tv;
  p.B = a->batch;
  p.xt_rows = a->xt_rows;
  if (a->srows > 0 && (rc = pi05_kv_handoff(a, stream)) != FA_OK) return rc;
  void* args[] = {&p};
  return host::coop_launch(k.kernel, NWG, NTH, args, k.lds, stream, "fa_pi05_denoise (batched)");
}

}  // namespace fa
