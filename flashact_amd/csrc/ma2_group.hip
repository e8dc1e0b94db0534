// MolmoAct2 flow loop for up to 16 samples (and single samples that the batch-1 kernel does not take):
// groups of XCDs, each running its own samples through the whole S-step loop with no grid-wide barrier,
// laid out like pi05_group.hip (group.h). ONE cooperative launch of 256 workgroups of 6 waves.
//
// G XCDs form a group (G = 4: 2 groups, G = 2: 4, G = 1: 8) of up to NB samples. XCD j of a group owns
// attention heads [8/G j, ..), MLP columns [3072/G j, ..) and those K windows of the three output
// projections, which are also split over C = 4/G K windows inside the XCD, so every residual update sums 4
// fp32 partials. A sample's tokens are TT tiles of 16 (TT = 2 up to Tv = 32, else 4). Compute wave w owns
// tile w % 2 of samples w / 2, w / 2 + 2, .. with TT = 2, tile w of every sample with TT = 4.
//
// Per layer ([W] = waits for the waves that wrote the operand, [X] = XCD barrier, {E} = waits for the
// group's partial sums):
//   N_msa  x += g_mlp (sum of the 4 down partials + b_dn) (layer 0: x = embed(x_t)); xn = adaRMS(x)
//   [W] QKV   q, k, v rows of the XCD's heads + bias, fp32, in the order the attention loads them
//   [X] SATT  (sample, head) per rank: per-head RMS, RoPE, softmax(q k^T) v over the action tokens
//   [W] SO {E} N_mca [W] CQ (rows of the XCD's heads)
//   [W] CATT  (sample, head, key chunk) per rank: 32-key context blocks from the ring
//   [W] COMB  key chunks combined
//   [W] CO {E} N_mlp [W] GU [W] DN {E}
// The stage engine (ma2.hip) runs these stages behind 12 grid barriers of about 2.2 us per layer, with 60
// to 240 tiles for 256 CUs. What bounds this kernel is the chain of its stages; a layer's weights (21.2 MB,
// 21.2/G per XCD) stream at 0.85-0.95 TB/s per XCD underneath it.
#include "group.h"
#include "ma2_attn.h"
#include "../../include/flashact_mi355x.h"
#include "fa_host.h"

namespace fa {
namespace mg {
using namespace fa::grp;
using fa::ma2att::frag_pos;
using fa::ma2att::keep_mask;
using fa::ma2att::kperm_row;
using fa::ma2att::pack4;
using fa::ma2att::rms96;

constexpr int D = 768, HD = 96, FF = 3072, AD = 32;
constexpr int KX = D / 32, KO = 6, KD = 24;  // k-steps: full rows, O windows (192), down windows (768)
constexpr int SB = 4;                        // 32-key context blocks per softmax segment

template <int G_, int TT_, int NB_>
struct Cfg {
  static constexpr int G = G_, TT = TT_, NB = NB_, NI = NB * TT / 4;  // token tiles per sample, per wave
  static constexpr int RING = TT == 2 ? 7 : 6;
  static constexpr int NGRP = NX / G, HX = 8 / G, C = 4 / G;
  static constexpr int NKC = NR / (NB * HX);          // context chunks per (sample, head): ranks
  static constexpr int NP = TT == 2 ? 2 : 1;          // waves that share a token tile's context blocks
  static constexpr int NCH = NKC * NP;                // context partials per (sample, head, tile)
  static constexpr int NT = NB * TT;                  // token tiles
  static constexpr int TQ = 18 * HX, RQ = G == 1 ? 5 : (G == 2 ? 3 : 2), NRQ = (TQ + RQ - 1) / RQ;  // QKV
  static constexpr int TC = 6 * HX, RC = G == 1 ? 2 : 1, NRC = TC / RC;                            // CQ
  static constexpr int RP = G == 1 ? 6 : (G == 2 ? 3 : 2), NRG = 48 / RP;  // output projections: C windows of NRG ranks
  static constexpr int RG = 12 / G, PG = G == 1 ? 2 : 1, RGP = RG / PG;    // gate/up
  static constexpr int pages(int frags) { return (frags + 15) / 16; }
  static constexpr int PQ = pages(RQ * KX), PO = pages(RP * KO), PC = pages(RC * KX), PGU = PG * pages(RGP * KX),
                       PD = pages(RP * KD);
  static_assert(NRQ <= NR && NRC <= NR && NRG * C <= NR && NB * HX * NKC == NR, "ranks");
  // workspace of one XCD (bytes)
  static constexpr uint32_t X_XN = 0;                              // [tile][24 k-steps][1 KB]
  static constexpr uint32_t X_QKV = X_XN + NT * KX * 1024;         // [tile][head][18 slots][64 lanes] f32x4
  static constexpr uint32_t X_ATT = X_QKV + NT * HX * 18 * 1024;   // [tile][3 HX k-steps][1 KB]
  static constexpr uint32_t X_QC = X_ATT + NT * HX * 3 * 1024;     // [tile][head][6 slots][64 lanes] f32x4
  static constexpr uint32_t X_CP = X_QC + NT * HX * 6 * 1024;      // [rank][wave][NI][3][1 KB] bf16 partials
  static constexpr uint32_t X_CML = X_CP + NR * NCW * NI * 3072;   // [rank][wave][NI][16] (m, l)
  static constexpr uint32_t X_H = X_CML + NR * NCW * NI * 128;     // [tile][96 / G k-steps][1 KB]
  static constexpr uint32_t XB = X_H + NT * (96 / G) * 1024;
  static constexpr uint32_t OFF_XCD = kWsDataBase;
  // fp32 partial sums [4 windows][tokens][768]; exchange e uses buffer e % 2 (one buffer with G = 1, where an
  // exchange's producers run after every reader of the one before)
  static constexpr uint32_t PB1 = 4u * NT * 16 * D * 4, NBUF = G == 1 ? 1 : 2;
  static constexpr uint32_t OFF_PART = OFF_XCD + NX * XB;
  static constexpr uint32_t WS = OFF_PART + NGRP * NBUF * PB1;
  // LDS (bytes)
  static constexpr uint32_t L_CTL = RING * PAGE;                   // ready[2], consumed[4], abort, -, SATT done [4]
  static constexpr uint32_t L_SATT = L_CTL + 64;                   // Q | K | V^T fragments of the self attention
  static constexpr uint32_t L_CQ = L_SATT + TT * 9 * 1024;         // [wave][3][1 KB] query fragments
  static constexpr int NS = 2 * NI;                                // residual rows per rank
  static constexpr uint32_t L_XRES = L_CQ + NCW * 3072;            // f32 [NS][768]
  static constexpr uint32_t L_XT = L_XRES + NS * D * 4;            // f32 [NS][32]
  static constexpr uint32_t LDS = L_XT + NS * AD * 4;
  static_assert(LDS <= 160 * 1024, "LDS of one CU");
};

struct Params {
  const bf16 *w_qkv, *w_so, *w_cq, *w_co, *w_gu, *w_dn;
  const float *b_qkv, *b_so, *b_cq, *b_co, *b_gu, *b_dn;
  const float *mods, *mod_final, *rope_cos, *rope_sin, *w_ain, *b_ain;
  const bf16* w_aout;
  const float* b_aout;
  const bf16* kctx;   // [B][NL][Lkmax][768]
  const bf16* vtctx;  // [B][NL][768][Lkmax]
  float* x_t;         // [B][xt_rows][32]
  unsigned long long* stage_cycles;
  unsigned char* ws;
  int NL, Lk, Lkmax, Tv, adim, S, B, xt_rows;
};

struct MCtx : Ctx {
  int an, ah, kbeg, kend, nblk;  // context item: sample slot, head, keys, 32-key blocks
};

// Byte offset of (token t of its tile, column k) inside a tile of a fragment-ordered operand.
__device__ __forceinline__ uint32_t tfrag(int t, int k) {
  return (uint32_t)((((k >> 5) * 4 + ((k >> 3) & 3)) * 16 + (t & 15)) * 16 + (k & 7) * 2);
}
// The wave's i-th token tile: sample slot, tile of the sample, index among all.
template <class K>
__device__ __forceinline__ int slot_of(const Ctx& c, int i) { return K::TT == 2 ? (c.wave >> 1) + 2 * i : i; }
template <class K>
__device__ __forceinline__ int tile_of(const Ctx& c) { return K::TT == 2 ? c.wave & 1 : c.wave; }
template <class K>
__device__ __forceinline__ int tidx(const Ctx& c, int i) { return slot_of<K>(c, i) * K::TT + tile_of<K>(c); }
// A wave with no token below Tv in its tile, or with no sample, has nothing to compute.
template <class K>
__device__ __forceinline__ bool idle(const Params& p, const Ctx& c) {
  return 16 * tile_of<K>(c) >= p.Tv || (K::TT == 2 && (c.wave >> 1) >= c.ns);
}
// Token t of a sample is normed by rank t % 32 on a wave that owns its tile.
template <class K>
__device__ __forceinline__ void wait_norm_rows(const Ctx& c) { xcd_wait(c, c.wave & 1 ? 0xffff0000u : 0xffffu); }

// ---------------------------------------------------------------- loader
template <class K>
struct Loader : LoaderBase<K> {
  const Params& p;
  const MCtx& c;
  __device__ Loader(const Params& p_, const MCtx& c_, int lw_) : LoaderBase<K>(c_, lw_), p(p_), c(c_) {}

  __device__ void run() {
    const int NL = p.NL;
    auto u8 = [](const bf16* q) { return reinterpret_cast<const unsigned char*>(q); };
    const int cr = copy_row(c.lane), cq = copy_chunk(c.lane);
    const uint32_t vx = cr * (D * 2) + cq * 16, vd = cr * (FF * 2) + cq * 16;
    const int win = c.r / K::NRG, rg = c.r % K::NRG;
    const bool po = c.r < K::NRG * K::C;
    const int b = c.grp + c.an * K::NGRP, hg = K::HX * c.j + c.ah;
#pragma unroll 1
    for (int li = 0; li < p.S * NL && this->ok; li++) {
      const int l = li % NL;
      if (c.r < K::NRQ) {
        const unsigned char* w = u8(p.w_qkv) + (size_t)l * 3 * D * D * 2;
        this->template stage<K::RQ, K::RQ * KX>(vx, [&](int rt) {
          const int g = min(K::RQ * c.r + rt, K::TQ - 1), pt = g / (6 * K::HX);  // q | k | v, this XCD's heads
          return w + (size_t)(pt * D + HD * K::HX * c.j + 16 * (g - 6 * K::HX * pt)) * (D * 2);
        });
      }
      const size_t oo = ((size_t)l * D * D + (size_t)16 * K::RP * rg * D + 192 * (K::C * c.j + win)) * 2;
      if (po) this->template stage<K::RP, K::RP * KO>(vx, [&](int rt) { return u8(p.w_so) + oo + (size_t)rt * 16 * D * 2; });
      if (c.r < K::NRC) {
        const unsigned char* w = u8(p.w_cq) + ((size_t)l * D * D + (size_t)(HD * K::HX * c.j + 16 * K::RC * c.r) * D) * 2;
        this->template stage<K::RC, K::RC * KX>(vx, [&](int rt) { return w + (size_t)rt * 16 * D * 2; });
      }
      // context: a page is one 32-key block, K fragments (key tile f / 3, k-step f % 3) in its first half,
      // V^T fragments (dim tile f) in its second (six of each; two more copies repeat the first ones)
      const unsigned char* kb = u8(p.kctx) + (((size_t)b * NL + l) * p.Lkmax * D + HD * hg) * 2;
      const unsigned char* vb = u8(p.vtctx) + (((size_t)b * NL + l) * D + HD * hg) * p.Lkmax * 2;
#pragma unroll 1
      for (int i = 0; i < c.nblk && this->ok; i++) {
        if (!this->room()) break;
        const int k0 = c.kbeg + 32 * i;
        const uint32_t d = this->dst();
        if (this->lw == 0) {
#pragma unroll
          for (int f = 0; f < 8; f++) {
            const int ff = f % 6, kt = ff / 3, ks = ff - 3 * kt;
            int key = k0 + 8 * (cr >> 2) + 4 * kt + (cr & 3);
            if (key >= c.kend) key = 0;
            dma16(kb + ks * 64, (uint32_t)key * (D * 2) + cq * 16, d + f * 1024);
          }
        } else {
          int kg = k0 + 8 * cq;
          if (kg >= c.kend) kg = 0;
          const uint32_t vv = (uint32_t)cr * p.Lkmax * 2 + kg * 2;
#pragma unroll
          for (int f = 0; f < 8; f++) dma16(vb + (size_t)(f % 6) * 16 * p.Lkmax * 2, vv, d + f * 1024);
        }
        this->pg++;
      }
      if (po) this->template stage<K::RP, K::RP * KO>(vx, [&](int rt) { return u8(p.w_co) + oo + (size_t)rt * 16 * D * 2; });
#pragma unroll 1
      for (int q = 0; q < K::PG; q++) {
        const unsigned char* w =
            u8(p.w_gu) + ((size_t)l * 2 * FF + (size_t)c.j * (2 * FF / K::G) + 16 * (K::RG * c.r + K::RGP * q)) * D * 2;
        this->template stage<K::RGP, K::RGP * KX>(vx, [&](int rt) { return w + (size_t)rt * 16 * D * 2; });
      }
      if (po) {
        const unsigned char* w = u8(p.w_dn) + ((size_t)l * D * FF + (size_t)16 * K::RP * rg * FF + 768 * (K::C * c.j + win)) * 2;
        this->template stage<K::RP, K::RP * KD>(vd, [&](int rt) { return w + (size_t)rt * 16 * FF * 2; });
      }
    }
    this->drain();
  }
};

// Workspace offsets of the wave's token rows of a fragment-ordered operand with KT k-steps, from k-step
// ks0; rows past Tv or of an absent sample read zeros.
template <class K>
__device__ __forceinline__ void tok_off(const Params& p, const Ctx& c, uint32_t base, int KT, int ks0, uint32_t (&o)[K::NI]) {
  const int t = 16 * tile_of<K>(c) + c.lr;
#pragma unroll
  for (int i = 0; i < K::NI; i++)
    o[i] = t < p.Tv && slot_of<K>(c, i) < c.ns
               ? c.xb + base + (uint32_t)((tidx<K>(c, i) * KT + ks0) * 1024 + c.lane * 16)
               : OOB;
}

// ---------------------------------------------------------------- norm stages
// MODE 0: x = embed(x_t). MODE 1: x += gate * (sum of the 4 partials + bias). MODE 2: as 1, then the final
// norm, the action projection and the Euler update of x_t[:, :adim]. Token t = r (TT = 2) or r + 32 (wave /
// 2) of the wave's samples; lane holds columns 4 lane + 256 k + i, k < 3.
template <class K, int MODE>
__device__ __forceinline__ void stage_norm(const Params& p, const Ctx& c, uint32_t part, const float* bias,
                                           const float* gate, const float* scale, const float* shift, float dt) {
  const int t = K::TT == 2 ? c.r : c.r + 32 * (c.wave >> 1);
  f32x4 sc[3], sh[3], gt[3], bs[3];
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const int d = 4 * c.lane + 256 * k;
    sc[k] = *reinterpret_cast<const f32x4*>(scale + d);
    sh[k] = *reinterpret_cast<const f32x4*>(shift + d);
    if (MODE != 0) {
      gt[k] = *reinterpret_cast<const f32x4*>(gate + d);
      bs[k] = *reinterpret_cast<const f32x4*>(bias + d);
    }
  }
  u32x4 v[K::NI][4][3];
  if (MODE != 0) {
    part_wait<K>(c);
#pragma unroll
    for (int i = 0; i < K::NI; i++)
#pragma unroll
      for (int s = 0; s < 4; s++)
#pragma unroll
        for (int k = 0; k < 3; k++)
          v[i][s][k] = ldb128<kCpSc1>(c.ws, c.part + part + s * (K::PB1 / 4) +
                                                (uint32_t)(((slot_of<K>(c, i) * K::TT * 16 + t) * D + 4 * c.lane + 256 * k) * 4));
  }
#pragma unroll
  for (int i = 0; i < K::NI; i++) {
    if (slot_of<K>(c, i) >= c.ns) continue;
    const int slot = 2 * i + (c.wave >> 1);
    float* xres = reinterpret_cast<float*>(fg_lds + K::L_XRES) + slot * D;
    float* xt = reinterpret_cast<float*>(fg_lds + K::L_XT) + slot * AD;
    f32x4 x[3];
    if (MODE == 0) {
      // coalesced 1 KB reads of W_ain [768][32] (see pi05_group.hip)
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
      for (int k = 0; k < 3; k++) {
        const int d = 4 * c.lane + 256 * k;
        x[k] = *reinterpret_cast<const f32x4*>(xres + d) + *reinterpret_cast<const f32x4*>(p.b_ain + d);
      }
    } else {
#pragma unroll
      for (int k = 0; k < 3; k++) {
        const f32x4 s = as_f32x4(v[i][0][k]) + as_f32x4(v[i][1][k]) + as_f32x4(v[i][2][k]) + as_f32x4(v[i][3][k]);
        x[k] = *reinterpret_cast<const f32x4*>(xres + 4 * c.lane + 256 * k) + gt[k] * (s + bs[k]);
      }
    }
    float ss = 0.f;
#pragma unroll
    for (int k = 0; k < 3; k++) ss += x[k][0] * x[k][0] + x[k][1] * x[k][1] + x[k][2] * x[k][2] + x[k][3] * x[k][3];
    const float rr = rsqrtf(wave_sum(ss) / (float)D + 1e-6f);
    f32x4 h[3];
#pragma unroll
    for (int k = 0; k < 3; k++)
#pragma unroll
      for (int e = 0; e < 4; e++) h[k][e] = x[k][e] * rr * (1.0f + sc[k][e]) + sh[k][e];
    if (MODE != 2) {
#pragma unroll
      for (int k = 0; k < 3; k++) {
        const int d = 4 * c.lane + 256 * k;
        *reinterpret_cast<f32x4*>(xres + d) = x[k];
        const unsigned lo = pack_bf16x2(h[k][0], h[k][1]), hi = pack_bf16x2(h[k][2], h[k][3]);
        const unsigned plo = swap_adj(lo), phi = swap_adj(hi);
        if ((c.lane & 1) == (k & 1))  // whole 16-byte slots (see pi05_group.hip)
          *reinterpret_cast<u32x4*>(p.ws + c.xb + K::X_XN + tidx<K>(c, i) * (KX * 1024) + tfrag(t, d & ~7)) =
              (c.lane & 1) ? u32x4{plo, phi, lo, hi} : u32x4{lo, hi, plo, phi};
      }
    } else {
#pragma unroll 1
      for (int a = 0; a < p.adim; a++) {
        float s = 0.f;
#pragma unroll
        for (int k = 0; k < 3; k++) {
          const u32x2 wv = *reinterpret_cast<const u32x2*>(p.w_aout + (size_t)a * D + 4 * c.lane + 256 * k);
          s += bf_lo(wv[0]) * h[k][0] + bf_hi(wv[0]) * h[k][1] + bf_lo(wv[1]) * h[k][2] + bf_hi(wv[1]) * h[k][3];
        }
        s = wave_sum(s);
        if (c.lane == 0) xt[a] += dt * (s + p.b_aout[a]);
      }
    }
  }
}

// ---------------------------------------------------------------- GEMM stages
// QKV and CQ: R row tiles of the XCD's head rows, finished (+ bias) into the order the attention stages
// load them: 16-byte group (tile, head, slot, lane lr + 16 g4) = dims 16 (slot % 6) + 4 g4 .. + 3 of part
// slot / 6, so a tile's rows are one contiguous 1 KB store.
template <class K, int R, int NTILE, int NPART>
__device__ __forceinline__ void stage_heads(const Params& p, const Ctx& c, int pg0, uint32_t out, const float* bias) {
  wait_norm_rows<K>(c);
  f32x4 acc[K::NI][R];
  uint32_t xo[K::NI];
  tok_off<K>(p, c, K::X_XN, KX, 0, xo);
  gemm<K, R, KX, K::NI>(acc, c, pg0, xo);
#pragma unroll
  for (int rt = 0; rt < R; rt++) {
    const int g = R * c.r + rt;
    if (g >= NTILE) continue;
    const int pt = g / (6 * K::HX), q = g - 6 * K::HX * pt, hh = q / 6, q6 = q - 6 * hh;
    const f32x4 bv = *reinterpret_cast<const f32x4*>(bias + pt * D + HD * K::HX * c.j + 16 * q + 4 * c.lq);
#pragma unroll
    for (int i = 0; i < K::NI; i++)
      if (slot_of<K>(c, i) < c.ns)
        *reinterpret_cast<f32x4*>(p.ws + c.xb + out +
                                  (uint32_t)(((tidx<K>(c, i) * K::HX + hh) * 6 * NPART + 6 * pt + q6) * 1024 + c.lane * 16)) =
            acc[i][rt] + bv;
  }
}

// Partial sums of an output projection: KS k-steps of the token operand at `act` (KT k-steps per tile).
template <class K, int KS>
__device__ __forceinline__ void stage_part(const Params& p, const Ctx& c, int pg0, uint32_t act, int KT, uint32_t part) {
  const int win = c.r / K::NRG, rg = c.r % K::NRG, t = 16 * tile_of<K>(c) + c.lr;
  f32x4 acc[K::NI][K::RP];
  uint32_t xo[K::NI];
  tok_off<K>(p, c, act, KT, KS * win, xo);
  gemm<K, K::RP, KS, K::NI>(acc, c, pg0, xo);
  if (t >= p.Tv) return;
#pragma unroll
  for (int i = 0; i < K::NI; i++) {
    if (slot_of<K>(c, i) >= c.ns) continue;
#pragma unroll
    for (int rt = 0; rt < K::RP; rt++)
      stb128<kCpPart<K>>(c.ws, c.part + part + (K::C * c.j + win) * (K::PB1 / 4) +
                                  (uint32_t)(((slot_of<K>(c, i) * K::TT * 16 + t) * D + 16 * (K::RP * rg + rt) + 4 * c.lq) * 4),
                         as_u32x4(acc[i][rt]));
  }
}

template <class K>
__device__ __forceinline__ void stage_gu(const Params& p, const Ctx& c, int l, int pg0) {
  wait_norm_rows<K>(c);
  uint32_t xo[K::NI];
  tok_off<K>(p, c, K::X_XN, KX, 0, xo);
#pragma unroll 1
  for (int q = 0; q < K::PG; q++) {
    f32x4 acc[K::NI][K::RGP];
#pragma unroll
    for (int i = 0; i < K::NI; i++) asm volatile("" : "+v"(xo[i]));  // operand offsets are derived in each pass
    gemm<K, K::RGP, KX, K::NI>(acc, c, pg0 + q * (K::PGU / K::PG), xo);
    int lr = c.lr;
    asm volatile("" : "+v"(lr));
    if (16 * tile_of<K>(c) + lr >= p.Tv) continue;
#pragma unroll
    for (int rt = 0; rt < K::RGP; rt++) {
      const int row = 16 * (K::RG * c.r + K::RGP * q + rt) + 4 * c.lq;  // 2f, 2f + 1 = gate f, up f of the slice
      const f32x4 b = *reinterpret_cast<const f32x4*>(p.b_gu + (size_t)l * 2 * FF + c.j * (2 * FF / K::G) + row);
#pragma unroll
      for (int i = 0; i < K::NI; i++) {
        if (slot_of<K>(c, i) >= c.ns) continue;
        const f32x4 v = acc[i][rt] + b;
        *reinterpret_cast<unsigned*>(p.ws + c.xb + K::X_H + tidx<K>(c, i) * (96 / K::G * 1024) + tfrag(lr, row >> 1)) =
            pack_bf16x2(silu(v[0]) * v[1], silu(v[2]) * v[3]);
      }
    }
  }
}

// ---------------------------------------------------------------- self attention
// Rank r < NB HX: (sample slot r / HX, head r % HX). Wave tt < TT prepares tokens 16 tt .. + 15 into the
// Q / K / V^T fragments in LDS (zeros past Tv), waits for the other tiles' waves and attends with its own.
template <class K>
__device__ __forceinline__ void stage_satt(const Params& p, const Ctx& c, int li) {
  constexpr int TT = K::TT;
  const int n = c.r / K::HX, hh = c.r % K::HX, w = c.wave;
  if (n >= c.ns || w >= TT) return;
  constexpr uint32_t SQ = K::L_SATT, SK = SQ + TT * 3 * 1024, SV = SK + TT * 3 * 1024;
  const int tau = 16 * w + c.lr;
  const bool tv = tau < p.Tv;
  float q[24], k[24], v[24];
  {
    u32x4 r[18];
    const uint32_t o = 16 * w < p.Tv ? c.xb + K::X_QKV + (uint32_t)(((n * TT + w) * K::HX + hh) * 18 * 1024 + c.lane * 16) : OOB;
#pragma unroll
    for (int s = 0; s < 18; s++) r[s] = ldb128<kCpSc1>(c.ws, o + s * 1024);
#pragma unroll
    for (int s = 0; s < 6; s++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        q[4 * s + i] = as_f32(r[s][i]);
        k[4 * s + i] = as_f32(r[6 + s][i]);
        v[4 * s + i] = as_f32(r[12 + s][i]);
      }
  }
  rms96(q);
  rms96(k);
  const float* rc = p.rope_cos + (tv ? tau : 0) * 48 + 4 * c.lq;
  const float* rs = p.rope_sin + (tv ? tau : 0) * 48 + 4 * c.lq;
#pragma unroll
  for (int s = 0; s < 3; s++) {  // pairs (j, j + 48) = elements (4 s + i, 4 s + 12 + i) of the lane
    const f32x4 c4 = *reinterpret_cast<const f32x4*>(rc + 16 * s), s4 = *reinterpret_cast<const f32x4*>(rs + 16 * s);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int a = 4 * s + i, b = a + 12;
      const float q0 = q[a], q1 = q[b], k0 = k[a], k1 = k[b];
      q[a] = q0 * c4[i] - q1 * s4[i];
      q[b] = q0 * s4[i] + q1 * c4[i];
      k[a] = k0 * c4[i] - k1 * s4[i];
      k[b] = k0 * s4[i] + k1 * c4[i];
    }
  }
  const uint32_t kr = kperm_row(tau);
  const unsigned keep = keep_mask(tv);
  unsigned short* l16 = reinterpret_cast<unsigned short*>(fg_lds);
#pragma unroll
  for (int s = 0; s < 6; s++) {
    const int d = 16 * s + 4 * c.lq;
    *reinterpret_cast<u32x2*>(fg_lds + SQ + (w * 3 + (d >> 5)) * 1024 + frag_pos(tau, d)) = pack4(q, s, keep);
    *reinterpret_cast<u32x2*>(fg_lds + SK + ((kr >> 4) * 3 + (d >> 5)) * 1024 + frag_pos(kr, d)) = pack4(k, s, keep);
#pragma unroll
    for (int i = 0; i < 4; i++)
      l16[(SV + (s * (TT / 2) + (tau >> 5)) * 1024 + frag_pos(d + i, tau)) >> 1] = (unsigned short)(bf16_bits(v[4 * s + i]) & keep);
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  if (c.lane == 0) ctl_st<K>(8 + w, (unsigned)li + 1u);
  for (unsigned it = 0;; ++it) {
    unsigned m = ctl_ld<K>(8);
#pragma unroll
    for (int i = 1; i < TT; i++) m = min(m, ctl_ld<K>(8 + i));
    if (m >= (unsigned)li + 1u || ctl_ld<K>(6)) break;
    if (it > kSpinCap) {
      ctl_st<K>(6, 1u);
      if (c.lane == 0) atomicOr(c.err, kErrSpin);
      break;
    }
    __builtin_amdgcn_s_sleep(1);
  }
  asm volatile("" ::: "memory");
  if (16 * w >= p.Tv) return;
  auto frag = [&](uint32_t o) { return *reinterpret_cast<const u32x4*>(fg_lds + o + c.lane * 16); };
  u32x4 qf[3];
#pragma unroll
  for (int ks = 0; ks < 3; ks++) qf[ks] = frag(SQ + (w * 3 + ks) * 1024);
  const float qscale = 1.4426950408889634f * 0.10206207261596575f;  // log2(e) / sqrt(96)
  f32x4 s[TT];
#pragma unroll
  for (int kt = 0; kt < TT; kt++) {
    f32x4 a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < 3; ks++) a = mfma16(frag(SK + (kt * 3 + ks) * 1024), qf[ks], a);
    s[kt] = a;
  }
  float m_ = -1e30f;
#pragma unroll
  for (int kt = 0; kt < TT; kt++)
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int key = 32 * (kt >> 1) + 8 * c.lq + 4 * (kt & 1) + i;
      s[kt][i] = key < p.Tv ? s[kt][i] * qscale : -1e30f;
      m_ = fmaxf(m_, s[kt][i]);
    }
  m_ = cols_max(m_);
  float ps = 0.f;
  u32x4 pb[TT / 2];
#pragma unroll
  for (int kt = 0; kt < TT; kt += 2) {
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        s[kt + h][i] = exp2_w(s[kt + h][i] - m_);
        ps += s[kt + h][i];
      }
    pb[kt / 2] = u32x4{pack_bf16x2(s[kt][0], s[kt][1]), pack_bf16x2(s[kt][2], s[kt][3]),
                       pack_bf16x2(s[kt + 1][0], s[kt + 1][1]), pack_bf16x2(s[kt + 1][2], s[kt + 1][3])};
  }
  const float inv = 1.0f / cols_sum(ps);
#pragma unroll
  for (int dt = 0; dt < 6; dt++) {
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int sp = 0; sp < TT / 2; sp++) o = mfma16(frag(SV + (dt * (TT / 2) + sp) * 1024), pb[sp], o);
    o *= inv;
    if (tv)
      *reinterpret_cast<u32x2*>(p.ws + c.xb + K::X_ATT + (n * TT + w) * (3 * K::HX * 1024) + tfrag(tau, HD * hh + 16 * dt + 4 * c.lq)) =
          u32x2{pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3])};
  }
}

// ---------------------------------------------------------------- cross attention
// Item of rank r: sample slot an, head ah, context keys [kbeg, kend) in 32-key blocks, one ring page each.
// With TT = 2 waves (tt, tt + 2) share tile tt of the item's sample, taking alternate blocks. Segments of SB
// blocks: S^T of all of the wave's blocks, one softmax, O^T of all of them (see pi05_group.hip).
template <class K>
__device__ __forceinline__ void stage_catt(const Params& p, const MCtx& c, int pgk) {
  constexpr int TT = K::TT, NBK = SB / K::NP;
  const int tt = TT == 2 ? c.wave & 1 : c.wave, pr = TT == 2 ? c.wave >> 1 : 0;
  if (16 * tt >= p.Tv || c.an >= c.ns) {
    page_release<K>(c, pgk + c.nblk);
    return;
  }
  // the CQ waves of the tile
  xcd_wait_w(c, 0xffffffffu, TT == 2 ? 2 * (c.an & 1) + tt : tt);
  const int t = 16 * tt + c.lr;
  const bool tv = t < p.Tv;
  u32x4 qf[3];
  {
    u32x4 r[6];
    const uint32_t o = c.xb + K::X_QC + (uint32_t)(((c.an * TT + tt) * K::HX + c.ah) * 6 * 1024 + c.lane * 16);
#pragma unroll
    for (int s = 0; s < 6; s++) r[s] = ldb128<kCpSc1>(c.ws, o + s * 1024);
    float q[24];
#pragma unroll
    for (int s = 0; s < 6; s++)
#pragma unroll
      for (int i = 0; i < 4; i++) q[4 * s + i] = as_f32(r[s][i]);
    rms96(q);
    const unsigned keep = keep_mask(tv);
    const uint32_t qb = K::L_CQ + c.wave * 3072;  // the wave's own fragments
#pragma unroll
    for (int s = 0; s < 6; s++) {
      const int d = 16 * s + 4 * c.lq;
      *reinterpret_cast<u32x2*>(fg_lds + qb + (d >> 5) * 1024 + frag_pos(t, d)) = pack4(q, s, keep);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int ks = 0; ks < 3; ks++) qf[ks] = *reinterpret_cast<const u32x4*>(fg_lds + qb + ks * 1024 + c.lane * 16);
  }
  const float qscale = 1.4426950408889634f * 0.10206207261596575f;  // log2(e) / sqrt(96)
  float m = -1e30f, lsum = 0.f;
  f32x4 o[6];
#pragma unroll
  for (int dt = 0; dt < 6; dt++) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (int b0 = 0; b0 < c.nblk; b0 += SB) {
    // TT = 2: the last segment may hold no block of this wave; m, l and O then stay. (A softmax over masked
    // scores alone would weigh them exp2(rounding error of -1e30 qscale): 0 here, infinite for some scales.)
    if (b0 + pr >= c.nblk) {
      page_release<K>(c, pgk + c.nblk);
      break;
    }
    f32x4 s[2 * NBK];
#pragma unroll
    for (int i = 0; i < NBK; i++) {
      const int bi = b0 + K::NP * i + pr, nv = c.kend - (c.kbeg + 32 * bi);  // its valid keys
      s[2 * i] = s[2 * i + 1] = f32x4{-1e30f, -1e30f, -1e30f, -1e30f};
      if (bi >= c.nblk) continue;
      page_wait<K>(c, pgk + bi);
      u32x4 kf[6];
#pragma unroll
      for (int f = 0; f < 6; f++) kf[f] = *reinterpret_cast<const u32x4*>(fg_lds + ((pgk + bi) % K::RING) * PAGE + f * 1024 + frag_slot(c.lr, c.lq));
#pragma unroll
      for (int kt = 0; kt < 2; kt++) {
        f32x4 a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < 3; ks++) a = mfma16(kf[3 * kt + ks], qf[ks], a);
        if (nv < 32) {
#pragma unroll
          for (int e = 0; e < 4; e++)
            if (8 * c.lq + 4 * kt + e >= nv) a[e] = -1e30f;
        }
        s[2 * i + kt] = a;
      }
    }
    float bm = -1e30f;
#pragma unroll
    for (int q = 0; q < 2 * NBK; q++) bm = fmaxf(bm, fmaxf(fmaxf(s[q][0], s[q][1]), fmaxf(s[q][2], s[q][3])));
    const float mnew = fmaxf(m, cols_max(bm) * qscale);
    const float alpha = exp2_w(m - mnew);
    m = mnew;
    float ps = 0.f;
    u32x4 pb[NBK];
#pragma unroll
    for (int i = 0; i < NBK; i++) {
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          s[2 * i + h][e] = exp2_w(fmaf(s[2 * i + h][e], qscale, -m));
          ps += s[2 * i + h][e];
        }
      pb[i] = u32x4{pack_bf16x2(s[2 * i][0], s[2 * i][1]), pack_bf16x2(s[2 * i][2], s[2 * i][3]),
                    pack_bf16x2(s[2 * i + 1][0], s[2 * i + 1][1]), pack_bf16x2(s[2 * i + 1][2], s[2 * i + 1][3])};
    }
    lsum = lsum * alpha + cols_sum(ps);
#pragma unroll
    for (int dt = 0; dt < 6; dt++) o[dt] *= alpha;
#pragma unroll
    for (int i = 0; i < NBK; i++) {
      const int bi = b0 + K::NP * i + pr, nv = c.kend - (c.kbeg + 32 * bi);
      if (bi >= c.nblk) continue;
      u32x4 vf[6];
#pragma unroll
      for (int f = 0; f < 6; f++)
        vf[f] = *reinterpret_cast<const u32x4*>(fg_lds + ((pgk + bi) % K::RING) * PAGE + 8192 + f * 1024 + frag_slot(c.lr, c.lq));
      if (nv < 32) {
        const int q = min(max(nv - 8 * c.lq, 0), 8);
#pragma unroll
        for (int f = 0; f < 6; f++)
#pragma unroll
          for (int e = 0; e < 4; e++) vf[f][e] &= q >= 2 * e + 2 ? 0xffffffffu : (q == 2 * e + 1 ? 0xffffu : 0u);
      }
#pragma unroll
      for (int dt = 0; dt < 6; dt++) o[dt] = mfma16(vf[dt], pb[i], o[dt]);
    }
    page_release<K>(c, pgk + min(b0 + SB, c.nblk));
  }
  // O^T / l as operand fragments (see pi05_bs1.hip)
  const float inv = lsum > 0.f ? 1.0f / lsum : 0.f;
  const bool odd = c.lq & 1;
  const uint32_t ob = c.xb + K::X_CP + (uint32_t)((c.r * NCW + c.wave) * K::NI * 3072 + (((c.lq >> 1) + 2 * (c.lq & 1)) * 16 + c.lr) * 16);
#pragma unroll
  for (int ks = 0; ks < 3; ks++) {
    const unsigned a0 = pack_bf16x2(o[2 * ks][0] * inv, o[2 * ks][1] * inv);
    const unsigned a1 = pack_bf16x2(o[2 * ks][2] * inv, o[2 * ks][3] * inv);
    const unsigned b0 = pack_bf16x2(o[2 * ks + 1][0] * inv, o[2 * ks + 1][1] * inv);
    const unsigned b1 = pack_bf16x2(o[2 * ks + 1][2] * inv, o[2 * ks + 1][3] * inv);
    const LanePair s0 = swap16(a0, b0), s1 = swap16(a1, b1);
    if (tv)
      *reinterpret_cast<u32x4*>(p.ws + ob + ks * 1024) = odd ? u32x4{s0.lo, s1.lo, b0, b1} : u32x4{a0, a1, s0.hi, s1.hi};
  }
  if (tv && c.lq == 0)
    *reinterpret_cast<f32x2*>(p.ws + c.xb + K::X_CML + (uint32_t)((c.r * NCW + c.wave) * K::NI * 128 + c.lr * 8)) = f32x2{m, lsum};
}

// Rank r < 3 HX: head r / 3, k-step r % 3 of it, for the wave's token tiles. A lane owns one 16-byte slot
// (token lane % 16, 8 dims).
template <class K>
__device__ __forceinline__ void stage_comb(const Params& p, const Ctx& c) {
  constexpr int TT = K::TT;
  if (c.r >= 3 * K::HX) return;
  const int hh = c.r / 3, ks = c.r - 3 * hh, tt = tile_of<K>(c), t = 16 * tt + c.lr;
  const bool tv = t < p.Tv;
#pragma unroll
  for (int i = 0; i < K::NI; i++) {
    const int n = slot_of<K>(c, i);
    if (n >= c.ns) continue;
    const int r0 = (n * K::HX + hh) * K::NKC;  // ranks of the (sample, head)
    xcd_wait_w2(c, ((1u << K::NKC) - 1u) << r0, tt, TT == 2 ? tt + 2 : tt);
    u32x2 ml[K::NCH];
    u32x4 v[K::NCH];
#pragma unroll
    for (int q = 0; q < K::NCH; q++) {
      const int rw = (r0 + q / K::NP) * NCW + tt + 2 * (q % K::NP);
      ml[q] = ldb64<kCpSc1>(c.ws, tv ? c.xb + K::X_CML + (uint32_t)(rw * K::NI * 128 + c.lr * 8) : OOB);
      v[q] = ldb128<kCpSc1>(c.ws, tv ? c.xb + K::X_CP + (uint32_t)(rw * K::NI * 3072 + ks * 1024 + c.lane * 16) : OOB);
    }
    __builtin_amdgcn_sched_barrier(0);
    float M = -1e30f;
#pragma unroll
    for (int q = 0; q < K::NCH; q++) M = fmaxf(M, as_f32(ml[q][0]));
    float L = 0.f, u[8];
#pragma unroll
    for (int e = 0; e < 8; e++) u[e] = 0.f;
#pragma unroll
    for (int q = 0; q < K::NCH; q++) {
      const float w = as_f32(ml[q][1]) * exp2_w(as_f32(ml[q][0]) - M);
      L += w;
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const unsigned d = w != 0.f ? v[q][e] : 0u;
        u[2 * e] = fmaf(w, bf_lo(d), u[2 * e]);
        u[2 * e + 1] = fmaf(w, bf_hi(d), u[2 * e + 1]);
      }
    }
    const float inv = L > 0.f ? 1.0f / L : 0.f;
    u32x4 out;
#pragma unroll
    for (int e = 0; e < 4; e++) out[e] = pack_bf16x2(u[2 * e] * inv, u[2 * e + 1] * inv);
    *reinterpret_cast<u32x4*>(p.ws + c.xb + K::X_ATT + (uint32_t)((tidx<K>(c, i) * 3 * K::HX + 3 * hh + ks) * 1024 + c.lane * 16)) = out;
  }
}

// ---------------------------------------------------------------- kernel
__device__ __forceinline__ void mark(const Params& p, const Ctx& c, int idx, uint64_t& t0) {
  if (p.stage_cycles && blockIdx.x == 0 && c.wave == 0 && c.lane == 0) {
    const uint64_t now = __builtin_amdgcn_s_memrealtime();
    p.stage_cycles[idx] += now - t0;
    t0 = now;
  }
}

template <int G, int TT, int NB>
__global__ void __launch_bounds__(NTH, 1) ma2_group_kernel(Params p) {
  using K = Cfg<G, TT, NB>;
  MCtx c;
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
  c.xb = K::OFF_XCD + (uint32_t)c.x * K::XB;
  c.part = K::OFF_PART + (uint32_t)c.grp * K::NBUF * K::PB1;
  c.lds_addr = (uint32_t)(uintptr_t)fg_lds;
  c.err = reinterpret_cast<unsigned*>(p.ws + OFF_CTRL + 8);
  {
    c.an = c.r / (K::HX * K::NKC);
    c.ah = (c.r / K::NKC) % K::HX;
    const int kc = c.r % K::NKC, chunk = 32 * ((p.Lk + 32 * K::NKC - 1) / (32 * K::NKC));
    c.kbeg = min(kc * chunk, p.Lk);
    c.kend = min(c.kbeg + chunk, p.Lk);
    c.nblk = c.an < c.ns ? (c.kend - c.kbeg + 31) / 32 : 0;
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
  const int t = TT == 2 ? c.r : c.r + 32 * (c.wave >> 1);
  // this wave owns a token in the norm stages
  const bool nw = (c.wave & 1) == (c.r >> 4) && t < p.Tv && (TT == 4 || (c.wave >> 1) < c.ns);
  auto each_token = [&](auto f) {  // (x_t row, its LDS copy) of the wave's tokens
    for (int i = 0; i < K::NI; i++) {
      const int n = slot_of<K>(c, i);
      if (n < c.ns)
        f(p.x_t + ((size_t)(c.grp + n * K::NGRP) * p.xt_rows + t) * AD,
          reinterpret_cast<float*>(fg_lds + K::L_XT) + (2 * i + (c.wave >> 1)) * AD);
    }
  };
  if (nw && c.lane < AD) each_token([&](const float* g, float* s) { s[c.lane] = g[c.lane]; });
  const float dt = 1.0f / (float)p.S;
  const bool skip = idle<K>(p, c), po = c.r < K::NRG * K::C;
  const int win = c.r / K::NRG;
  int pg = 0;  // next ring page
  // a stage of np pages on this rank: run it, or release its pages unread
  auto stage = [&](bool mine, int np, auto f) {
    if (!mine) return;
    if (skip)
      page_release<K>(c, pg + np);
    else
      f(pg);
    pg += np;
  };
  auto buf = [&](int e) { return K::NBUF == 1 ? 0u : (uint32_t)(e & 1) * K::PB1; };
  uint64_t t0 = __builtin_amdgcn_s_memrealtime();
  auto signal = [&](int idx) {
    mark(p, c, idx, t0);
    xcd_signal(c);
    launder(c);
    mark(p, c, 15, t0);
  };
  auto publish = [&](int idx) {
    mark(p, c, idx, t0);
    part_signal<K>(c);
    launder(c);
    mark(p, c, 15, t0);
  };
  // ranks (per sample slot) whose self attention wrote heads 2 win, 2 win + 1, and the wave of the tile there
  uint32_t sm = 0;
  for (int i = 0; i < K::NI; i++) sm |= 3u << (slot_of<K>(c, i) * K::HX + 2 * win);
#pragma unroll 1
  for (int step = 0; step < p.S; step++) {
#pragma unroll 1
    for (int l = 0; l < NL; l++) {
      launder(c);
      const int li = step * NL + l;
      const float* mo = p.mods + (size_t)li * 9 * D;  // [3 norms][scale, shift, gate][D]
      const int e0 = 3 * li;
      if (nw) {
        if (l == 0)
          stage_norm<K, 0>(p, c, 0, nullptr, nullptr, mo, mo + D, 0.f);
        else
          stage_norm<K, 1>(p, c, buf(e0 - 1), p.b_dn + (size_t)(l - 1) * D, mo - 9 * D + 8 * D, mo, mo + D, 0.f);
      }
      signal(0);
      stage(c.r < K::NRQ, K::PQ, [&](int g) {
        stage_heads<K, K::RQ, K::TQ, 3>(p, c, g, K::X_QKV, p.b_qkv + (size_t)l * 3 * D);
      });
      mark(p, c, 1, t0);
      xcd_sync(c);
      launder(c);
      mark(p, c, 15, t0);
      stage_satt<K>(p, c, li);
      signal(2);
      stage(po, K::PO, [&](int g) {
        xcd_wait_w(c, sm, tile_of<K>(c));
        stage_part<K, KO>(p, c, g, K::X_ATT, 3 * K::HX, buf(e0));
      });
      publish(3);
      if (nw) stage_norm<K, 1>(p, c, buf(e0), p.b_so + (size_t)l * D, mo + 2 * D, mo + 3 * D, mo + 4 * D, 0.f);
      signal(4);
      stage(c.r < K::NRC, K::PC, [&](int g) {
        stage_heads<K, K::RC, K::TC, 1>(p, c, g, K::X_QC, p.b_cq + (size_t)l * D);
      });
      signal(5);
      stage_catt<K>(p, c, pg);
      pg += c.nblk;
      signal(6);
      if (!skip) stage_comb<K>(p, c);
      signal(7);
      stage(po, K::PO, [&](int g) {
        xcd_wait(c, 0x3fu << (6 * win));  // the combine of heads 2 win, 2 win + 1
        stage_part<K, KO>(p, c, g, K::X_ATT, 3 * K::HX, buf(e0 + 1));
      });
      publish(8);
      if (nw) stage_norm<K, 1>(p, c, buf(e0 + 1), p.b_co + (size_t)l * D, mo + 5 * D, mo + 6 * D, mo + 7 * D, 0.f);
      signal(9);
      stage(true, K::PGU, [&](int g) { stage_gu<K>(p, c, l, g); });
      signal(10);
      stage(po, K::PD, [&](int g) {
        constexpr int GW = 8 * G;  // gate/up ranks of a 768-column window
        xcd_wait(c, GW == 32 ? 0xffffffffu : ((1u << (GW & 31)) - 1u) << (GW * win));
        stage_part<K, KD>(p, c, g, K::X_H, 96 / G, buf(e0 + 2));
      });
      publish(12);
    }
    if (nw) {
      const int li = step * NL + NL - 1;
      const float* ml = p.mods + (size_t)li * 9 * D;
      const float* mf = p.mod_final + (size_t)step * 2 * D;
      stage_norm<K, 2>(p, c, buf(3 * li + 2), p.b_dn + (size_t)(NL - 1) * D, ml + 8 * D, mf, mf + D, dt);
    }
    mark(p, c, 13, t0);
  }
  if (c.j == 0 && nw && c.lane < p.adim) each_token([&](float* g, const float* s) { g[c.lane] = s[c.lane]; });
  if (c.j == 0 && c.r == 0 && c.wave == 0 && c.lane == 0)
    finish_group(p.ws, seq, (unsigned)min(p.B, K::NGRP), kOwnerMa2Group);
}

struct Choice {
  const void* kernel;
  unsigned lds;
  size_t ws;
};
template <int G, int TT, int NB>
Choice choice() {
  return {(const void*)ma2_group_kernel<G, TT, NB>, Cfg<G, TT, NB>::LDS, Cfg<G, TT, NB>::WS};
}
// Wider groups stream fewer weights per XCD but exchange partial sums between XCDs. ms per launch (Lk = 493,
// Tv = 30, 10 steps), against the stage engine's, all before the copies of copy_row, with which batches 2, 4
// and 16 run 12.5, 16.4 and 21.5:
//   batch 2   (4 XCDs, 2 samples) 12.6, (4, 4) 13.7   stage engine 27.6
//   batch 4   (4, 2) 16.5, (4, 4) 18.3                             28.9
//   batch 8   (2, 2) 17.7, (4, 4) 21.7                             28.8
//   batch 16  (2, 4) 22.1, (1, 2) 23.4                             31.2
// Two token tiles per wave is the most the registers hold, so past Tv = 32 (four tiles per sample) a group
// has two samples (batch 7, Tv = 64: 22.7 against 30.9). Past 16 samples the stage engine's tiles are full.
Choice pick(int batch, int Tv) {
  const bool t2 = Tv <= 32;
  if (batch <= 4) return t2 ? choice<4, 2, 2>() : choice<4, 4, 2>();
  if (batch <= 8) return t2 ? choice<2, 2, 2>() : choice<2, 4, 2>();
  return t2 ? choice<2, 2, 4>() : choice<1, 4, 2>();
}

}  // namespace mg

// ---------------------------------------------------------------- host
bool ma2_group_eligible(int batch, int Tv) { return batch >= 1 && batch <= 16 && Tv >= 1 && Tv <= 64; }
size_t ma2_group_workspace_bytes(int batch, int Tv) { return mg::pick(batch, Tv).ws; }

int ma2_group_launch(const fa_ma2_args* a, fa_stream_t stream) {
  using namespace fa::mg;
  const Choice k = pick(a->batch, a->Tv);
  const int rc = host::check_device(k.kernel, NTH, k.lds, NWG, "fa_ma2_flow");
  if (rc != FA_OK) return rc;
  Params p;
  p.w_qkv = static_cast<const bf16*>(a->w_qkv);
  p.w_so = static_cast<const bf16*>(a->w_so);
  p.w_cq = static_cast<const bf16*>(a->w_cq);
  p.w_co = static_cast<const bf16*>(a->w_co);
  p.w_gu = static_cast<const bf16*>(a->w_gu);
  p.w_dn = static_cast<const bf16*>(a->w_dn);
  p.b_qkv = a->b_qkv;
  p.b_so = a->b_so;
  p.b_cq = a->b_cq;
  p.b_co = a->b_co;
  p.b_gu = a->b_gu;
  p.b_dn = a->b_dn;
  p.mods = a->mods;
  p.mod_final = a->mod_final;
  p.rope_cos = a->rope_cos;
  p.rope_sin = a->rope_sin;
  p.w_ain = a->w_ain;
  p.b_ain = a->b_ain;
  p.w_aout = static_cast<const bf16*>(a->w_aout);
  p.b_aout = a->b_aout;
  p.kctx = static_cast<const bf16*>(a->kctx);
  p.vtctx = static_cast<const bf16*>(a->vtctx);
  p.x_t = a->x_t;
  p.stage_cycles = a->stage_cycles;
  p.ws = static_cast<unsigned char*>(a->workspace);
  p.NL = a->num_layers;
  p.Lk = a->Lk;
  p.Lkmax = a->Lkmax;
  p.Tv = a->Tv;
  p.adim = a->adim;
  p.S = a->num_steps;
  p.B = a->batch;
  p.xt_rows = a->xt_rows;
  void* args[] = {&p};
  return host::coop_launch(k.kernel, NWG, NTH, args, k.lds, stream, "fa_ma2_flow");
}

}  // namespace fa
