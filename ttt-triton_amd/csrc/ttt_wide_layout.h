// Shapes, LDS and `saved` layouts of the ttt_wide.h kernels, as plain constexpr
// integers (no HIP types): the kernels and their host code take them from here, and a
// host program compiled from this header alone checks them.
#pragma once

namespace ttt {

// K = 16 KT tokens, F = 16 FT features, hidden units in NSL slices of 64
// (the Linear loop: one "slice", its F = 64 output columns).
template <int KT_, int FT_, int NSL_, bool MLP_> struct WideShape {
  static constexpr int KT = KT_, FT = FT_, NSL = NSL_;
  static constexpr bool MLP = MLP_;
  static constexpr int K = 16 * KT, F = 16 * FT, S = 64, FF = S * NSL;
  static constexpr int NW = 4 * KT;        // waves: the 16 x 16 tiles of a K x 64 product
  static constexpr int NTH = 64 * NW;      // 16 threads per token row
  static constexpr int V = F / 16;         // features per thread in a row pass
  static constexpr int TW = FT * 4;        // 16 x 16 tiles of one slice of W1 or W2
  static constexpr int NT = (TW + NW - 1) / NW;  // of those, per wave
  // whether every wave has a tile in each pass over them (no branch then)
  static constexpr bool ALLT = TW % NW == 0, ALLF = FT == 4, ALLK = KT == 4;
  // the state launches of 16 waves, MLP: addresses out of the registers (see pinned:
  // backward at K = F = FF = 64, B32 H4, 8 mini-batches 247 -> 172 us).  (K = 48 has 168
  // registers a wave and spills 69 of the MLP's backward; not tried there.)
  static constexpr bool PIN = KT == 4 && MLP;
  // the state launches' products onto a state: term by term (see wmm)
  static constexpr bool CHAIN = KT == 1;
  // LDS rows are padded by 4 floats: row-major float4 reads (16 rows x 4 lane
  // groups) and column reads (4 rows x 16 lanes) both touch 64 distinct banks
  static constexpr int LS = S + 4, LF = F + 4, LK = K + 4;
  static constexpr int SLOT = 64 * LS;     // one LDS matrix of up to 64 x 64
  static constexpr int KSLOT = K * LS;     // one of K rows
  // whether wave w has a tile of a K x F product, and the token whose eta a lane
  // holds for it (-1: none; the tile's row would be past the mini-batch, and
  // past eta's end at the last one)
  static constexpr bool f_tile(int w) { return ALLF || w < KT * FT; }
  static constexpr int f_token(int w, int lane) { return f_tile(w) ? 16 * (w / FT) + (lane & 15) : -1; }
  static_assert(MLP || (FT == 4 && NSL == 1), "the Linear loop: 64 features, one slice");
};

// the readout launches, which have registers to spare and no loop: not pinned
template <class C> struct WideFree {
  static constexpr int KT = C::KT, NSL = C::NSL;
  static constexpr bool PIN = false, CHAIN = false;
};

// floats of one (chain, mini-batch) slot of `saved`: what the forward writes, then
// the handoff, which the backward writes.  A forward's `saved` may hold the first
// part alone (half of it); a backward then begins with wide_spread_kernel.
// (With the two parts at strides of their own the state launches of the backward
// lost 3%: K = F = FF = 64, B32 H4, 8 mini-batches 166 -> 170 us, the split form's
// F = 32, FF = 128, 64 chains, 32 mini-batches 313 -> 326.)
template <class C> struct WideSlot {
  static constexpr int STATE = C::MLP ? 2 * C::F * C::FF + C::FF + C::F : C::F * C::F + C::F;
  // the state entering the mini-batch
  static constexpr int W1 = 0;
  static constexpr int B1 = C::MLP ? C::F * C::FF : C::F * C::F;
  static constexpr int W2 = B1 + (C::MLP ? C::FF : C::F);
  static constexpr int B2 = W2 + C::FF * C::F;
  // written by wide_fwd_state: Z1 + b1 and P = G2 W2^T (MLP), G2 (Linear: G),
  // the normalised Z2 (Linear: Z) and its sigma
  static constexpr int Z1 = STATE;
  static constexpr int P = Z1 + (C::MLP ? C::K * C::FF : 0);
  static constexpr int G2 = P + (C::MLP ? C::K * C::FF : 0);
  static constexpr int ZH = G2 + C::K * C::F;
  static constexpr int SIG = ZH + C::K * C::F;
  static constexpr int FWD = SIG + C::K;
  // the handoff from wide_bwd_readout to wide_bwd_state: the readout's terms
  // of dG1, dX2, dG2, dXK, the state gradient, the LayerNorm parameters'
  // gradients, and deta's last row (for an lr rule: dlr)
  static constexpr int HG1 = FWD;
  static constexpr int HX2 = HG1 + (C::MLP ? C::K * C::FF : 0);
  static constexpr int HG2 = HX2 + (C::MLP ? C::K * C::FF : 0);
  static constexpr int HXK = HG2 + C::K * C::F;
  static constexpr int HST = HXK + C::K * C::F;  // dW1, db1[, dW2, db2] laid out as the state
  static constexpr int HLW = HST + STATE;
  static constexpr int HLB = HLW + C::F;
  static constexpr int HDE = HLB + C::F;
  static constexpr int FLOATS = HDE + C::K;
};

}  // namespace ttt
