// Host check of csrc/ttt_wide_layout.h: prints the first violated statement and
// returns 1, or the number of shapes checked.
#include <cstdio>

#include "ttt_wide_layout.h"

using namespace ttt;

#define HOLD(x)                                                                          \
  do {                                                                                   \
    if (!(x)) {                                                                          \
      std::printf("K %d F %d FF %d mlp %d: " #x "\n", C::K, C::F, C::FF, (int)C::MLP);    \
      return false;                                                                      \
    }                                                                                    \
  } while (0)

template <class C> bool check() {
  // every wave's reads of eta's last row stay in the mini-batch, and every
  // (token, tile column) of a K x F product has exactly one wave
  int seen[C::K][C::FT] = {};
  for (int w = 0; w < C::NW; ++w)
    for (int lane = 0; lane < 64; ++lane) {
      const int t = C::f_token(w, lane), s = 16 * (w / 4) + (lane & 15);
      HOLD(t >= -1 && t < C::K);
      HOLD(s >= 0 && s < C::K);
      if (t >= 0 && lane < 16) ++seen[t][w % C::FT];
    }
  for (int t = 0; t < C::K; ++t)
    for (int j = 0; j < C::FT; ++j) HOLD(seen[t][j] == 1);
  // the slot's parts follow each other without a gap, the handoff last
  using Sl = WideSlot<C>;
  const int hid = C::MLP ? C::K * C::FF : 0;
  HOLD(Sl::B1 == C::F * (C::MLP ? C::FF : C::F));
  HOLD(!C::MLP || (Sl::W2 == Sl::B1 + C::FF && Sl::B2 + C::F == Sl::STATE));
  HOLD(Sl::Z1 == Sl::STATE && Sl::P == Sl::Z1 + hid && Sl::G2 == Sl::P + hid);
  HOLD(Sl::FWD == Sl::G2 + 2 * C::K * C::F + C::K && Sl::HG1 == Sl::FWD && Sl::HG2 == Sl::HG1 + 2 * hid);
  HOLD(Sl::HST == Sl::HG2 + 2 * C::K * C::F && Sl::HST + Sl::STATE == Sl::HLW && Sl::HLB == Sl::HLW + C::F);
  HOLD(Sl::FLOATS == Sl::HLB + C::F + C::K);
  // 16-byte accesses
  HOLD(Sl::FLOATS % 4 == 0 && Sl::FWD % 4 == 0 && Sl::STATE % 4 == 0 && C::LS % 4 == 0 && C::LF % 4 == 0 && C::LK % 4 == 0);
  // the nine matrices and the bias rows of a state launch fit the LDS
  HOLD((9 * C::SLOT + C::FF + C::F + 8 * C::K) * 4 <= 160 * 1024);
  return true;
}

template <int KT> bool check_kt() {
  return check<WideShape<KT, 4, 1, false>>() && check<WideShape<KT, 4, 1, true>>() && check<WideShape<KT, 4, 4, true>>() &&
         check<WideShape<KT, 2, 2, true>>();
}

int main() {
  if (!(check_kt<1>() && check_kt<2>() && check_kt<3>() && check_kt<4>())) return 1;
  std::printf("16\n");
  return 0;
}
