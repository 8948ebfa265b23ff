// Lanes per atom of the pair kernels that split an atom's list.
#pragma once
#include <algorithm>

namespace emdee {

// 1, 4, 16, 32 or 64 lanes for N atoms whose lists hold `entries` entries in
// all: enough wavefronts to fill the chip (at least 2^18 lanes) and about 24
// entries per lane, so that long lists (water at rc 10 A holds ~700 entries
// per atom) are spread over many waves.
// Small systems with long lists go past 16, as long as all blocks are resident
// at once; a few blocks left over for later cost more than the shorter walks
// save.  A CU holds four blocks of the FP64 kernels (103 to 122 registers) and
// five of the mixed (83 to 91), so 32 lanes reach to 8,192 and 10,240 atoms
// and 64 to 4,096.  Step times, us, with 16 / 32 / 64 lanes:
//   64 lanes: up to 1,024 atoms, a block per CU (800 LJ atoms, 125 entries
//   38.9 / 37.8 / 37.2), and longer lists (2,000, 320: 48.7 / 45.9 / 45.0;
//   3,072, 349: 51.0 / 48.6 / 48.3; 3,000 water atoms, 698: 114.5 / 107.1 /
//   101.6).
//   32 lanes: shorter lists (1,500 LJ atoms, 132: 39.9 / 38.6 / 39.0; 3,072,
//   122: 44.6 / 44.4 / 45.8; 4,096, 353: 51.5 / 48.7 / 49.6) and more atoms
//   (8,192, 727: 67.8 / 62.5 / 67.4).
//   16 lanes: 12,288 LJ atoms, 735: 77.3 / 82.4 / 82.7, mixed 79.9 / 83.8 /
//   80.6.  Water's FP64 terms hide the late blocks (12,288 atoms, 721:
//   143.1 / 141.8 / 144.8), so several types keep 32 to 16,384 atoms.
// Below 96 entries 16 and 32 lanes are even (2,000 atoms, 91: 43.2 / 42.5).
inline int pair_lanes(int N, double entries, bool mixed, bool uniform) {
  const long lanes = std::max(1L << 18, (long)(entries / 24.0));
  const long want = lanes / std::max(N, 1);
  const double each = entries / std::max(N, 1);
  if (N <= 4096 && want >= 64 && each >= 96.0) return each >= (N <= 1024 ? 96.0 : N <= 3072 ? 200.0 : 600.0) ? 64 : 32;
  const int most = mixed ? 10240 : uniform ? 8192 : 16384;
  if (N <= most && want >= 24 && each >= 384.0) return 32;
  return want >= 16 ? 16 : (want >= 4 ? 4 : 1);
}

}  // namespace emdee
