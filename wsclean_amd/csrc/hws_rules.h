// Rules of the launches that depend on sizes alone (no device code).
#ifndef HWS_RULES_H
#define HWS_RULES_H

namespace hws {

// Workgroups per CU of a kernel whose workgroups each take a static share of
// the work, from the number that is resident at once: whole rounds of them, and
// five or more, so that shares of unequal weight even out. Degridding at
// oversampling 1023, where LDS leaves room for four, four, three and three
// workgroups with one to four images (2048^2 x 33 layers, 14 M samples):
//   five, a round and a part of one:    375, 433, 616, 634 us
//   as many as registers alone allow
//   (8, 7, 5, 4):                       330, 374, 623, 693
//   one round:                          314, 358, 560, 593
//   whole rounds from five up:          323, 369, 527, 571
// and 6144^2 x 96 layers, one image: 1922 us with five, 1541 with one round of
// four, 1467 with two.
constexpr int wholeRounds(int resident) {
  const int r = resident > 1 ? resident : 1;
  return r * ((4 + r) / r);
}

}  // namespace hws

#endif
