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

// Whether the runtime-radix transforms of lines of n values run fused with the
// image-domain work: the backward columns with the w-projection (one column per
// workgroup, layer after layer), the forward rows from the model image for every
// layer. Below, a column of 32 of every 128 bytes and a workgroup per column
// leave the chip waiting on memory and on itself, and the separate passes, whose
// workgroups own four lines of one layer, are faster. Invert of one image in the
// mixed precision, 48 layers, 0.15 M samples, fused and separate in us:
//   300: 331, 127; 600: 486, 188; 1000: 534, 381; 1200: 592, 516; 1500: 915, 850;
//   1680: 876, 1038; 1920: 863, 1194; 3072: 1946, 2979
// and of four images, two of them complex: 1500: 3790, 3161; 1680: 3862, 4073.
// Predict of the four: 720: 1053, 793; 1500: 4396, 4181; 1680: 4349, 5470.
constexpr bool fusedRuntimeRadix(int n) { return n >= 1600; }

}  // namespace hws

#endif
