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

// Whether the backward columns run fused with the w-projection at a
// runtime-radix size: one column of one image per workgroup, layer after layer,
// `columns` of them (the width times the images of a kind) of `waves` waves each.
// Too few wait on memory and on themselves, and the separate passes, whose
// workgroups own four columns of one layer, are faster. Invert of one image in the
// mixed precision, 48 layers, 0.15 M samples, fused and separate in us:
//   300^2: 331, 127; 600^2: 486, 188; 1000^2: 534, 381; 1200^2: 592, 516;
//   480 x 3000: 765, 558; 512 x 6144: 830, 1121;
//   1680^2: 876, 1038; 1920^2: 863, 1194; 3072^2: 1946, 2979
// Near the line the difference is of either sign (1500^2: 915, 850; two images
// of 480 x 3000: 982, 1047; two of a kind, 13 M samples: 960^2 3768, 4125 and 1152^2
// 4316, 4061).
constexpr bool fusedColumns(long columns, int waves) {
  return columns >= 1600 || columns * waves >= 2800;
}

// Whether the forward rows of a runtime-radix size (`rows` of `n` values) run from
// the model image for every layer: a workgroup then owns four rows, or two, for a
// group of layers. Predict of four images, 48 layers, fused and separate in us:
// 720^2: 1053, 793; 1000^2: 1795, 1784; 1200^2: 2394, 2499; 1500^2: 4396, 4181
// (but two of 1500 x 1260, 24 layers: 60 us less fused); 1680^2: 4349, 5470; 1920^2:
// 5180, 6389; 1800 values x 300 rows: 1083, 1166; 480 x 3000: 2658, 2745; 512 x 6144:
// 5155, 5415; and of one image 300 x 1800: 334, 277.
constexpr bool fusedModelRows(int n, int rows) { return n >= 1400 || rows >= 2800; }

}  // namespace hws

#endif
