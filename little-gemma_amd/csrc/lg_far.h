// lg_far.h — units of q8 rows that a launch hands from one XCD to others, and the marks that tell a unit of this launch from what lay there before.
//
// 16 bytes, three dwords of data: {x, mark a | low half of y, z, high half of y | mark b}.  Memory keeps accesses of 8 bytes whole and wider ones by no rule, so either half
// of a unit has a mark of its own, 16 bits: the launch's layer in both (8 bits, never 0: cleared memory fits no launch), and 8 of the step's number, in a its low
// ones, in b the next ones plus these.  Both together tell steps apart up to 2^16 of them (LG_MARK_STEPS).  A half alone tells launches of different layers apart, which is
// what two launches that follow each other at a unit are, the next layer's or, in the next step, the first one's behind the last one's; and, where one layer of a
// model has such launches, steps up to 254 apart.  (x, y, z and the tag exclusive-or'ed with them would not do: a unit whose first half is old fits wherever x ^ y has
// not changed, two zeros say.  With two halves to join where they are taken, E4B shape, one to eight rows, a step is -9 to +15 us of 1470 to 2000 against that, 3 in the
// mean, which is what two builds of the same kernels differ by.)
//
// No includes: the host's tests build it as it is.
#pragma once
#ifdef __HIPCC__
#define LG_FAR_FN __host__ __device__ __forceinline__ static
#else
#define LG_FAR_FN static inline
#endif

// Both marks in one word, a in its upper half.  tag: lg_tag of the launch, whose number is 256 times the step's and the layer
LG_FAR_FN unsigned lg_far_marks(unsigned tag) {
    const unsigned layer = tag >> 4 & 255, step = tag >> 12;
    return layer << 24 | (step & 255) << 16 | layer << 8 | ((step + (step >> 8)) & 255);
}
// (lower half of x, upper half of y: one instruction)
LG_FAR_FN unsigned lg_far_halves(unsigned x, unsigned y) { return (x & 0xFFFF) | (y & 0xFFFF0000u); }
template <typename V>                // V: x, y, z, w of 32 bits each
LG_FAR_FN V lg_far_unit(unsigned x, unsigned y, unsigned z, unsigned marks) { V v; v.x = x; v.y = lg_far_halves(y, marks); v.z = z; v.w = lg_far_halves(marks, y); return v; }
// 0 if the unit is of this launch (of several units: all of them or'ed together)
template <typename V>
LG_FAR_FN unsigned lg_far_miss(const V &v, unsigned marks) { return lg_far_halves(v.w, v.y) ^ marks; }
template <typename V>
LG_FAR_FN unsigned lg_far_y(const V &v) { return lg_far_halves(v.y, v.w); }
