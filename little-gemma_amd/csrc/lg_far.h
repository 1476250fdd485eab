// lg_far.h — units of q8 rows that a launch hands from one XCD to others, and the marks that tell a unit of this launch from what lay there before.
//
// 16 bytes, three dwords of data: {x, mark a | low half of y, z, mark b | high half of y}.  Memory keeps accesses of 8 bytes whole, wider ones by no rule, so either half of
// a unit has a mark of its own.  A mark is 16 bits: the launch's layer in both (8 bits, never 0: cleared memory fits no launch), and 8 of the step's number, in a its low ones, in b
// the next ones plus these.  Both together tell steps apart up to 2^16 of them (LG_MARK_STEPS).  A half alone tells launches of different layers apart, which is what two
// launches that follow each other at a unit are, the next layer's or, in the next step, the first one's behind the last one's; and, where one layer of a model has such
// launches, steps up to 254 apart.  (Until then x, y, z and the tag exclusive-or'ed with them: a unit whose first half was old fitted wherever x ^ y had not
// changed, two zeros say.  The same number of operations on either side, one more to join y's halves.)
//
// No includes: the host's tests build it as it is.
#pragma once
#ifdef __HIPCC__
#define LG_FAR_FN __host__ __device__ __forceinline__ static
#else
#define LG_FAR_FN static inline
#endif

struct LgFarMarks { unsigned a, b; };
// tag: lg_tag of the launch, whose number is 256 times the step's and the layer
LG_FAR_FN LgFarMarks lg_far_marks(unsigned tag) {
    const unsigned layer = tag >> 4 & 255, step = tag >> 12;
    LgFarMarks m; m.a = layer << 24 | (step & 255) << 16; m.b = layer << 24 | ((step + (step >> 8)) & 255) << 16;
    return m;
}
template <typename V>                // V: x, y, z, w of 32 bits each
LG_FAR_FN V lg_far_unit(unsigned x, unsigned y, unsigned z, LgFarMarks m) { V v; v.x = x; v.y = (y & 0xFFFF) | m.a; v.z = z; v.w = y >> 16 | m.b; return v; }
// Below 2^16 if the unit is of this launch (of several units: all of them or'ed together)
template <typename V>
LG_FAR_FN unsigned lg_far_miss(const V &v, LgFarMarks m) { return (v.y ^ m.a) | (v.w ^ m.b); }
template <typename V>
LG_FAR_FN unsigned lg_far_y(const V &v) { return v.w << 16 | (v.y & 0xFFFF); }
