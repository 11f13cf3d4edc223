// hwt_scale.h -- scaling a state that grows sixfold a step (hwt_tri.h).  No HIP in
// here: a host program can run the bookkeeping by itself.
#pragma once

#include <stdint.h>

namespace hwt {

// The powers of two a state is scaled back by, in step with its growth of log2 6 bits
// a step: the whole bits of all steps so far, so that what is left over stays below
// one bit after each scaling, however many steps there are and however they are
// divided into calls.  (At a fixed 2^-165 for 64 steps 0.44 bits would be left each
// time.)  Scaling by powers of two changes no bit of a price.
struct SixfoldScale {
    static constexpr int EVERY = 64;  // steps between scalings; at most 2^166 in between
    static constexpr uint64_t BITS = 11102329402;  // log2 6 in units of 2^-32
    uint32_t frac = 0;  // of a bit, not yet scaled away
    int32_t run = 0;    // steps since the last scaling

    // whole bits to scale away after `steps` more steps
    constexpr int bits(int steps)
    {
        const uint64_t g = frac + (uint64_t)steps * BITS;
        frac = (uint32_t)g;
        return (int)(g >> 32);
    }
    // steps that may follow before the next scaling
    constexpr int room() const { return EVERY - run; }
    // after c <= room() steps: bits to scale away now, 0 if it is not yet time
    constexpr int after(int c)
    {
        run += c;
        if (run < EVERY) return 0;
        run = 0;
        return bits(EVERY);
    }
};

// Bits by which a state is larger (below 0: smaller) than it would be had it been
// scaled at each of its own steps, to one bit or two: its steps were those from the
// `from`th to the `to`th counted.
constexpr int sixfold_left(int from, int to)
{
    return (int)(2.5849625f * (float)((to & (SixfoldScale::EVERY - 1)) - (from & (SixfoldScale::EVERY - 1))));
}

// 2^-bits, bits < 1023
constexpr double pow2_down(int bits) { return __builtin_bit_cast(double, (uint64_t)(1023 - bits) << 52); }

// n steps in pieces that end where the scaling falls due: steps(c) makes c of them,
// scale(f) multiplies the state by f.
template <class Steps, class Scale>
__attribute__((always_inline)) constexpr void scaled_steps(SixfoldScale &s, int n, Steps &&steps, Scale &&scale)
{
    while (n > 0) {
        const int c = n < s.room() ? n : s.room();
        steps(c);
        n -= c;
        const int bits = s.after(c);
        if (bits) scale(pow2_down(bits));
    }
}

} // namespace hwt
