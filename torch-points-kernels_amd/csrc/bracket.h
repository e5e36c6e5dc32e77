// A bracket around the distance a selection looks for (survivors.h): plain arithmetic, without a word of device code, so that
// it can be tried on the host.
#pragma once

// Guesses narrow [lo, hi) down: at first along the caller's estimate, then - after a few, or when an estimate leaves the bracket -
// by halving the number of floats in it, which at most 31 times leaves none.
constexpr int BRACKET_ESTIMATES = 6; // guesses along the estimate
constexpr int BRACKET_TRIES = 40;    // guesses in all: beyond these no distance separates

struct Bracket
{
    float lo = 0.0f, hi = __builtin_inff(); // too few candidates lie within lo, too many within hi

    // The guess after `guess`, which was too small (few) or too large; estimate: where the caller expects it.
    constexpr float next(float guess, bool few, float estimate, int tries)
    {
        if (few)
            lo = guess;
        else
            hi = guess;
        if (estimate > lo && estimate < hi && tries < BRACKET_ESTIMATES)
            return estimate;
        // (both are >= 0, so their bit patterns order like them; hi is mostly +inf here, whose pattern added to another one
        // is beyond an int)
        const int low = __builtin_bit_cast(int, lo), high = __builtin_bit_cast(int, hi);
        return __builtin_bit_cast(float, low + (high - low) / 2);
    }
};
