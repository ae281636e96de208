// The first entries of a seeded random permutation, without making the permutation.
//
// A quantiser's initial codewords are the first few hundred elements of torch.randperm(n) for n in the hundreds of thousands:
// made whole, on the host, that permutation took 1.7 ms per codebook - more than all the iterations behind it.  Its elements
// are those of a forward Fisher-Yates shuffle (Durstenfeld 1964) driven by MT19937 (Matsumoto and Nishimura 1998): step i
// swaps elements i and i + r % (n - i), r the next 32-bit output, so the first `count` elements follow from `count` draws,
// and what the rest of the shuffle would draw only has to be skipped when another permutation follows from the same
// generator.  Skipping advances the generator's state and tempers nothing (vectorised: 0.3 ns a draw).
#pragma once

#include <cstdint>
#include <vector>

namespace vq {

class Mt19937 {
public:
    explicit Mt19937(uint32_t seed)
    {
        s_[0] = seed;
        for (int i = 1; i < kN; i++) s_[i] = 1812433253u * (s_[i - 1] ^ (s_[i - 1] >> 30)) + (uint32_t)i;
        at_ = kN;
    }
    uint32_t next()
    {
        if (at_ == kN) refill();
        uint32_t y = s_[at_++];
        y ^= y >> 11;
        y ^= (y << 7) & 0x9d2c5680u;
        y ^= (y << 15) & 0xefc60000u;
        return y ^ (y >> 18);
    }
    void skip(int64_t n)
    {
        while (n > 0) {
            if (at_ == kN) refill();
            const int64_t step = n < kN - at_ ? n : kN - at_;
            at_ += (int)step;
            n -= step;
        }
    }

private:
    static constexpr int kN = 624, kM = 397;
    static uint32_t mix(uint32_t hi, uint32_t lo)
    {
        const uint32_t y = (hi & 0x80000000u) | (lo & 0x7fffffffu);
        return (y >> 1) ^ ((0u - (y & 1u)) & 0x9908b0dfu);
    }
    void refill()
    {
        twist(s_);
        at_ = 0;
    }
    // (element i needs i + 1 and i + 397, old or already new: every loop reads at least 227 elements away from what it writes)
    __attribute__((optimize("O3"), target_clones("avx512f", "avx2", "default"))) static void twist(uint32_t *s)
    {
        for (int i = 0; i < kN - kM; i++) s[i] = s[i + kM] ^ mix(s[i], s[i + 1]);
        for (int i = kN - kM; i < kN - 1; i++) s[i] = s[i + kM - kN] ^ mix(s[i], s[i + 1]);
        s[kN - 1] = s[kM - 1] ^ mix(s[kN - 1], s[0]);
    }
    uint32_t s_[kN];
    int at_;
};

// out[0 .. count) = the first elements of the permutation of 0 .. n-1; `another`: one more follows from the same generator,
// which then moves on by the whole permutation's draws
inline void first_of_permutation(Mt19937 &gen, int64_t n, int64_t count, bool another, int32_t *out)
{
    // elements that are not where they started: open addressing, at most half full (as a node-based map, four fifths of the
    // time: 256 draws 9.5 us)
    size_t slots = 16;
    while (slots < 4 * (size_t)count) slots *= 2;
    std::vector<int64_t> where(slots, -1);
    std::vector<int32_t> what(slots);
    auto find = [&](int64_t i) {
        size_t at = (size_t)((uint64_t)i * 0x9e3779b97f4a7c15ull >> 32) & (slots - 1);
        while (where[at] >= 0 && where[at] != i) at = (at + 1) & (slots - 1);
        return at;
    };
    auto value = [&](int64_t i) {
        const size_t at = find(i);
        return where[at] < 0 ? (int32_t)i : what[at];
    };
    for (int64_t i = 0; i < count; i++) {
        const int64_t j = i < n - 1 ? i + (int64_t)(gen.next() % (uint32_t)(n - i)) : i;
        const int32_t mine = value(i);
        const size_t at = find(j);
        out[i] = where[at] < 0 ? (int32_t)j : what[at];
        where[at] = j;
        what[at] = mine;
    }
    if (another) gen.skip(n - 1 - (count < n - 1 ? count : n - 1));
}

}  // namespace vq
