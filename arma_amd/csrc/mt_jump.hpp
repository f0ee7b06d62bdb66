// Jump-ahead polynomials of the p = 521 dynamic-creator generators (n = 17
// words, m = 8, w = 32, r = 23).
//
// The word sequence x_1, x_2, ... of such a generator satisfies the scalar
// recurrence over GF(2) whose polynomial is the characteristic polynomial
// chi of its state transition (Cayley-Hamilton; chi need not be primitive),
// so x_(J+k) = sum of g_i x_(i+k) over the set bits of g = t^J mod chi
// (Haramoto, Matsumoto, Nishimura, Panneton and L'Ecuyer, "Efficient jump
// ahead for F2-linear random number generators", INFORMS JoC 20(3), 2008).
// With a_i bit i of aaa, A = t^n + t^m and B = t^(n-1) + t^(m-1),
//   chi = A^(w-r) B^r + sum_(i<r) a_i A^(w-r) B^(r-1-i)
//                     + sum_(i=r..w-1) a_i A^(w-1-i)
// (Matsumoto and Nishimura, "Mersenne Twister", ACM TOMACS 8(1), 1998,
// appendix), so chi is the exclusive or of 33 fixed polynomials, tabled
// here, selected by the bits of aaa.
#pragma once

#include <cstdint>

namespace arma_hip {

constexpr int kJumpN = 17, kJumpM = 8, kJumpR = 23;
constexpr int kJumpDegree = 521;                 // n w - r
constexpr int kJumpWords = 17;                   // words of a residue mod chi
constexpr int kJumpTop = kJumpDegree - 32 * 16;  // bits of its last word

// Polynomials of degree up to 521, bit i of word i / 32 the coefficient of t^i.
struct JumpPoly {
	uint32_t w[kJumpWords] = {};
};

// a * (t^i + t^j)
constexpr JumpPoly jump_times(const JumpPoly& a, int i, int j) {
	JumpPoly r;
	for (int b = 0; b <= kJumpDegree; ++b) {
		if (!((a.w[b >> 5] >> (b & 31)) & 1u)) continue;
		for (int s : {i, j})
			if (b + s <= kJumpDegree) r.w[(b + s) >> 5] ^= 1u << ((b + s) & 31);
	}
	return r;
}

// The residue of t^521 modulo chi is base plus the sum of a[i] over the set
// bits i of aaa (chi without its leading term).
struct JumpTable {
	JumpPoly base, a[32];
};

constexpr JumpTable jump_table() {
	JumpTable t;
	JumpPoly p;  // A^k, then A^(w-r) B^k
	p.w[0] = 1u;
	for (int k = 0; k <= 32 - kJumpR; ++k) {
		// A^k goes with bit w - 1 - k where that is at least r
		if (31 - k >= kJumpR) t.a[31 - k] = p;
		if (k < 32 - kJumpR) p = jump_times(p, kJumpN, kJumpM);
	}
	for (int k = 0; k < kJumpR; ++k) {
		t.a[kJumpR - 1 - k] = p;  // A^(w-r) B^k
		p = jump_times(p, kJumpN - 1, kJumpM - 1);
	}
	t.base = p;
	t.base.w[16] &= (1u << kJumpTop) - 1u;  // without t^521
	return t;
}

}  // namespace arma_hip
