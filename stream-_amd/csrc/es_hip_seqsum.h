// The pieces of an in-order double sum evaluated in parallel, for sums of non-negative terms (rmsnorm's squares).
//
// The reference adds a row's squares one after another in double (src/es_engine.c:189-194), and every addition rounds, so
// the result depends on the order. Inside one binade [2^E, 2^(E+1)) of the running sum s the spacing of doubles is a fixed
// u = 2^(E-52), and s is a multiple of it: adding a term moves s by the term rounded to a multiple of u, where only a tie
// looks at s itself, at the parity of s / u (round half to even). A run of consecutive terms inside a binade is therefore
// a function of that one parity: an increment and an end parity for an even start, and the same for an odd start. Such
// functions compose associatively, and their increments (multiples of u below 2^53 u) add exactly. So:
//   * an ordinary parallel prefix sum says in which binade each thread's terms begin and end;
//   * a thread whose terms stay in one binade adds them onto an even and onto an odd representative of that binade (plain
//     double additions: the hardware rounds and breaks the ties) and so has its run's function;
//   * the functions of consecutive such threads are composed by a scan; a thread whose terms leave the binade (one for
//     each doubling of the sum) is an event, whose terms are added one by one onto the exact sum.
// The prefix sum is rounded differently from the in-order sum, so the binades it gives are checked against the exact sum
// at both ends of every run (s is monotone, so the ends vouch for the middle); where one is wrong the caller adds the row
// in order instead. Terms are squares of floats: no subnormal double occurs, and a sum of binade 0 is zero.
//
// ESQ_SEQSUM_QUAL is the function qualifier: __device__ in the library, plain static inline in the CPU check.
#ifndef ES_HIP_SEQSUM_H
#define ES_HIP_SEQSUM_H
#include <stdint.h>

#ifndef ESQ_SEQSUM_QUAL
#define ESQ_SEQSUM_QUAL __device__ __forceinline__
#endif

// increments from an even and from an odd start; bit 0 of e: the end is odd from an even start, bit 1: it is even from an
// odd start. All zero is the empty run.
struct SeqRun { double a0, a1; uint32_t e; };

ESQ_SEQSUM_QUAL uint32_t seq_binade(double s) { return (uint32_t)(__builtin_bit_cast(uint64_t, s) >> 52); }   // s >= 0

// terms whose running sum goes from `from` to `to` (approximately) can be a run: one binade, finite
ESQ_SEQSUM_QUAL bool seq_is_run(double from, double to) {
    const uint32_t b = seq_binade(from);
    return b == seq_binade(to) && b < 0x7ff;
}

// the run of n terms in binade b
template <int N> ESQ_SEQSUM_QUAL SeqRun seq_run(const double (&q)[N], uint32_t b) {
    if (b == 0) return SeqRun{0.0, 0.0, 0};   // the sum is zero and stays so
    const uint64_t even = (uint64_t)b << 52;
    const double s0 = __builtin_bit_cast(double, even), s1 = __builtin_bit_cast(double, even + 1);
    double t0 = s0, t1 = s1;
    for (int i = 0; i < N; i++) {
        t0 = t0 + q[i];
        t1 = t1 + q[i];
    }
    const uint32_t p0 = (uint32_t)__builtin_bit_cast(uint64_t, t0) & 1u, p1 = (uint32_t)__builtin_bit_cast(uint64_t, t1) & 1u;
    return SeqRun{t0 - s0, t1 - s1, p0 | (p1 ^ 1u) << 1};
}

// b if odd, else a, by masks (a choice between two fields of a struct can become an indexed load from the stack)
ESQ_SEQSUM_QUAL double seq_pick(bool odd, double a, double b) {
    const uint64_t m = odd ? ~0ull : 0ull;
    return __builtin_bit_cast(double, (__builtin_bit_cast(uint64_t, b) & m) | (__builtin_bit_cast(uint64_t, a) & ~m));
}

// x, then y
ESQ_SEQSUM_QUAL SeqRun seq_join(const SeqRun &x, const SeqRun &y) {
    const bool o0 = x.e & 1u, o1 = !(x.e & 2u);   // x ends odd from an even, from an odd start
    const uint32_t ye0 = y.e & 1u, ye1 = (y.e >> 1 & 1u) ^ 1u;
    const uint32_t e0 = o0 ? ye1 : ye0, e1 = o1 ? ye1 : ye0;
    return SeqRun{x.a0 + seq_pick(o0, y.a0, y.a1), x.a1 + seq_pick(o1, y.a0, y.a1), e0 | (e1 ^ 1u) << 1};
}

// the sum after a run from s; b: the binade the run was formed in. ok is cleared when s was or is not in it.
ESQ_SEQSUM_QUAL double seq_add_run(double s, const SeqRun &r, uint32_t b, bool &ok) {
    const double t = s + seq_pick(__builtin_bit_cast(uint64_t, s) & 1u, r.a0, r.a1);
    ok = ok && seq_binade(s) == b && seq_binade(t) == b;
    return t;
}
#endif
