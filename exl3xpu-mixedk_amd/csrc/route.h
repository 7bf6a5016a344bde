// route.h -- how a batch of sequences is launched: the sequences per forward
// workgroup, and the fused two-pass launch or separate ones.  Host code
// without a device, from times measured on 256 CUs.
#pragma once

namespace xtq {

// Microseconds one CU takes per step of one sequence, by K and sequences per
// workgroup (1, 2, 4, 8), measured over tail-bites of 16,384 sequences.
inline double forward_step_us(int K, int T) {
    static const double us[6][4] = {{1.350, 1.350, 1.350, 1.350}, {1.258, 1.255, 1.255, 1.255},
                                    {1.190, 1.219, 1.171, 1.171}, {1.242, 1.235, 1.217, 1.198},
                                    {1.281, 1.292, 1.235, 1.220}, {1.309, 1.298, 1.261, 1.231}};
    if (K < 2 || K > 7) return 1.0;
    return us[K - 2][T <= 1 ? 0 : T <= 2 ? 1 : T <= 4 ? 2 : 3];
}

// Estimated microseconds per step of a launch of nseq >= 1 sequences, T per
// workgroup, on ncu CUs.  One workgroup per CU is resident, so the launch runs
// in rounds of ncu workgroups, each T sequences long.  The last workgroup takes
// the nseq % T sequences that are left, and where the others fill whole rounds
// it is a round by itself: of its own length, not of T sequences (K=4, T = 4 on
// 256 CUs, us a step: 1024 / 1025 / 1026 / 1028 sequences 4.60 / 6.02 / 7.35 /
// 9.20).  It has its CU to itself without enough sequences to cover each
// other's latency, which takes it 1.2 times the one-sequence time for each (1.43
// to 1.57 us alone, two 2.7 to 2.9, four of eight 5.2 to 5.6), up to a whole
// workgroup's.
inline double forward_cost_us(int K, int T, int nseq, int ncu) {
    if (ncu < 1) ncu = 1;
    const int full = nseq / T, rest = nseq % T;
    const double round = T * forward_step_us(K, T);
    double us = (double)(full / ncu) * round;
    if (full % ncu) {
        us += round;
    } else if (rest) {
        const double own = 1.2 * rest * forward_step_us(K, 1);
        us += own < round ? own : round;
    }
    return us;
}

// Sequences per workgroup, at most max_T (the LDS bounds it by K), that finish
// nseq sequences first: a group that fills its last round beats a larger one
// that does not (K=4, tail-bite calls on 256 CUs: 2000 sequences T = 1 in eight
// rounds 5.10 ms, T = 4 in two 5.05; 1500 T = 1 in six 3.84, T = 4 in two 4.93).
inline int forward_group(int K, int max_T, int nseq, int ncu) {
    int best = 1;
    double cost = forward_cost_us(K, 1, nseq, ncu);
    for (int T = 2; T <= max_T; T *= 2) {
        const double c = forward_cost_us(K, T, nseq, ncu);
        if (c <= cost) {
            best = T;
            cost = c;
        }
    }
    return best;
}

// Steps until the last of a fused launch's 2 nseq workgroups ends: each CU
// takes the next of nseq first passes and then of nseq second passes, of d1 and
// d2 steps, as soon as it is free.
inline double fused_steps(int nseq, int d1, int d2, int ncu) {
    const int r = nseq / ncu, m = nseq % ncu;  // pass 1: m CUs take r + 1, the others r
    const int cus[2] = {ncu - m, m};
    double t[2] = {(double)r * d1, (double)(r + 1) * d1};
    double end = m ? t[1] : t[0];
    for (int left = nseq; left > 0;) {
        const int g = m && t[1] < t[0] ? 1 : 0;            // the CUs free first
        t[g] = (t[g] < d1 ? d1 : t[g]) + d2;               // (a pass 2 waits for its pass 1)
        if (t[g] > end) end = t[g];
        left -= cus[g];
    }
    return end;
}

// Whether a tail-bite of nseq sequences (n1 steps of pass 1, its pivot, nsteps
// of pass 2, row_bytes of backpointers per step) ends sooner as one fused
// launch than as separate ones.
//   The fused launch fills its rounds with 2 nseq passes of one sequence, each
// with its own traceback: 26 (K=7) to 40 steps' time (K=2), half of what a pair
// of passes takes beyond 512 steps at 16,384 sequences.  Separate launches run
// T sequences per workgroup and read the kept rows again, at 4.7 TB/s, or in
// 0.3 ms with one lane per sequence.  The fused estimate is raised by 1.5 %:
// with that the choices lose least against the faster route, 0.1 % on average
// and 4 % at most over 474 batches of 257 to 6000 sequences (K = 2..7, three
// pivots, two devices), which is as far as two runs of one batch differ.
//   Up to one sequence per CU both take two rounds at best.  On the GPU the
// separate launches are the sooner from some 40 sequences on: a fused launch's
// waiting workgroups poll, and where its 2 nseq are not all resident (above half
// a sequence per CU) second passes that start early hold CUs, presumably
// unevenly over the dies to which workgroups are dealt in turn, and the time is
// that of three rounds.  Between other kernels, as in quantize_seq_tailbite,
// four launches take some 20 us longer than back to back and one launch does
// not: there the two cross at 80 to 90 sequences of 256 CUs, where the line is.
// From 16 sequences per CU a round is a small part of the whole.
//   quantize_seq_tailbite, pivot 128, fused / separate, us.  K=4: 1 sequence
// 671 / 669, 8 682 / 728, 64 729 / 734, 80 737 / 746, 96 763 / 738, 128 756 /
// 731, 192 1061 / 740, 256 768 / 743, 300 1096 / 1316, 400 1421 / 1326, 513
// 1768 / 1909, 600 1778 / 1943, 1003 2804 / 2578.  K=2: 8 771 / 828, 64 823 /
// 837, 96 854 / 832, 128 845 / 856, 192 1195 / 850, 256 859 / 857, 300 1240 /
// 1528, 400 1642 / 1548, 513 2004 / 2225, 1003 3189 / 3145.  K=7: 8 744 / 783,
// 64 792 / 812, 80 800 / 847, 96 809 / 809, 128 838 / 811, 192 1162 / 817, 300
// 1180 / 1495, 600 1915 / 2138, 1003 3014 / 2732.
//   The library's own entry, K=4: 64 713 / 670, 768 2105 / 1960, 1025 3058 /
// 3061, 2049 5844 / 5622; K=2: 512 1599 / 1559, 1025 3539 / 3693, 1537 5094 /
// 5199.
inline bool fused_ends_first(int K, int max_T, double row_bytes, int nseq, int n1, int pivot,
                             int nsteps, int ncu) {
    if (K < 2 || K > 7) return false;
    if (ncu < 1) ncu = 1;
    if (nseq <= ncu) return 3 * nseq <= ncu;
    if (nseq >= 16 * ncu) return false;
    static const int tb[6] = {40, 39, 35, 28, 31, 26};
    const double fused = 1.015 * forward_step_us(K, 1) *
                         fused_steps(nseq, n1 + tb[K - 2], nsteps + tb[K - 2], ncu);
    double rows = row_bytes * nseq * (n1 - 1 - pivot + nsteps - 1) / 4.7e6;        // us
    if (rows > 300.0) rows = 300.0;
    const int T = forward_group(K, max_T, nseq, ncu);
    return fused < forward_cost_us(K, T, nseq, ncu) * (n1 + nsteps) + rows;
}

}  // namespace xtq
