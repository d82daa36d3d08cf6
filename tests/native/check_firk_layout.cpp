// check_firk_layout.cpp -- the FIRK kernels' areas (boundaryvaluediffeq.jl_amd/csrc/firk_layout.h):
// every value of every interval of every instance has a place of its own inside them, and they
// are at most a line per instance larger than packed ones.  Exit status 0 when that holds.
#include "../../boundaryvaluediffeq.jl_amd/csrc/firk_layout.h"

#include <cstdio>
#include <vector>

using namespace bvpdev;

static int failures = 0;
static void expect(bool ok, const char *what, int cap, int N) {
    if (!ok && ++failures < 20) std::printf("FAILED: %s (cap %d, %d)\n", what, cap, N);
}

// the chunk partition of N intervals over 64 lanes
static void chunk_of(int N, int lane, int &start, int &len) {
    const int P = N < 64 ? N : 64, q = N / P, r = N % P;
    len = lane < P ? q + (lane < r) : 0;
    start = lane < P ? lane * q + (lane < r ? lane : r) : N;
}

int main() {
    const int nf = 6, n = 67;
    for (int cap : {2, 3, 4, 5, 9, 10, 17, 22, 32, 33, 34, 64, 65, 66, 100, 129, 130, 200, 1025}) {
        const int most = (int)firk_intervals(cap);
        const size_t total = firk_stage_values(n, cap, nf), slot = firk_lines(most) * nf;
        for (int N : {1, 2, most / 2, most - 1, most}) {
            if (N < 1 || N > most) continue;
            std::vector<char> used(total, 0);
            for (int b = 0; b < n; ++b) {
                int seen = 0;
                for (int lane = 0; lane < 64; ++lane) {
                    int start, len;
                    chunk_of(N, lane, start, len);
                    for (int i = 0; i < len; ++i, ++seen)
                        for (int q = 0; q < nf; ++q) {
                            const size_t o = firk_cell(lane, i, nf) + (size_t)q * 64;
                            const size_t at = firk_stage_base(b, cap, nf) + o;
                            expect(o < slot, "inside the slot's area", cap, N);
                            expect(at < total, "inside the batch's area", cap, N);
                            if (at < total) expect(!used[at]++, "a place of its own", cap, N);
                        }
                }
                expect(seen == N, "every interval", cap, N);
            }
        }
        // against packed areas (cap intervals per instance): no larger where lines are shared, but
        // for the last line; less than a line more otherwise
        for (size_t m : {1, 7, 1000, 16384}) {
            const size_t packed = m * cap * nf, v = firk_stage_values(m, cap, nf);
            if (most <= 32) expect(v <= packed * 64 / (64 / most * most) + 64 * nf, "shared lines", cap, (int)m);
            else expect(v <= packed + m * 62 * nf, "whole lines", cap, (int)m);
        }
        for (int S : {1, 3, 7}) {
            const size_t f = 2 * S * 2 + S * 2 * 3;
            expect(firk_aux_values(cap, 2, S) <= (size_t)cap * (4 + f) + 62 * f, "slot size", cap, S);
        }
    }
    std::printf("%s: %d failures\n", failures ? "FAIL" : "OK", failures);
    return failures ? 1 : 0;
}
