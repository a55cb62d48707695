// The exact coarse level's host set-up (stz::direct_inverse) on three levels of
// 4 x 2 nodes: diagonal, singular, and with a u-u block that differs left and
// right.  Prints each verdict and the diagonal level's first entries.
#include <cstdio>
#include <vector>

namespace stz {
const char *direct_inverse(const double *S, int M, int Nn, std::vector<double> &D);
}

int main() {
    const int M = 4, Nn = 2;
    std::vector<double> S(40 * Nn, 0.0), D;
    auto verdict = [&] {
        const char *why = stz::direct_inverse(S.data(), M, Nn, D);
        std::printf("%s\n", why ? why : "solved");
    };
    for (int j = 0; j < Nn; j++) S[40 * j + 16] = 2, S[40 * j + 19] = 4;
    verdict();
    std::printf("%g %g %g\n", D[0], D[1], D[5]);  // mode 0, weight 1/4: 1/2, 0, 1/4 times it
    S[40 + 19] = 0;
    verdict();
    S[40 + 19] = 4;
    S[12] = 1e-3;
    verdict();
    return 0;
}
