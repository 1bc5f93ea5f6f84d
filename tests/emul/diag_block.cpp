// potrf_block on the CPU: the factor and the inverse of a diagonal block against
// a plain Cholesky factorization (a non-positive pivot reported and replaced by
// 1), and bit for bit the same whichever wave is first between two barriers.
//
//   diag_block fp64|fp32 nb [column whose diagonal entry is negative]
//   diag_block publish       a tail that publishes its block to other workgroups
#include "kernels_factor.h"

using namespace mxc;

template <typename T>
static int check(int nb, int bad) {
    const int ld = nb + 3;
    const double tol = std::is_same<T, double>::value ? 1e-13 : 1e-4;
    std::vector<double> A(nb * nb), L(nb * nb, 0.0), X(nb * nb, 0.0);
    unsigned seed = 12345u + nb;
    auto rnd = [&] { return (int)((seed = seed * 1664525u + 1013904223u) >> 8) / 8388608.0 - 1.0; };
    for (int j = 0; j < nb; j++)
        for (int i = j; i < nb; i++) A[i + j * nb] = (double)(T)(i == j ? 4.0 + rnd() : rnd() / sqrt((double)nb));
    if (bad >= 0) A[bad + bad * nb] = -1.0;
    int first = INT_MAX;
    for (int j = 0; j < nb; j++)
        for (int i = j; i < nb; i++) {
            double s = A[i + j * nb];
            for (int k = 0; k < j; k++) s -= L[i + k * nb] * L[j + k * nb];
            if (i == j && !(s > 0)) {
                first = min(first, 100 + j);
                s = 1.0;
            }
            L[i + j * nb] = i == j ? sqrt(s) : s / L[j + j * nb];
        }
    for (int c = 0; c < nb; c++)
        for (int i = c; i < nb; i++) {
            double s = i == c;
            for (int k = c; k < i; k++) s -= L[i + k * nb] * X[k + c * nb];
            X[i + c * nb] = s / L[i + i * nb];
        }
    std::vector<T> W0((size_t)ld * nb + nb * nb, (T)7), out[2];
    for (int j = 0; j < nb; j++)
        for (int i = j; i < nb; i++) W0[i + j * ld] = (T)A[i + j * nb];
    const DiagTask t{0, (long long)ld * nb, ld, nb, 100, 0};
    const int orders[2][4] = {{0, 1, 2, 3}, {3, 2, 1, 0}};
    for (int o = 0; o < 2; o++) {
        std::vector<T> W = W0, S(potrf_lds<T>(false) / sizeof(T));
        int sfail[2], fail = INT_MAX;
        emu::run(orders[o], [&] {
            potrf_block<T, false>(t, W.data(), S.data(), sfail, &fail, (const double *)nullptr, 0.0, Redo{},
                                  (double *)nullptr);
        });
        double err = 0;
        for (int j = 0; j < nb; j++)
            for (int i = j; i < nb; i++) {
                const double e = max(fabs((double)W[i + j * ld] - L[i + j * nb]),
                                     fabs((double)W[t.winv + i + j * nb] - X[i + j * nb]));
                if (!(e <= err)) err = e;          // (a NaN stays)
            }
        printf("first wave %d: error %.2e, fail %d\n", orders[o][0], err, fail);
        if (!(err <= tol) || fail != first) return 1;
        out[o] = W;
    }
    if (memcmp(out[0].data(), out[1].data(), out[0].size() * sizeof(T))) {
        printf("the result depends on the order of the waves\n");
        return 1;
    }
    return 0;
}

static int publish() {
    const int nb = NB;
    std::vector<double> W(2 * nb * nb, 0.0);
    for (int i = 0; i < nb; i++) W[i + i * nb] = 4.0;
    const DiagTask t{0, nb * nb, nb, nb, 0, 0};
    int fail = INT_MAX, ready = 0, abort = 0;
    const PdArgs pda{&t, &fail, 0.0, Redo{}, &ready, &abort, 1};
    std::vector<double> smem(potrf_lds<double>(false) / sizeof(double));
    emu::run({0, 1, 2, 3}, [&] {
        pd_tail<double, false>(pda, 0, W.data(), (unsigned char *)smem.data(), (const double *)nullptr, true);
    });
    printf("flag %d, lanes whose stores were not released before it: %d\n", ready, emu::unreleased_flags);
    return ready == 1 && emu::unreleased_flags == 0 && W[0] == 2.0 && W[nb * nb] == 0.5 ? 0 : 1;
}

int main(int argc, char **argv) {
    if (argc == 2 && !strcmp(argv[1], "publish")) return publish();
    if (argc < 3) return 2;
    const int nb = atoi(argv[2]), bad = argc > 3 ? atoi(argv[3]) : -1;
    return !strcmp(argv[1], "fp64") ? check<double>(nb, bad) : check<float>(nb, bad);
}
