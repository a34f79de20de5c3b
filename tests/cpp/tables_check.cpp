// The Hamiltonian's quadratic-form tables against 113-bit arithmetic: every entry is the exact sum
// over the interactions, rounded once: half a unit in its last place, and 16 units of 64-bit
// significands of the size of the summed tensors (their eigenvalues: the rotations' elements are
// themselves sums of products of size one) for the sum itself.  Prints OK.
#include "fake_hip.h"

#include "../../blochlib_amd/csrc/blfid_host.cpp"

#include <quadmath.h>

typedef __float128 Q;

// C = R diag(p) R^T and the size of p
static void tensor(const Q p[3], const double *eul, Q C[6], Q M[6]) {
    const Q rad = M_PIq / 180, a = eul[0] * rad, b = eul[1] * rad, g = eul[2] * rad;
    const Q ca = cosq(a), sa = sinq(a), cb = cosq(b), sb = sinq(b), cg = cosq(g), sg = sinq(g);
    const Q R[3][3] = {{ca * cb * cg - sa * sg, sa * cb * cg + ca * sg, -sb * cg},
                       {-ca * cb * sg - sa * cg, -sa * cb * sg + ca * cg, sb * sg},
                       {ca * sb, sa * sb, cb}};
    const int I[6] = {0, 1, 2, 0, 0, 1}, J[6] = {0, 1, 2, 1, 2, 2};
    for (int q = 0; q < 6; q++) {
        C[q] = M[q] = 0;
        for (int k = 0; k < 3; k++) {
            const Q v = R[I[q]][k] * p[k] * R[J[q]][k];
            C[q] += v;
            M[q] += fabsq(p[k]);
        }
    }
}

int main() {
    const int S = 5, N = 1 << S;
    int fails = 0;
    for (int seed = 0; seed < 20; seed++) {
        unsigned long x = 88172645463325252ul + seed;
        auto rnd = [&](double lo, double hi) { // xorshift
            x ^= x << 13; x ^= x >> 7; x ^= x << 17;
            return lo + (hi - lo) * (double)(x >> 11) / 9007199254740992.0;
        };
        const std::vector<int> iso = {2, 1, 1, 1, 1};
        std::vector<double> csa, dip, jc;
        for (int i = 0; i < S; i++)
            for (double v : {rnd(-1000, 1000), rnd(1000, 8000), rnd(0, 1), (double)i, rnd(0, 360), rnd(0, 360), rnd(0, 360)})
                csa.push_back(v);
        for (int i = 0; i < S; i++)
            for (int j = i + 1; j < S; j++)
                for (double v : {rnd(-30000, -500), (double)i, (double)j, 0.0, rnd(0, 180), rnd(0, 360)}) dip.push_back(v);
        for (double v : {rnd(10, 150), 0.0, 1.0, 0.0, rnd(5, 15), 1.0, 2.0, 1.0}) jc.push_back(v);
        const blfid_system sys = {S, iso.data(), S, csa.data(), (int)dip.size() / 6, dip.data(), 2, jc.data()};
        blfid_plan *p = nullptr;
        if (blfid_plan_create(&sys, 10000, 54.7356, 160000, 64, 0, BLFID_FP64, &p)) return 2;
        auto m = [&](int s, int i) { return (Q)(s >> (S - 1 - i) & 1 ? -0.5 : 0.5); };
        auto check = [&](const double *got, const Q *sum, const Q *mag, const char *what, int at) {
            for (int q = 0; q < 7; q++) {
                const Q err = fabsq((Q)got[q] - sum[q]);
                if (err > fabsq(sum[q]) * 0x1p-53 * (1 + 0x1p-9) + mag[q] * 0x1p-60) {
                    if (fails++ < 5) std::printf("FAIL seed %d %s %d entry %d: off by %.3g of %.3g\n", seed, what, at, q, (double)err, (double)mag[q]);
                }
            }
        };
        auto add = [](Q *sum, Q *mag, int q, Q v) { sum[q] += v; mag[q] += fabsq(v); };
        auto add_tensor = [](Q *sum, Q *mag, const Q *C, const Q *M, Q f) {
            for (int q = 0; q < 6; q++) {
                sum[1 + q] += C[q] * f;
                mag[1 + q] += M[q] * fabsq(f);
            }
        };
        for (int s = 0; s < N; s++) {
            Q sum[7] = {0}, mag[7] = {0}, C[6], M[6];
            for (int i = 0; i < S; i++) {
                const double *c = &csa[7 * i];
                const Q d = c[1], e = c[2], t[3] = {d * (e - 1) / 2, -d * (e + 1) / 2, d};
                tensor(t, c + 4, C, M);
                add(sum, mag, 0, -(Q)c[0] * m(s, i));
                add_tensor(sum, mag, C, M, m(s, i));
            }
            for (size_t z = 0; z < dip.size(); z += 6) {
                const int i = (int)dip[z + 1], j = (int)dip[z + 2];
                const Q d = dip[z], t[3] = {-d / 2, -d / 2, d};
                tensor(t, &dip[z + 3], C, M);
                add_tensor(sum, mag, C, M, 2 * m(s, i) * m(s, j));
            }
            for (int z = 0; z < 8; z += 4) add(sum, mag, 0, (Q)jc[z] * m(s, (int)jc[z + 1]) * m(s, (int)jc[z + 2]));
            check(&p->xd_cst[7 * s], sum, mag, "state", s);
        }
        for (int i = 0; i < S; i++)
            for (int j = 0; j < S; j++) {
                Q sum[7] = {0}, mag[7] = {0}, C[6], M[6];
                if (i == 1 && j == 2 || i == 2 && j == 1) add(sum, mag, 0, (Q)jc[4] / 2);
                for (size_t z = 0; z < dip.size(); z += 6) {
                    const int a = (int)dip[z + 1], b = (int)dip[z + 2];
                    if (iso[a] != iso[b] || !(a == i && b == j || a == j && b == i)) continue;
                    const Q d = dip[z], t[3] = {-d / 2, -d / 2, d};
                    tensor(t, &dip[z + 3], C, M);
                    add_tensor(sum, mag, C, M, (Q)-0.5);
                }
                check(&p->xd_fpr[7 * (i * S + j)], sum, mag, "pair", i * S + j);
            }
        blfid_plan_destroy(p);
    }
    if (!fails) std::printf("OK\n");
    return fails ? 1 : 0;
}
