// Host-side check of the ghost-cell rules (fill_value of
// mesoflow_amd/csrc/mf_kernels.inc.h and its adjoint Rev::fill_rev), compiled
// for the host from the sources the kernels use. Every boundary code in every
// direction and on every side, on domains of 1, 2, 3 and more cells:
//  - values: bit for bit the rules as FillPatch words them, written here as a
//    recursion (a cell outside in periodic directions only is its periodic
//    image; else foextrap and wall reflection in x, y, z order, then the
//    ext_dir functor in x, y, z order, each reading its source cell's value);
//  - adjoint: <lambda, dF> by central differences of the fill against the
//    adjoint folded into the valid cells.
// Prints a summary and exits non-zero on failure.
#define main adjoint_core_main
#include "adjoint_core_check.hip"
#undef main

struct Dom {
    FillArgs a;
    const Tab *T;
};

static void ref_value(const Dom &D, const int *iv, double *v) {
    const FillArgs &a = D.a;
    bool np = false;
    int s[3];
    for (int d = 0; d < 3; ++d) {
        const bool o = iv[d] < 0 || iv[d] >= a.n[d];
        if (o && !a.periodic[d]) np = true;
        s[d] = a.periodic[d] ? ((iv[d] % a.n[d]) + a.n[d]) % a.n[d] : iv[d];
    }
    if (!np) {
        for (int c = 0; c < NV; ++c) v[c] = a.s(s[0], s[1], s[2], c);
        return;
    }
    for (int d = 0; d < 3; ++d) {
        if (a.periodic[d]) continue;
        const int side = iv[d] < 0 ? 0 : (iv[d] >= a.n[d] ? 1 : -1);
        if (side < 0) continue;
        const int bc = side == 0 ? a.lo_bc[d] : a.hi_bc[d];
        if (bc == MF_BC_EXT_DIR) continue;
        int m[3] = {iv[0], iv[1], iv[2]};
        const bool refl = bc == MF_BC_WALL;
        if (!refl) m[d] = side == 0 ? 0 : a.n[d] - 1;
        else m[d] = side == 0 ? -iv[d] - 1 : 2 * (a.n[d] - 1) - iv[d] + 1;
        ref_value(D, m, v);
        for (int c = 0; c < NV; ++c)
            if (refl && ((c >= RHOU && c <= RHOW) || (c >= VELX && c <= VELZ))) v[c] = -v[c];
    }
    double x[3];
    for (int d = 0; d < 3; ++d) x[d] = a.prob_lo[d] + (iv[d] + 0.5) * a.dx[d];
    for (int d = 0; d < 3; ++d) {
        if (a.periodic[d]) continue;
        int sgn = 0, m[3] = {iv[0], iv[1], iv[2]};
        if (a.lo_bc[d] == MF_BC_EXT_DIR && iv[d] < 0) { sgn = 1; m[d] = 0; }
        else if (a.hi_bc[d] == MF_BC_EXT_DIR && iv[d] >= a.n[d]) { sgn = -1; m[d] = a.n[d] - 1; }
        if (!sgn) continue;
        double si[NV], se[NV];
        ref_value(D, m, si);
        for (int c = 0; c < NV; ++c) se[c] = 0.0;
        P::externalbc(*D.T, x, si, se, d, sgn, 0.0);
        for (int c = 0; c < NV; ++c) v[c] = se[c];
    }
}

template <class F>
static void each_ghost(const int *n, F f) {
    const int G = MF_NGROW;
    const int64_t PX = n[0] + 2 * G, PY = n[1] + 2 * G;
    const int64_t nzs = 2 * G * PX * PY, nys = (int64_t)n[2] * 2 * G * PX, nxs = (int64_t)n[2] * n[1] * 2 * G;
    for (int64_t q = 0; q < nzs + nys + nxs; ++q) {
        int iv[3];
        ghost_cell(q, nzs, nys, (int)PX, (int)PY, n[0], n[1], n[2], iv);
        f(iv);
    }
}

// boundary code of (direction, combination): 0 periodic, else lo and hi of {foextrap, ext_dir, wall}
static void set_dir(FillArgs &a, int d, int combo) {
    static const int codes[3] = {MF_BC_FOEXTRAP, MF_BC_EXT_DIR, MF_BC_WALL};
    a.periodic[d] = combo == 0;
    a.lo_bc[d] = combo == 0 ? MF_BC_PERIODIC : codes[(combo - 1) % 3];
    a.hi_bc[d] = combo == 0 ? MF_BC_PERIODIC : codes[(combo - 1) / 3];
}

int main() {
    Tab T = make_tab();
    static const int sizes[8][3] = {{1, 2, 3}, {2, 3, 1}, {3, 1, 2}, {1, 1, 1}, {2, 2, 2}, {3, 3, 3}, {4, 3, 5}, {7, 1, 4}};
    long cells = 0, bad = 0, count = 0;
    for (int z = 0; z < 8; ++z) {
        const int *n = sizes[z];
        HostLevel L(n[0], n[1], n[2]);
        for (int combo = 0; combo < 1000; ++combo) {
            Dom D;
            memset(&D.a, 0, sizeof(D.a));
            D.T = &T;
            D.a.s = L.v;
            for (int d = 0; d < 3; ++d) {
                D.a.n[d] = n[d];
                D.a.dx[d] = 1e-3 * (d + 1);
                D.a.prob_lo[d] = -0.5 * d;
            }
            set_dir(D.a, 0, combo % 10);
            set_dir(D.a, 1, (combo / 10) % 10);
            set_dir(D.a, 2, combo / 100);
            // ghost cells hold NaN: a rule that reads one before it is filled shows
            for (double &v : L.a) v = NAN;
            for (int k = 0; k < n[2]; ++k)
                for (int j = 0; j < n[1]; ++j)
                    for (int i = 0; i < n[0]; ++i) {
                        double S[NV];
                        random_cell(T, S, 0.5);
                        for (int c = 0; c < NV; ++c) L.v(i, j, k, c) = S[c];
                    }
            each_ghost(n, [&](const int *iv) {
                double want[NV], got[NV];
                ref_value(D, iv, want);
                fill_value<P, true>(D.a, iv, T, 0.0, got);
                ++cells;
                if (memcmp(want, got, sizeof(want)) != 0) {
                    if (++bad <= 5) printf("value: n %d,%d,%d combo %d cell %d,%d,%d differs\n", n[0], n[1], n[2], combo, iv[0], iv[1], iv[2]);
                }
            });
            // the whole array filled, then the adjoint on a few combinations
            each_ghost(n, [&](const int *iv) { fill_cell<P, true>(D.a, iv, T, 0.0); });
            for (double v : L.a)
                if (!(v == v)) { if (++bad <= 5) printf("n %d,%d,%d combo %d: a cell left unfilled\n", n[0], n[1], n[2], combo); break; }
            if (combo % 37 != z) continue;
            ++count;
            std::vector<double> lam(L.a.size()), dir(L.a.size(), 0.0), base = L.a;
            for (double &l : lam) l = urand(-1.0, 1.0);
            for (int k = 0; k < n[2]; ++k)
                for (int j = 0; j < n[1]; ++j)
                    for (int i = 0; i < n[0]; ++i)
                        for (int c = 0; c < NV; ++c) {
                            const size_t q = (size_t)(L.v.off(i, j, k) + (int64_t)c * L.v.ns);
                            dir[q] = urand(-1.0, 1.0) * fabs(base[q]) * 1e-6;
                        }
            double fd = 0.0;
            std::vector<double> up;
            for (int s = 1; s >= -1; s -= 2) {
                for (size_t q = 0; q < base.size(); ++q) L.a[q] = base[q] + s * dir[q];
                each_ghost(n, [&](const int *iv) { fill_cell<P, true>(D.a, iv, T, 0.0); });
                if (s > 0) up = L.a;
            }
            for (size_t q = 0; q < base.size(); ++q) fd += lam[q] * (up[q] - L.a[q]) * 0.5;
            L.a = base;
            double ad = 0.0, invelb = 0.0;
            std::vector<double> fold = lam;
            each_ghost(n, [&](const int *iv) {
                int c[3] = {iv[0], iv[1], iv[2]};
                double l[NV];
                const int64_t from = L.v.off(c[0], c[1], c[2]);
                for (int m = 0; m < NV; ++m) { l[m] = lam[from + m * L.v.ns]; fold[from + m * L.v.ns] = 0.0; }
                R::fill_rev(T, D.a, c, l, invelb);
                for (int d = 0; d < 3; ++d) if (c[d] < 0 || c[d] >= n[d]) ++bad;
                const int64_t to = L.v.off(c[0], c[1], c[2]);
                for (int m = 0; m < NV; ++m) fold[to + m * L.v.ns] += l[m];
            });
            double scale = 0.0;
            for (size_t q = 0; q < base.size(); ++q) { ad += fold[q] * dir[q]; scale += fabs(fold[q] * dir[q]); }
            // central differences over a relative step of 1e-6: truncation ~1e-12,
            // rounding ~1e-16/1e-6 of the terms
            if (fabs(ad - fd) > 1e-8 * scale) {
                if (++bad <= 10) printf("adjoint: n %d,%d,%d combo %d: %.12e fd %.12e\n", n[0], n[1], n[2], combo, ad, fd);
            }
        }
    }
    printf("fill: %ld ghost cells, %ld adjoints, %ld wrong\n%s\n", cells, count, bad, bad ? "FAILED" : "PASSED");
    return bad ? 1 : 0;
}
