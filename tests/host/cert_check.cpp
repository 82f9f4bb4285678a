// Host build of the device headers: the FP32 certificates of the facet lists
// (cert_write, cert_class) against the FP64 point-triangle test they stand
// for, on facets from regular to needles and beyond the certificate's range,
// points at every distance, across the eps limit and at the facets' edges and
// corners; the certified runs (SampleGen::run_left / run_at, and a triangle
// whose corners one facet certifies) against every sample in between; and
// in_envelope_cert against the FP64 test of every listed facet.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <vector>

#include "twg_bvh.hpp"

using namespace twg;

static long failures = 0;
#define CHECK(c, ...)                 \
    do {                              \
        if (!(c)) {                   \
            if (++failures <= 20) printf(__VA_ARGS__); \
        }                             \
    } while (0)

static std::mt19937_64 rng(7);
static double U(double a, double b) { return std::uniform_real_distribution<double>(a, b)(rng); }
static double LU(double a, double b) { return std::exp(U(std::log(a), std::log(b))); }
static V3<double> unit()
{
    std::normal_distribution<double> n;
    return normalize(mk3(n(rng), n(rng), n(rng)));
}

static double d2(const double* t, V3<double> p)
{
    V3<double> cp;
    return point_tri_d2<double, false>(p, ld3(t), ld3(t + 3), ld3(t + 6), cp);
}

struct Setup {
    double eps, eps2, amax, d;
    V3<double> center;
    double half;
    CertFrame F;
};

static Setup setup(double scale, double at)
{
    Setup S;
    S.eps = scale * LU(1e-4, 1.0);
    S.eps2 = S.eps * S.eps;
    S.d = S.eps * LU(0.5, 4.0);
    S.center = mulv(unit(), at);
    S.half = S.eps * LU(1.0, 3e3);
    const double lo[3] = {S.center.x - S.half, S.center.y - S.half, S.center.z - S.half};
    const double hi[3] = {S.center.x + S.half, S.center.y + S.half, S.center.z + S.half};
    S.amax = at + S.half;
    S.F = cert_frame(lo, hi, S.amax, S.eps2, S.d);
    return S;
}

static void facet(const Setup& S, double* t)
{
    // a facet near the box's middle: size, aspect and angle over wide ranges
    const V3<double> a = S.center + mulv(unit(), U(0, S.half));
    const V3<double> e = unit();
    const double len0 = S.eps * LU(1e-2, 1e6), h = len0 * LU(1e-9, 2.0);
    const V3<double> w = normalize(cross(e, unit()));
    const V3<double> b = a + mulv(e, len0), c = a + mulv(e, len0 * U(-0.5, 1.5)) + mulv(w, h);
    const V3<double> v[3] = {a, b, c};
    const int r = (int)(rng() % 3);
    for (int k = 0; k < 3; ++k) {
        t[3 * k] = v[(k + r) % 3].x;
        t[3 * k + 1] = v[(k + r) % 3].y;
        t[3 * k + 2] = v[(k + r) % 3].z;
    }
    if (rng() % 16 == 0) std::memcpy(t + 3, t, 24);  // degenerate
}

static V3<double> near_point(const Setup& S, const double* t)
{
    // a point of the facet (inside, edge or corner) pushed to about eps
    double u = U(0, 1), v = U(0, 1);
    if (u + v > 1) u = 1 - u, v = 1 - v;
    switch (rng() % 4) {
    case 0: u = 0; break;
    case 1: u = (double)(rng() % 2), v = u == 0 ? (double)(rng() % 2) : 0; break;
    default: break;
    }
    const V3<double> a = ld3(t), b = ld3(t + 3), c = ld3(t + 6);
    V3<double> p = a + mulv(b - a, u) + mulv(c - a, v);
    V3<double> n = normalize(cross(b - a, c - a));
    if (rng() % 2) n = unit();
    double dist = S.eps * U(0, 3);
    if (rng() % 2) dist = S.eps * (1 + U(-1, 1) * LU(1e-9, 1e-2));
    return p + mulv(n, dist);
}

static bool inside_box(const Setup& S, V3<double> p)
{
    return std::fabs(p.x - S.center.x) <= S.half && std::fabs(p.y - S.center.y) <= S.half &&
           std::fabs(p.z - S.center.z) <= S.half;
}

int main()
{
    long n = 0, in = 0, out = 0, plain = 0, plain_sure = 0, tris = 0, runs = 0, run_samples = 0, lists = 0, past = 0, past_hint = 0,
         ends = 0;
    for (int s = 0; s < 4000; ++s) {
        const double scale = s % 5 == 0 ? LU(1e-12, 1e9) : 1.0;
        const Setup S = setup(scale, s % 3 == 0 ? scale * LU(1, 1e9) : scale * U(0, 2));
        std::vector<double> T(9 * 12);
        std::vector<float> C(kCertFloats * 12);
        for (int f = 0; f < 12; ++f) {
            facet(S, &T[9 * f]);
            cert_write(&C[kCertFloats * f], &T[9 * f], S.F, S.eps2);
        }
        for (int f = 0; f < 12; ++f)
            for (int k = 0; k < 60; ++k) {
                V3<double> p = near_point(S, &T[9 * f]);
                if (!inside_box(S, p)) p = S.center + mulv(unit(), U(0, S.half));
                const int r = cert_class(&C[kCertFloats * f], cert_local(S.F, p), S.F);
                const double dd = d2(&T[9 * f], p);
                CHECK(r != 1 || dd <= S.eps2, "set %d: certified in at %.17g of eps2 %.17g\n", s, dd, S.eps2);
                CHECK(r != -1 || dd > S.eps2, "set %d: certified out at %.17g of eps2 %.17g\n", s, dd, S.eps2);
                ++n;
                in += r == 1;
                out += r == -1;
                if (scale == 1.0 && s % 3 && S.half < 200 * S.eps &&
                    len2(ld3(&T[9 * f + 3]) - ld3(&T[9 * f])) < 1e6 * S.eps2 && std::fabs(std::sqrt(dd) - S.eps) > 0.05 * S.eps &&
                    len2(cross(ld3(&T[9 * f + 3]) - ld3(&T[9 * f]), ld3(&T[9 * f + 6]) - ld3(&T[9 * f]))) >
                        0.01 * len2(ld3(&T[9 * f + 3]) - ld3(&T[9 * f])) * len2(ld3(&T[9 * f + 6]) - ld3(&T[9 * f]))) {
                    ++plain;
                    plain_sure += r != 0;
                }
            }
        // the whole list's decision, with and without a hint, on lists up to
        // the masks' end: few facets hold p, on either side of position 64
        const int lens[] = {1 + (int)(rng() % 12), 63, 64, 65, 80, 92, 128};
        const int nl = lens[s % 7];
        struct Node { int32_t leaf, pad; };
        std::vector<Node> L(nl);
        std::vector<double> LT(9 * nl);
        std::vector<float> LC(kCertFloats * nl);
        for (int f = 0; f < nl; ++f) {
            L[f] = {f, 0};
            if (f < 12) std::memcpy(&LT[9 * f], &T[9 * f], 72);
            else facet(S, &LT[9 * f]);
        }
        for (int f = 0; f < nl; ++f)  // the twelve the points lie about at places of the whole list
            if (f < 12) {
                const int g = (int)(rng() % nl);
                for (int q = 0; q < 9; ++q) std::swap(LT[9 * f + q], LT[9 * g + q]);
            }
        for (int f = 0; f < nl; ++f) cert_write(&LC[kCertFloats * f], &LT[9 * f], S.F, S.eps2);
        BvhWalk W;
        std::memset(&W, 0, sizeof W);
        W.tri = LT.data();
        for (int k = 0; k < 60; ++k) {
            V3<double> p = near_point(S, &T[9 * (rng() % 12)]);
            if (!inside_box(S, p)) continue;
            bool ref = false, low = false, high = false;
            uint64_t mask[2] = {0, 0};
            for (int f = 0; f < nl; ++f)
                if (rng() % 8) {
                    mask[f / 64] |= 1ull << (f % 64);
                    const bool holds = d2(&LT[9 * f], p) <= S.eps2;
                    ref = ref || holds;
                    (f < 64 ? low : high) |= holds;
                }
            int hl = -1;
            if (rng() % 2) hl = (int)(rng() % nl);  // (a hint counts outside the mask too)
            const int hint = hl;
            ref = ref || (hint >= 0 && d2(&LT[9 * hint], p) <= S.eps2);
            bool sure = false;
            const bool got = in_envelope_cert(W, L.data(), LC.data(), nl, mask, p, S.F, S.eps2, hl, sure);
            CHECK(got == ref, "set %d: list of %d, decision %d, FP64 %d\n", s, nl, got, ref);
            CHECK(!got || (hl >= 0 && hl < nl && d2(&LT[9 * hl], p) <= S.eps2), "set %d: the facet left does not hold p\n", s);
            ++lists;
            past += high && !low;
            past_hint += hint >= 64;
            if (nl == 64) {  // the word past the list's end is not read
                mask[1] = ~0ull;
                int h2 = hint;
                CHECK(in_envelope_cert(W, L.data(), LC.data(), nl, mask, p, S.F, S.eps2, h2, sure) == ref,
                      "set %d: a list that ends a word reads past it\n", s);
                ++ends;
            }
        }
        if (!S.F.runs) continue;
        // triangles near the facets, their samples between certified ones
        for (int k = 0; k < 12; ++k) {
            const double* t = &T[9 * k];
            const float* c = &C[kCertFloats * k];
            const double size = std::min(S.half, 40 * S.d) * LU(0.003, 1);
            V3<double> p[3];
            const V3<double> m = near_point(S, t);
            for (int j = 0; j < 3; ++j) {
                p[j] = m + mulv(unit(), size);
                // into the facet's plane, then off it
                const V3<double> un = normalize(cross(ld3(t + 3) - ld3(t), ld3(t + 6) - ld3(t)));
                p[j] = p[j] - mulv(un, dot(p[j] - ld3(t), un)) + mulv(un, S.eps * U(-1, 1));
            }
            bool fits = true, all = true;
            for (int j = 0; j < 3; ++j) {
                fits = fits && inside_box(S, p[j]);
                all = all && cert_class(c, cert_local(S.F, p[j]), S.F) > 0;
            }
            if (!fits) continue;
            tris += all;
            SampleGen g;
            g.init(p[0], p[1], p[2], S.d);
            V3<double> q;
            while (g.next(q)) {
                if (all) CHECK(d2(t, q) <= S.eps2, "set %d: a sample of a certified triangle is out\n", s);
                const int64_t left = g.run_left(1 + (int64_t)(rng() % 40));
                if (left < 1) continue;
                const V3<double> e = g.run_at(left);
                SampleGen h = g;
                V3<double> z = q;
                bool held = cert_class(c, cert_local(S.F, q), S.F) > 0 && cert_class(c, cert_local(S.F, e), S.F) > 0;
                for (int64_t i = 0; i < left; ++i) {
                    const bool more = h.next(z);
                    CHECK(more && h.phase == g.phase, "set %d: the run ends early\n", s);
                    if (held) {
                        CHECK(d2(t, z) <= S.eps2, "set %d: a sample of a certified run is out\n", s);
                        ++run_samples;
                    }
                }
                runs += held;
                CHECK(z.x == e.x && z.y == e.y && z.z == e.z, "set %d: run_at is not next's sample\n", s);
                double rec[kFaceRec];
                if (g.phase != 9) {
                    SampleGen g0;
                    g0.init(p[0], p[1], p[2], S.d);
                    g0.store(rec);
                    SampleGenC<const double*> gc;
                    gc.load(rec, S.d);
                    gc.phase = g.phase; gc.k = g.k; gc.N = g.N; gc.N1 = g.N1; gc.m = g.m; gc.rowv = g.rowv;
                    const V3<double> ec = gc.run_at(left);
                    CHECK(gc.run_left(left) == left && ec.x == e.x && ec.y == e.y && ec.z == e.z,
                          "set %d: the stored-record run differs\n", s);
                }
            }
        }
    }
    printf("%ld facet decisions (%ld certified in, %ld out), %ld lists (%ld held past position 64 alone, %ld hints past it, %ld at a word's end), %ld certified triangles, %ld runs (%ld "
           "samples); ordinary facets off the limit: %ld of %ld certified\n",
           n, in, out, lists, past, past_hint, ends, tris, runs, run_samples, plain_sure, plain);
    CHECK(in > 100000 && out > 100000 && tris > 500 && runs > 5000 && lists > 50000 && past > 5000 && past_hint > 5000 && ends > 5000, "too few cases\n");
    CHECK(plain_sure > 0.8 * plain && plain > 10000, "certificates miss ordinary cases\n");
    printf("%ld failures\n", failures);
    return failures ? 1 : 0;
}
