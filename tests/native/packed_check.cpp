// Host-side check of the packed nodes (no GPU), run by tests/test_packed_nodes.py: the kernels' own
// box arithmetic (lightmetrica_amd/csrc/boxes.hpp) on the trees of the builder and on nodes with
// extents from 0 and denormal to 1e7.
//
//   packed_check tree <num_triangles> <seed> <max_leaf> | nodes <seed>
//
// Checks:
//   1. place_leaves gives every record one place, leaves of two or more on an even one, with and
//      without padding;
//   2. a packed child's planes lie outside the built ones (exact arithmetic), on the lowest plane or
//      by the margin; empty slots are inverted one-record leaves;
//   3. whatever ray and interval the built box's test accepts, the packed test accepts, and an entry
//      is not taken off the stack by a hit that comes after it (hit_order): rays from inside, from
//      faces, at corners and edges, from 1 to 1e6 extents away, in planes and with denormal direction
//      components, with reciprocals 1 ulp off, forward and behind the origin.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>

#include "../../lightmetrica_amd/csrc/boxes.hpp"

using namespace lmgpu;

static int failures = 0;
#define CHECK(c, ...)                                   \
    do {                                                \
        if (!(c)) {                                     \
            if (failures < 20) std::printf(__VA_ARGS__); \
            failures++;                                 \
        }                                               \
    } while (0)

static std::mt19937_64 rng;
static double U() { return std::uniform_real_distribution<double>(0.0, 1.0)(rng); }

static float safe_rcp(float d) {  // the hardware's, within 1 ulp
    const float r = 1.f / (std::fabs(d) > 1e-30f ? d : std::copysign(1e-30f, d));
    const unsigned pick = unsigned(rng() % 3);
    return pick == 0 ? r : std::nextafter(r, pick == 1 ? INFINITY : -INFINITY);
}

static void check_places(WideBVH w, bool pad) {
    if (!pad) w.num_leaves = kMaxLeafFirst;  // as if the padded array outgrew the 27-bit offsets
    const uint32_t n = place_leaves(w);
    std::vector<int> used(n, 0);
    size_t records = 0;
    for (const Node4& nd : w.nodes)
        for (int i = 0; i < 4; i++) {
            if (nd.child[i] == kEmptyChild || !(nd.child[i] & kLeafBit)) continue;
            const uint32_t count = ((nd.child[i] >> 27) & 0xfu) + 1u;
            CHECK(!pad || count == 1 || nd.pad[i] % 2 == 0, "leaf of %u records at %u\n", count, nd.pad[i]);
            CHECK(nd.pad[i] + count <= n, "leaf at %u + %u of %u\n", nd.pad[i], count, n);
            for (uint32_t k = nd.pad[i]; k < std::min(nd.pad[i] + count, n); k++) used[k]++;
            records += count;
        }
    CHECK(records == w.tris.size(), "%zu records placed of %zu\n", records, w.tris.size());
    for (uint32_t k = 0; k < n; k++) CHECK(used[k] <= 1, "place %u used %d times\n", k, used[k]);
    CHECK(pad || n == w.tris.size(), "%u places without padding\n", n);
}

static uint64_t tested = 0, accepted = 0;

static void check_ray(const Node4& n, const NodeQ& q, int i, const float o[3], const float d[3], float tmin, float tmax) {
    const Slab s = make_slab(o[0], o[1], o[2], safe_rcp(d[0]), safe_rcp(d[1]), safe_rcp(d[2]));
    const PackedAxis x = packed_axis(q.origin[0], q.step[0], q.planes[0][0], q.planes[0][1], s.ix, s.nx, s.fx);
    const PackedAxis y = packed_axis(q.origin[1], q.step[1], q.planes[1][0], q.planes[1][1], s.iy, s.ny, s.fy);
    const PackedAxis z = packed_axis(q.origin[2], q.step[2], q.planes[2][0], q.planes[2][1], s.iz, s.nz, s.fz);
    for (int rep = 0; rep < 2; rep++) {
        float tn, tf, pn, pf;
        box_span(s, n.lo_x[i], n.hi_x[i], n.lo_y[i], n.hi_y[i], n.lo_z[i], n.hi_z[i], tmin, tmax, tn, tf);
        tested++;
        if (!(tn <= widened(tf, kBoxRobustExact))) return;
        accepted++;
        // As it is, and with the nearest hit so far just behind this child's earliest one.
        const float near = rep == 0 ? tmax : std::nextafter(tn * kOrderScale, INFINITY);
        if (!(near <= tmax)) return;
        packed_span(x, y, z, i, tmin, near, pn, pf);
        CHECK(pn <= widened(pf, kBoxRobust) && !(pn > fmaxf(near * kBoxRobust, 0.f)),
              "child %d entered [%.9g, %.9g] (nearest %.9g), packed [%.9g, %.9g]: o %g %g %g d %g %g %g\n", i, double(tn),
              double(tf), double(near), double(pn), double(pf), double(o[0]), double(o[1]), double(o[2]), double(d[0]),
              double(d[1]), double(d[2]));
    }
}

static void check_node(const Node4& n, int rays) {
    const NodeQ q = pack_node(n);
    const float* lo[3] = {n.lo_x, n.lo_y, n.lo_z};
    const float* hi[3] = {n.hi_x, n.hi_y, n.hi_z};
    double ext = 0.0;
    for (int a = 0; a < 3; a++)
        for (int i = 0; i < 4; i++) {
            const unsigned ql = q.planes[a][0] >> (8 * i) & 255u, qh = q.planes[a][1] >> (8 * i) & 255u;
            if (n.child[i] == kEmptyChild) {
                CHECK(ql == 255u && qh == 0u && q.child[i] == kLeafBit, "empty slot %d: planes %u %u\n", i, ql, qh);
                continue;
            }
            CHECK(q.child[i] == n.child[i], "child word %d\n", i);
            const long double l = (long double)q.origin[a] + (long double)q.step[a] * ql;
            const long double h = (long double)q.origin[a] + (long double)q.step[a] * qh;
            const long double margin = (long double)q.step[a] * (kPlaneMargin * 0.999);
            CHECK(ql == 0u ? l <= lo[a][i] : l + margin <= lo[a][i], "axis %d child %d: lo %.9g, packed %.12Lg\n", a, i,
                  double(lo[a][i]), l);
            CHECK(q.step[a] == 0.f ? h == hi[a][i] : h - margin >= hi[a][i], "axis %d child %d: hi %.9g, packed %.12Lg\n",
                  a, i, double(hi[a][i]), h);
            ext = std::max(ext, double(hi[a][i]) - double(lo[a][i]));
        }
    for (int i = 0; i < 4; i++) {
        if (n.child[i] == kEmptyChild) continue;
        for (int r = 0; r < rays; r++) {
            // A target in, on a face, an edge or a corner of the child; an origin in the box, on a face
            // or away by 1 to 1e6 extents.
            float t[3], o[3], d[3];
            const int where = int(rng() % 4), from = int(rng() % 3);
            const double away = std::max(ext, 1e-20) * std::pow(10.0, 6.0 * U());
            for (int a = 0; a < 3; a++) {
                const double w = double(hi[a][i]) - double(lo[a][i]);
                const bool on = int(rng() % 4) < where;
                t[a] = on ? (rng() & 1 ? hi[a][i] : lo[a][i]) : float(lo[a][i] + U() * w);
                const bool face = from == 1 && rng() % 2;
                o[a] = face ? (rng() & 1 ? hi[a][i] : lo[a][i])
                            : from < 2 ? float(lo[a][i] + U() * w) : float(t[a] + (2.0 * U() - 1.0) * away);
                if (rng() % 16 == 0) o[a] = t[a];  // in a plane with the target
            }
            // Past the target by what the robust factor forgives, or nearly.
            if (from == 2 && rng() % 2)
                for (int a = 0; a < 3; a++) t[a] = float(t[a] + away * 1.2e-6 * (U() - 0.5));
            double len = 0.0, v[3];
            for (int a = 0; a < 3; a++) {
                v[a] = double(t[a]) - double(o[a]);
                if (from < 2 && rng() % 4) v[a] = 2.0 * U() - 1.0;
                len += v[a] * v[a];
            }
            len = std::sqrt(len);
            if (!(len > 0.0)) continue;
            for (int a = 0; a < 3; a++) {
                d[a] = float(v[a] / len);
                if (rng() % 32 == 0) d[a] = rng() & 1 ? 0.f : -1e-40f;
            }
            const float tmin = rng() % 2 ? 0.f : float(len * U());
            check_ray(n, q, i, o, d, tmin, rng() % 2 ? 3.4028234e38f : float(len * (0.5 + U())));
            // The same behind the origin.
            for (float& x : d) x = -x;
            check_ray(n, q, i, o, d, rng() % 2 ? -3.4028234e38f : float(-len * (0.5 + U())), -tmin);
        }
    }
}

int main(int argc, char** argv) {
    if (argc > 4 && !std::strcmp(argv[1], "tree")) {
        const uint32_t nt = uint32_t(std::atoi(argv[2]));
        rng.seed(uint64_t(std::atoi(argv[3])));
        std::vector<float> P(9 * size_t(nt));
        std::vector<uint32_t> F(3 * size_t(nt));
        for (uint32_t t = 0; t < nt; t++) {
            const double s = t % 3 ? 0.05 : 0.5;
            double c[3];
            for (double& x : c) x = U();
            for (int k = 0; k < 9; k++) {
                double x = c[k % 3] + s * (U() - 0.5);
                if (t % 5 == 0) x = std::round(x * 16.0) / 16.0;  // shared planes, flat boxes
                P[9 * size_t(t) + k] = float(x);
            }
            for (int k = 0; k < 3; k++) F[3 * t + k] = 3 * t + k;
        }
        BuildParams bp;
        bp.max_leaf_size = uint32_t(std::atoi(argv[4]));
        WideBVH w;
        std::string err;
        if (!build_wide_bvh(P.data(), 3 * nt, F.data(), nt, bp, w, err)) {
            std::printf("build failed: %s\n", err.c_str());
            return 2;
        }
        check_places(w, true);
        check_places(w, false);
        for (const Node4& n : w.nodes) check_node(n, 400000 / int(w.nodes.size()) + 8);
    } else if (argc > 2 && !std::strcmp(argv[1], "nodes")) {
        rng.seed(uint64_t(std::atoi(argv[2])));
        for (int k = 0; k < 20000; k++) {
            Node4 n{};
            float* lo[3] = {n.lo_x, n.lo_y, n.lo_z};
            float* hi[3] = {n.hi_x, n.hi_y, n.hi_z};
            const int children = 1 + int(rng() % 4);
            const double centre = rng() % 3 ? (2.0 * U() - 1.0) * std::pow(10.0, 7.0 * U() - 3.0) : 0.0;
            for (int a = 0; a < 3; a++) {
                const unsigned kind = unsigned(rng() % 6);
                const double ext = kind == 0 ? 0.0 : kind == 1 ? 1e-42 * U() : std::pow(10.0, 14.0 * U() - 7.0);
                for (int i = 0; i < 4; i++) {
                    const float p = float(centre + ext * U()), r = float(centre + ext * U());
                    lo[a][i] = std::min(p, r);
                    hi[a][i] = std::max(p, r);
                    if (rng() % 4 == 0) hi[a][i] = lo[a][i];
                }
                // Planes on the steps themselves, where only the margin moves them out.
                const float l = *std::min_element(lo[a], lo[a] + children), h = *std::max_element(hi[a], hi[a] + children);
                const double step = double(float((double(h) - double(l)) * (1.0 / 254.9)));
                if (step > 0.0 && rng() % 2)
                    for (int i = 0; i < children; i++) {
                        if (lo[a][i] != l) lo[a][i] = float(l + step * std::round((double(lo[a][i]) - l) / step));
                        if (hi[a][i] != h) hi[a][i] = std::max(lo[a][i], float(l + step * std::round((double(hi[a][i]) - l) / step)));
                    }
            }
            for (int i = 0; i < 4; i++) n.child[i] = i < children ? uint32_t(4 * k + i) : kEmptyChild;
            check_node(n, 40);
        }
    } else {
        std::printf("usage: packed_check tree <triangles> <seed> <leaf> | nodes <seed>\n");
        return 2;
    }
    std::printf("spans %llu, accepted %llu, failures %d\n", (unsigned long long)tested, (unsigned long long)accepted,
                failures);
    std::printf(failures ? "packed_check: FAILED\n" : "packed_check: OK\n");
    return failures ? 1 : 0;
}
