// Host checks of the walks' box tests (traverse.h, lbvh.h, compiled into this
// test from the same headers): SlabTestQ on quantised nodes and SlabTest4 with
// the same ray, against box intervals in long double.
//   * a box whose interval is not empty is hit, and its near bound does not
//     exceed the interval's (by more than the walk's pruning allows for);
//   * a box that a ray misses by more than the test's stated margins is missed
//     (a test that left every interval unbounded would pass the first check).
// Usage: slab_check EXTENT OFFSET DIRSCALE TMAX SEED COUNT.  Prints "ok" on success.
#include "../../mray_amd/csrc/traverse.h"

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>

using namespace mray;

namespace
{
typedef long double LD;
int fails = 0;
struct Box { float lo[3], hi[3]; };

// Interval of a box grown by `grow` per axis; false if empty.
bool Interval(const float* o, const float* d, const Box& b, const LD* grow, float tMin, float tMax, LD& n, LD& f)
{
    n = tMin;
    f = tMax;
    for(int k = 0; k < 3; k++)
    {
        const LD lo = LD(b.lo[k]) - grow[k] - o[k], hi = LD(b.hi[k]) + grow[k] - o[k];
        if(d[k] == 0.0f)
        {
            if(lo > 0 || hi < 0) return false;
            continue;
        }
        const LD a = lo / d[k], c = hi / d[k];
        n = std::fmax(n, std::fmin(a, c));
        f = std::fmin(f, std::fmax(a, c));
    }
    return n <= f;
}
} // namespace

int main(int argc, char** argv)
{
    if(argc < 7) { std::printf("usage: slab_check extent offset dirscale tmax seed count\n"); return 2; }
    const double extent = std::atof(argv[1]), offset = std::atof(argv[2]), scale = std::atof(argv[3]);
    const float tMax = float(std::atof(argv[4]));
    std::mt19937_64 rng(std::strtoull(argv[5], nullptr, 10));
    const int count = std::atoi(argv[6]);
    std::uniform_real_distribution<double> uni(0.0, 1.0);
    auto pick = [&](int n) { return int(rng() % uint64_t(n)); };
    const float tiny[8] = {0.0f, -0.0f, 1e-38f, -1e-35f, 1e-28f, -1e-22f, 1e-17f, -1e-9f};
    long hits = 0, misses = 0;
    for(int it = 0; it < count; it++)
    {
        // a node's four boxes, one slot empty now and then, flat boxes among them
        BNode4 node;
        Box box[4];
        float* lo[3] = {node.lox, node.loy, node.loz};
        float* hi[3] = {node.hix, node.hiy, node.hiz};
        const int empty = (it % 5 == 0) ? pick(4) : -1;
        float coord[3] = {0, 0, 0}, L[3], H[3];
        for(int a = 0; a < 3; a++) { L[a] = INFINITY; H[a] = -INFINITY; }
        for(int k = 0; k < 4; k++)
        {
            node.child[k] = (k == empty) ? kInvalid : uint32_t(k + 1);
            for(int a = 0; a < 3; a++)
            {
                double p = (uni(rng) - 0.5) * extent, w = (k == 0) ? extent : uni(rng) * extent * 0.3;
                if(pick(6) == 0) w = 0.0;
                if(pick(6) == 0) p = -0.5 * w;
                box[k].lo[a] = float(p + offset);
                box[k].hi[a] = std::fmax(float(p + w + offset), box[k].lo[a]);
                lo[a][k] = (k == empty) ? INFINITY : box[k].lo[a];
                hi[a][k] = (k == empty) ? -INFINITY : box[k].hi[a];
                if(k == empty) continue;
                L[a] = std::fmin(L[a], box[k].lo[a]);
                H[a] = std::fmax(H[a], box[k].hi[a]);
                coord[a] = std::fmax(coord[a], std::fmax(std::fabs(L[a]), std::fabs(H[a])));
            }
        }
        const QNode4 q = QuantizeNode(node);
        // a ray: components zero, tiny or ordinary; origins inside, on planes, outside
        float o[3], d[3];
        const int target = (empty == 0) ? 1 : 0;
        for(int a = 0; a < 3; a++)
        {
            const int w = pick(4), k = (pick(2) == 0) ? target : ((pick(4) + 1) % 4);
            const Box& b = box[(k == empty) ? target : k];
            o[a] = (w == 0) ? b.lo[a] : (w == 1) ? b.hi[a] : (w == 2) ? float(b.lo[a] + (b.hi[a] - b.lo[a]) * uni(rng))
                 : float((uni(rng) - 0.5) * 3.0 * extent + offset);
            d[a] = (pick(2) == 0) ? tiny[pick(8)] : float(2.0 * uni(rng) - 1.0);
        }
        if(pick(3) != 0)
        {
            // point it at the first box
            const int a = pick(3);
            const double to = 0.5 * (double(box[target].lo[a]) + box[target].hi[a]) - o[a];
            d[a] = (to < 0) ? -1.0f : 1.0f;
        }
        for(int a = 0; a < 3; a++) d[a] = float(d[a] * scale);
        const float m = std::fmax(std::fabs(d[0]), std::fmax(std::fabs(d[1]), std::fabs(d[2])));
        if(m == 0.0f) continue;
        const V3 dir = {d[0], d[1], d[2]};
        // the caller's form, and the renderers' for unit vectors
        const float maxInv = SceneMaxInv(std::fmax(coord[0], std::fmax(coord[1], coord[2])));
        const bool unit = m >= 0.5f && m < 2.0f && it % 2 == 0;
        const RayReach reach = unit ? kUnitReach : CallerReach(dir, tMax, maxInv);
        const RayQ r = MakeRayQ(V3{o[0], o[1], o[2]}, dir, reach);
        for(int kind = 0; kind < 2; kind++)
        {
            float tn[4];
            uint4 child;
            if(kind == 0) SlabTestQ(&q, r, 0.0f, tMax, tn, child);
            else SlabTest4(&node, r, 0.0f, tMax, tn, child);
            for(int k = 0; k < 4; k++)
            {
                if(k == empty) continue;
                LD n, f;
                const LD none[3] = {0, 0, 0};
                const bool hit = Interval(o, d, box[k], none, 0.0f, tMax, n, f) && n <= 1e14L / std::fmin(1.0f, m);
                if(hit)
                {
                    hits++;
                    if(tn[k] == INFINITY || LD(tn[k]) > n * (1.0L + 4e-7L))
                        if(fails++ < 10)
                            std::printf("FAIL: kind %d box [%g %g] [%g %g] [%g %g] o %g %g %g d %g %g %g: interval %Lg %Lg, near %g\n",
                                        kind, box[k].lo[0], box[k].hi[0], box[k].lo[1], box[k].hi[1], box[k].lo[2], box[k].hi[2],
                                        o[0], o[1], o[2], d[0], d[1], d[2], n, f, tn[k]);
                    continue;
                }
                LD grow[3];
                // (directions so short that the scene's size caps their reciprocal may be loose)
                bool bounded = LD(reach.maxInv) * m >= 1e19L;
                for(int a = 0; a < 3; a++)
                {
                    const LD ext = LD(H[a]) - L[a];
                    grow[a] = 0.02L * ext + 2e-6L * (coord[a] + std::fabs(LD(o[a]))) + 2.0L * reach.reach / reach.maxInv + 1e-26L;
                    bounded = bounded && coord[a] + 6 * ext < 1e18L;
                }
                if(bounded && !Interval(o, d, box[k], grow, 0.0f, tMax, n, f))
                {
                    misses++;
                    if(tn[k] != INFINITY)
                        if(fails++ < 10)
                            std::printf("FAIL: kind %d box [%g %g] [%g %g] [%g %g] o %g %g %g d %g %g %g is missed, near %g\n",
                                        kind, box[k].lo[0], box[k].hi[0], box[k].lo[1], box[k].hi[1], box[k].lo[2], box[k].hi[2],
                                        o[0], o[1], o[2], d[0], d[1], d[2], tn[k]);
                }
            }
        }
    }
    std::printf("%ld hits, %ld misses\n", hits, misses);
    if(hits < count / 4) { std::printf("FAIL: too few hits\n"); fails++; }
    std::printf(fails ? "%d failures\n" : "ok\n", fails);
    return fails ? 1 : 0;
}
