// bbx_shapes.hip -- collider shapes: SDF grids (uploaded or built from a
// triangle mesh on the device), device evaluation of the collider-set rule,
// and the solver's collider list.
#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstring>
#include <mutex>
#include <new>
#include <string>
#include <vector>

#include "bbx_collider.h"

using namespace bbx;

struct bbx_sdf {
    int nodes[3] = {0, 0, 0};
    double origin[3] = {0, 0, 0};
    double spacing[3] = {0, 0, 0};
    float *field = nullptr;  // device, x fastest
};

namespace {

// Routes of a mesh's SDF, by triangles and nodes; whole from_mesh calls in us.
// Up to kSdfFew triangles, or twice that on a grid that leaves the chip idle,
// every pair is evaluated: bounds / all pairs 1 triangle 33 / 30, 8 and 1M nodes
// 157 / 158, 12 and 16k nodes 48 / 42, 12 and 275k 70 / 81.  Up to a triangle per
// lane, one wave has a brick of 4 x 4 x 4 nodes; above, four share it: four /
// one 20 triangles and 730k nodes 181 / 109, 60 and 100k 177 / 140, 320 and 110k
// 178 / 302.
constexpr int kSdfFew = 8;
constexpr long long kSdfFewNodes = 1 << 17;
constexpr int kSdfOneWave = 64;
constexpr int kSdfWaves = 4;

__device__ __forceinline__ double sgn_d(double a) { return a > 0 ? 1.0 : (a < 0 ? -1.0 : 0.0); }
__device__ __forceinline__ double clamp_d(double v, double lo, double hi) {
    return v < lo ? lo : (v > hi ? hi : v);
}

// DistanceTriangle (src/shapes/bvh.cpp:212-242), FP64 without contraction:
// squared distance to triangle abc (edge parameters clamped to [1e-4, 1])
__device__ double tri_dist2(const double *t, double px, double py, double pz) {
#pragma clang fp contract(off)
    const double ax = t[0], ay = t[1], az = t[2], bx = t[3], by = t[4], bz = t[5];
    const double cx = t[6], cy = t[7], cz = t[8];
    const double bax = bx - ax, bay = by - ay, baz = bz - az, pax = px - ax, pay = py - ay, paz = pz - az;
    const double cbx = cx - bx, cby = cy - by, cbz = cz - bz, pbx = px - bx, pby = py - by, pbz = pz - bz;
    const double acx = ax - cx, acy = ay - cy, acz = az - cz, pcx = px - cx, pcy = py - cy, pcz = pz - cz;
    // nor = ba x ac
    const double nx = bay * acz - baz * acy, ny = baz * acx - bax * acz, nz = bax * acy - bay * acx;
    // (e x nor) . p_e for the three edges
    const double s0 = (bay * nz - baz * ny) * pax + (baz * nx - bax * nz) * pay + (bax * ny - bay * nx) * paz;
    const double s1 = (cby * nz - cbz * ny) * pbx + (cbz * nx - cbx * nz) * pby + (cbx * ny - cby * nx) * pbz;
    const double s2 = (acy * nz - acz * ny) * pcx + (acz * nx - acx * nz) * pcy + (acx * ny - acy * nx) * pcz;
    if (sgn_d(s0) + sgn_d(s1) + sgn_d(s2) < 2.0) {
        const double t0 = clamp_d((bax * pax + bay * pay + baz * paz) / (bax * bax + bay * bay + baz * baz), 0.0001, 1.0);
        const double t1 = clamp_d((cbx * pbx + cby * pby + cbz * pbz) / (cbx * cbx + cby * cby + cbz * cbz), 0.0001, 1.0);
        const double t2 = clamp_d((acx * pcx + acy * pcy + acz * pcz) / (acx * acx + acy * acy + acz * acz), 0.0001, 1.0);
        const double ex = bax * t0 - pax, ey = bay * t0 - pay, ez = baz * t0 - paz;
        const double fx = cbx * t1 - pbx, fy = cby * t1 - pby, fz = cbz * t1 - pbz;
        const double gx = acx * t2 - pcx, gy = acy * t2 - pcy, gz = acz * t2 - pcz;
        const double d0 = ex * ex + ey * ey + ez * ez;
        const double d1 = fx * fx + fy * fy + fz * fz;
        const double d2 = gx * gx + gy * gy + gz * gz;
        return fmin(fmin(d0, d1), d2);
    }
    const double np = nx * pax + ny * pay + nz * paz;
    return np * np / (nx * nx + ny * ny + nz * nz);
}

// signed solid angle of triangle abc seen from p (Van Oosterom-Strackee);
// the sum over a closed mesh is 4 pi inside and 0 outside
__device__ double tri_solid_angle(const double *t, double px, double py, double pz) {
#pragma clang fp contract(off)
    const double ax = t[0] - px, ay = t[1] - py, az = t[2] - pz;
    const double bx = t[3] - px, by = t[4] - py, bz = t[5] - pz;
    const double cx = t[6] - px, cy = t[7] - py, cz = t[8] - pz;
    const double la = sqrt(ax * ax + ay * ay + az * az);
    const double lb = sqrt(bx * bx + by * by + bz * bz);
    const double lc = sqrt(cx * cx + cy * cy + cz * cz);
    const double det = ax * (by * cz - bz * cy) - ay * (bx * cz - bz * cx) + az * (bx * cy - by * cx);
    const double den = la * lb * lc + (ax * bx + ay * by + az * bz) * lc + (ax * cx + ay * cy + az * cz) * lb +
                       (bx * cx + by * cy + bz * cz) * la;
    return 2.0 * atan2(det, den);
}

__device__ __forceinline__ double det3(double ax, double ay, double az, double bx, double by, double bz, double cx,
                                       double cy, double cz) {
    return ax * (by * cz - bz * cy) - ay * (bx * cz - bz * cx) + az * (bx * cy - by * cx);
}

// By how much the winding number of a mesh changes from q to p through
// triangle abc: 0, or +-1 where the segment crosses it (tri_solid_angle is
// positive on the side where det(a - p, b - p, c - p) is).  A determinant
// within eps of zero tells nothing; *sure = 0 where the answer needs it.
__device__ __forceinline__ double tri_crossing(const double *t, double px, double py, double pz, double qx, double qy,
                                               double qz, double eps, int *sure) {
    const double ax = t[0] - px, ay = t[1] - py, az = t[2] - pz;
    const double bx = t[3] - px, by = t[4] - py, bz = t[5] - pz;
    const double cx = t[6] - px, cy = t[7] - py, cz = t[8] - pz;
    const double dx = qx - px, dy = qy - py, dz = qz - pz;
    // signed volumes: p and q against the plane, the segment against the edges
    const double sp = det3(ax, ay, az, bx, by, bz, cx, cy, cz);
    const double sq = det3(ax - dx, ay - dy, az - dz, bx - dx, by - dy, bz - dz, cx - dx, cy - dy, cz - dz);
    const double e0 = det3(dx, dy, dz, ax, ay, az, bx, by, bz);
    const double e1 = det3(dx, dy, dz, bx, by, bz, cx, cy, cz);
    const double e2 = det3(dx, dy, dz, cx, cy, cz, ax, ay, az);
    const bool beside = (fmax(fmax(e0, e1), e2) > eps && fmin(fmin(e0, e1), e2) < -eps) ||  // the line misses it
                        fmin(sp, sq) > eps || fmax(sp, sq) < -eps;                          // one side of the plane
    const bool through = (fmin(fmin(e0, e1), e2) > eps || fmax(fmax(e0, e1), e2) < -eps) &&
                         fmin(sp, sq) < -eps && fmax(sp, sq) > eps;
    *sure = beside || through;
    return beside || !through ? 0.0 : (sp > 0.0 ? 1.0 : -1.0);
}

__device__ __forceinline__ float lane_of(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// A triangle's bounding sphere (centroid and radius, FP32, relative to the
// grid's origin).  `slack` covers the FP32 rounding of a position inside the
// grid.  A triangle that tri_dist2 cannot measure (an edge of no length, no
// area, coordinates that are not finite) gets an infinite radius: it is never
// passed over and bounds nothing.
__device__ __forceinline__ float4 tri_sphere(const double *__restrict__ v, double ox, double oy, double oz,
                                             float slack) {
    const double cx = (v[0] + v[3] + v[6]) / 3.0, cy = (v[1] + v[4] + v[7]) / 3.0, cz = (v[2] + v[5] + v[8]) / 3.0;
    double r2 = 0.0, e2 = DBL_MAX;
    for (int k = 0; k < 3; k++) {
        const double *a = v + 3 * k, *b = v + 3 * ((k + 1) % 3);
        r2 = fmax(r2, (a[0] - cx) * (a[0] - cx) + (a[1] - cy) * (a[1] - cy) + (a[2] - cz) * (a[2] - cz));
        e2 = fmin(e2, (a[0] - b[0]) * (a[0] - b[0]) + (a[1] - b[1]) * (a[1] - b[1]) + (a[2] - b[2]) * (a[2] - b[2]));
    }
    const double ux = v[3] - v[0], uy = v[4] - v[1], uz = v[5] - v[2];
    const double wx = v[6] - v[0], wy = v[7] - v[1], wz = v[8] - v[2];
    const double nx = uy * wz - uz * wy, ny = uz * wx - ux * wz, nz = ux * wy - uy * wx;
    const bool sound = e2 > 0.0 && nx * nx + ny * ny + nz * nz > 0.0 && r2 < 1e30 && fabs(cx) + fabs(cy) + fabs(cz) < 1e30;
    return make_float4((float)(cx - ox), (float)(cy - oy), (float)(cz - oz),
                       sound ? (float)sqrt(r2) * 1.000001f + slack : __builtin_inff());
}

__global__ void __launch_bounds__(256) k_tri_spheres(const double *__restrict__ tri, int ntri, double ox, double oy,
                                                     double oz, float slack, float4 *__restrict__ sphere) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < ntri) sphere[t] = tri_sphere(tri + 9 * (size_t)t, ox, oy, oz, slack);
}

// Every triangle's distance and solid angle at every node, a node per lane: what
// the kernel below saves itself, for meshes and grids so small that its bounds
// only lengthen each lane's chain.
__global__ void __launch_bounds__(64) k_sdf_all_pairs(const double *__restrict__ tri, int ntri, int nx, int ny, int nz,
                                                      double ox, double oy, double oz, double dx,
                                                      float *__restrict__ out) {
#pragma clang fp contract(off)
    const unsigned node = blockIdx.x * 64u + threadIdx.x, row = node / (unsigned)nx;
    if (node >= (unsigned)nx * ny * nz) return;  // below 2^31
    const double px = ox + dx * (double)(node % (unsigned)nx), py = oy + dx * (double)(row % (unsigned)ny),
                 pz = oz + dx * (double)(row / (unsigned)ny);
    double best = DBL_MAX, wind = 0.0;
    for (int t = 0; t < ntri; t++) {
        best = fmin(best, tri_dist2(tri + 9 * t, px, py, pz));
        wind += tri_solid_angle(tri + 9 * t, px, py, pz);
    }
    const double psd = fmax(sqrt(best), 0.00001);
    out[node] = (float)(fabs(wind) > 2.0 * M_PI ? -psd : psd);  // |winding number| > 1/2
}

// SetNodeSDFKernel (src/core/shape.cpp:411-424) for a mesh: distance to the
// closest triangle, at least 1e-5, negative inside.  Inside is decided by
// the winding number of the mesh (the reference counts ray hits towards the
// mesh's bounds centre, src/core/shape.cpp:356-373).
//
// A workgroup holds a brick of 4 x 4 x 4 nodes, one per lane in each of its
// waves, and splits the triangles between them.  FP64 distances and solid angles
// of every (node, triangle) pair bounded the kernel (4.03 ms at 229k nodes
// and 1,280 triangles, about 2,100 cycles per pair of a wave), so most pairs
// get neither (0.31 ms; 34 to 2.1 ms at 572k nodes and 5,120 triangles of a
// ball, whose centre no bound helps and one wave alone took 4.6 ms over):
//  - Centroids bound the brick's distances from above, bounding spheres bound
//    them from below: FP32, a triangle per lane.  Only triangles that some
//    node of the brick may be closest to go on to a test per node and then
//    to tri_dist2.  The minimum is over the same values as before.
//  - The winding number of a closed mesh changes by one where a path meets
//    the surface.  The brick's farthest node is evaluated by the workgroup (a
//    256th of the triangles per lane), the others by the triangles that
//    the path from it crosses, of those that reach into the brick.
//  - A node whose path is too close to an edge or a plane to tell, and every
//    node of a mesh that is not closed (or has a triangle without area),
//    takes the whole sum in triangle order: at the surface and in an opening
//    the winding number is 1/2 up to its rounding.
template <int kWaves>
__global__ void __launch_bounds__(64 * kWaves) k_sdf_from_mesh(const double *__restrict__ tri,
                                                               const float4 *__restrict__ sphere, int ntri, int nx,
                                                               int ny, int nz, double ox, double oy, double oz,
                                                               double dx, float slack, int closed,
                                                               float *__restrict__ out) {
#pragma clang fp contract(off)
    constexpr int kSdfBlock = 64 * kWaves;
    __shared__ unsigned near_up[64];   // per node: bits of the smallest bound so far
    __shared__ double part[kWaves][64];
    __shared__ float red[3][kWaves];
    __shared__ int red_at[kWaves];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int bx = (nx + 3) / 4, by = (ny + 3) / 4;
    const int brick = (int)blockIdx.x;
    const int i = brick % bx * 4 + (lane & 3), j = brick / bx % by * 4 + (lane >> 2 & 3),
              k = brick / (bx * by) * 4 + (lane >> 4);
    const bool live = i < nx && j < ny && k < nz;
    const double px = ox + dx * (double)i, py = oy + dx * (double)j, pz = oz + dx * (double)k;
    const float fx = (float)(px - ox), fy = (float)(py - oy), fz = (float)(pz - oz);
    // the brick's centre and the radius that holds its nodes
    const float half = 1.5f * (float)dx;
    const float cx = __shfl(fx, 0, 64) + half, cy = __shfl(fy, 0, 64) + half, cz = __shfl(fz, 0, 64) + half;
    const float brad = 1.7321f * half + slack;
    // a small mesh's spheres are made here, a triangle per lane, without a launch before this one
    float4 own = make_float4(0.f, 0.f, 0.f, 0.f);
    if constexpr (kWaves == 1)
        if (lane < ntri) own = tri_sphere(tri + 9 * (size_t)lane, ox, oy, oz, slack);
    auto sphere_of = [&](int t) {
        if constexpr (kWaves == 1)
            return own;
        else
            return t < ntri ? sphere[t] : make_float4(0.f, 0.f, 0.f, 0.f);
    };
    float c2 = __builtin_inff(), rmax = 0.f, edge = 0.f;
    int nearest = 0;
    for (int t = wave * 64 + lane; t < ntri; t += kSdfBlock) {
        const float4 s = sphere_of(t);
        const float ax = cx - s.x, ay = cy - s.y, az = cz - s.z, d2 = ax * ax + ay * ay + az * az;
        const bool sound = s.w < 3.4e38f;
        if (sound && d2 < c2) {
            c2 = d2;
            nearest = t;
        }
        rmax = fmaxf(rmax, s.w);
        edge = fmaxf(edge, sound ? s.w : 0.f);
    }
    for (int off = 32; off > 0; off >>= 1) {
        const float o2 = __shfl_xor(c2, off, 64);
        const int ot = __shfl_xor(nearest, off, 64);
        if (o2 < c2) {
            c2 = o2;
            nearest = ot;
        }
        rmax = fmaxf(rmax, __shfl_xor(rmax, off, 64));
        edge = fmaxf(edge, __shfl_xor(edge, off, 64));
    }
    if (lane == 0) {
        red[0][wave] = c2;
        red[1][wave] = rmax;
        red[2][wave] = edge;
        red_at[wave] = nearest;
    }
    if (wave == 0) near_up[lane] = 0x7f800000u;
    __syncthreads();
    for (int w = 0; w < kWaves; w++) {
        if (red[0][w] < c2) {
            c2 = red[0][w];
            nearest = red_at[w];
        }
        rmax = fmaxf(rmax, red[1][w]);
        edge = fmaxf(edge, red[2][w]);
    }
    // lanes of a wave may hold different triangles at equal distances
    nearest = __builtin_amdgcn_readfirstlane(nearest);
    // every node's distance is below `up`: the nearest centroid's, plus what
    // the lower end of the edge parameters (1e-4 of an edge) can add
    float up = sqrtf(c2) * 1.000001f + brad + slack + 1e-3f * edge;
    const float brick_up = up + brad;
    double best = DBL_MAX;
    auto measure = [&](int t) {
        best = fmin(best, tri_dist2(tri + 9 * (size_t)t, px, py, pz));
        up = fminf(up, (float)sqrt(best) * 1.000001f + slack);
    };
    measure(nearest);
    for (int t0 = wave * 64; t0 < ntri; t0 += kSdfBlock) {
        const float4 s = sphere_of(t0 + lane);
        const float ax = cx - s.x, ay = cy - s.y, az = cz - s.z, reach = brick_up + s.w;
        // both tests are written so that a NaN keeps the triangle
        unsigned long long keep =
            __ballot(t0 + lane < ntri && !(ax * ax + ay * ay + az * az > reach * reach * 1.00001f));
        for (; keep; keep &= keep - 1) {
            const int l = __builtin_ctzll(keep);
            const float ux = fx - lane_of(s.x, l), uy = fy - lane_of(s.y, l), uz = fz - lane_of(s.z, l);
            const float r = up + lane_of(s.w, l);
            if (__ballot(live && !(ux * ux + uy * uy + uz * uz > r * r * 1.00001f))) {
                measure(t0 + l);
                // what one wave finds narrows the search of the others
                up = fminf(up, __uint_as_float(atomicMin(&near_up[lane], __float_as_uint(up))));
            }
        }
    }
    part[wave][lane] = best;
    __syncthreads();
    for (int w = 0; w < kWaves; w++) best = fmin(best, part[w][lane]);
    __syncthreads();
    const double dist = sqrt(best);
    bool interior = false;
    unsigned long long todo = __ballot(live);
    if (closed && rmax < 3.4e38f) {
        // the brick's farthest node, by the whole workgroup
        const float far = live ? (float)dist : -1.f;
        float top = far;
        for (int off = 32; off > 0; off >>= 1) top = fmaxf(top, __shfl_xor(top, off, 64));
        const unsigned long long at = __ballot(live && far == top);
        const int rep = at ? __builtin_ctzll(at) : 0;
        const double qx = __shfl(px, rep, 64), qy = __shfl(py, rep, 64), qz = __shfl(pz, rep, 64);
        double turns = 0.0;
        for (int t = wave * 64 + lane; t < ntri; t += kSdfBlock) turns += tri_solid_angle(tri + 9 * (size_t)t, qx, qy, qz);
        for (int off = 32; off > 0; off >>= 1) turns += __shfl_xor(turns, off, 64);
        // the others by the triangles between them and it; each lane its own path
        double number = 0.0;
        bool unsure = false;
        for (int t0 = wave * 64; t0 < ntri; t0 += kSdfBlock) {
            const float4 s = sphere_of(t0 + lane);
            const float ax = cx - s.x, ay = cy - s.y, az = cz - s.z, reach = brad + s.w;
            unsigned long long near = __ballot(t0 + lane < ntri && !(ax * ax + ay * ay + az * az > reach * reach * 1.00001f));
            for (; near; near &= near - 1) {
                const int l = __builtin_ctzll(near);
                const double len = 2.0 * ((double)lane_of(s.w, l) + (double)brad);
                int sure;
                number += tri_crossing(tri + 9 * (size_t)(t0 + l), px, py, pz, qx, qy, qz,
                                       1e-10 * len * len * (len + 1e6 * (double)slack), &sure);
                unsure = unsure || (!sure && lane != rep);
            }
        }
        // crossings are whole numbers: 1e6 marks a path that cannot tell
        part[wave][lane] = (unsure ? 1e6 : 0.0) + number + turns / (4.0 * M_PI);
        __syncthreads();
        double sum = 0.0;
        for (int w = 0; w < kWaves; w++) sum += part[w][lane];
        number = rint(sum);
        interior = fabs(number) > 0.5;
        todo &= __ballot(!(fabs(sum - number) < 1e-3) || fabs(number) > 5e5);
    }
    if (wave > 0) return;
    // Every node for itself, or one after the other by the whole wave, 64
    // triangles at a time, whose additions in order cost as much as two more
    // solid angles: the latter for few nodes and many triangles.
    if (__popcll(todo) > (kWaves == 1 ? 3 * ntri / 8 : 24)) {
        double wind = 0.0;
        for (int t = 0; t < ntri; t++) wind += tri_solid_angle(tri + 9 * (size_t)t, px, py, pz);
        if (todo >> lane & 1ull) interior = fabs(wind) > 2.0 * M_PI;  // |winding number| > 1/2
        todo = 0ull;
    }
    for (; todo; todo &= todo - 1) {
        const int rep = __builtin_ctzll(todo);
        const double qx = __shfl(px, rep, 64), qy = __shfl(py, rep, 64), qz = __shfl(pz, rep, 64);
        double wind = 0.0;
        for (int t0 = 0; t0 < ntri; t0 += 64) {
            const double a = t0 + lane < ntri ? tri_solid_angle(tri + 9 * (size_t)(t0 + lane), qx, qy, qz) : 0.0;
            auto add = [&](int l) {
                wind += __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(a), l),
                                         __builtin_amdgcn_readlane(__double2loint(a), l));
            };
            if (ntri - t0 >= 64) {
                for (int l = 0; l < 64; l++) add(l);
            } else {
                for (int l = 0; l < ntri - t0; l++) add(l);
            }
        }
        if (lane == rep) interior = fabs(wind) > 2.0 * M_PI;
    }
    if (live) {
        const double psd = fmax(dist, 0.00001);
        out[(size_t)i + (size_t)nx * ((size_t)j + (size_t)ny * (size_t)k)] = (float)(interior ? -psd : psd);
    }
}

__global__ void __launch_bounds__(256) k_sdf_sample(DevCollider c, const float4 *__restrict__ pts, int n,
                                                    float4 *__restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float3 p = make_float3(pts[i].x, pts[i].y, pts[i].z);
    const float3 g = sdf_gradient(c, p);
    out[i] = make_float4(sdf_sample(c, p), g.x, g.y, g.z);
}

__global__ void __launch_bounds__(256) k_resolve(const DevCollider *__restrict__ cs, int nc, float radius, float e,
                                                 float4 *__restrict__ pos, float4 *__restrict__ vel,
                                                 int *__restrict__ hit, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float3 p = make_float3(pos[i].x, pos[i].y, pos[i].z);
    float3 v = make_float3(vel[i].x, vel[i].y, vel[i].z);
    const bool h = resolve_colliders(cs, nc, radius, e, p, v);
    pos[i] = make_float4(p.x, p.y, p.z, 0.f);
    vel[i] = make_float4(v.x, v.y, v.z, 0.f);
    hit[i] = h ? 1 : 0;
}

// The same rule over the caller's FP64 arrays as staged in device memory:
// each coordinate rounds to FP32 exactly as the host conversion of
// k_resolve's caller does, and the result widens back to FP64.
__global__ void __launch_bounds__(256) k_resolve_f64(const DevCollider *__restrict__ cs, int nc, float radius,
                                                     float e, double *__restrict__ pos, double *__restrict__ vel,
                                                     int *__restrict__ hit, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double *pp = pos + 3 * (size_t)i;
    double *vv = vel + 3 * (size_t)i;
    float3 p = make_float3((float)pp[0], (float)pp[1], (float)pp[2]);
    float3 v = make_float3((float)vv[0], (float)vv[1], (float)vv[2]);
    const bool h = resolve_colliders(cs, nc, radius, e, p, v);
    pp[0] = p.x;
    pp[1] = p.y;
    pp[2] = p.z;
    vv[0] = v.x;
    vv[1] = v.y;
    vv[2] = v.z;
    hit[i] = h ? 1 : 0;
}

// ---------------------------------------------------------------------------
// Staging of bbx_colliders_resolve_noalloc: one file-scope device array per
// GPU, laid out as [collider table | positions | velocities | flags].  Its
// address is looked up once per device with hipGetSymbolAddress; host code
// never passes the array's name itself to a kernel or a copy.
// ---------------------------------------------------------------------------
constexpr size_t kNoAllocCollBytes = ((sizeof(DevCollider) * kMaxColliders + 255) / 256) * 256;
constexpr size_t kNoAllocVecBytes = (size_t)BBX_NOALLOC_MAX_POINTS * 3 * sizeof(double);
constexpr size_t kNoAllocBytes = kNoAllocCollBytes + 2 * kNoAllocVecBytes + (size_t)BBX_NOALLOC_MAX_POINTS * sizeof(int);
static_assert(kNoAllocVecBytes % 256 == 0, "scratch segments stay 256-byte aligned");

static __device__ __align__(256) unsigned char scratch[kNoAllocBytes];

constexpr int kNoAllocDevices = 64;
std::mutex g_scratch_mu;
unsigned char *g_scratch_ptr[kNoAllocDevices] = {};

// Device address of the current device's scratch array (looked up on the
// first call made with that device current).
int scratch_for_current_device(unsigned char **out) {
    int dev = -1;
    BBX_HIP_CHECK(hipGetDevice(&dev));
    if (dev < 0 || dev >= kNoAllocDevices) return fail(BBX_E_RANGE, "device ordinal beyond the scratch table");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return fail(BBX_E_HIP, std::string("scratch address: ") + hipGetErrorString(e));
        g_scratch_ptr[dev] = (unsigned char *)p;
    }
    *out = g_scratch_ptr[dev];
    return BBX_OK;
}

void sdf_fields(const bbx_sdf *s, DevCollider &d) {
    d.field = s->field;
    d.nx = s->nodes[0];
    d.ny = s->nodes[1];
    d.nz = s->nodes[2];
    d.ox = (float)s->origin[0];
    d.oy = (float)s->origin[1];
    d.oz = (float)s->origin[2];
    d.sx = (float)s->spacing[0];
    d.sy = (float)s->spacing[1];
    d.sz = (float)s->spacing[2];
}

int to_device(const bbx_collider &h, DevCollider &d) {
    std::memset(&d, 0, sizeof(d));
    if (h.kind < BBX_SHAPE_BOX || h.kind > BBX_SHAPE_SDF) return fail(BBX_E_INVALID, "unknown collider kind");
    d.kind = h.kind;
    d.reverse = h.reverse_orientation ? 1 : 0;
    d.active = h.active ? 1 : 0;
    d.friction = (float)h.friction;
    for (int k = 0; k < 12; k++) {
        d.m[k] = (float)h.to_world[k];
        d.mi[k] = (float)h.to_object[k];
    }
    d.hx = (float)(h.size[0] / 2.0);
    d.hy = (float)(h.size[1] / 2.0);
    d.hz = (float)(h.size[2] / 2.0);
    d.radius = (float)h.radius;
    for (int k = 0; k < 3; k++) {
        d.lin[k] = (float)h.linear_velocity[k];
        d.ang[k] = (float)h.angular_velocity[k];
        d.bmin[k] = (float)h.bounds_min[k];
        d.bmax[k] = (float)h.bounds_max[k];
    }
    if (h.kind == BBX_SHAPE_MESH || h.kind == BBX_SHAPE_SDF) {
        if (!h.sdf || !h.sdf->field) return fail(BBX_E_INVALID, "mesh and SDF colliders need an SDF");
        sdf_fields(h.sdf, d);
    }
    return BBX_OK;
}

// Whether the triangles' directed edges cancel (each edge is walked as often
// one way as the other), so that the winding number is the same along any
// path off the surface.  Edges are compared by vertex index; a mesh whose
// triangles do not share vertices counts as open (as does any without the
// memory to tell).
bool closed_mesh(const int *triangles, int ntriangles) try {
    size_t cap = 64;
    while (cap < 6 * (size_t)ntriangles) cap *= 2;
    std::vector<unsigned long long> key(cap, 0);
    std::vector<int> net(cap, 0);
    for (int t = 0; t < ntriangles; t++)
        for (int c = 0; c < 3; c++) {
            const unsigned a = (unsigned)triangles[3 * (size_t)t + c], b = (unsigned)triangles[3 * (size_t)t + (c + 1) % 3];
            if (a == b) continue;
            const unsigned long long k = ((unsigned long long)(std::min(a, b) + 1) << 32) | (std::max(a, b) + 1);
            size_t h = (size_t)((k * 0x9E3779B97F4A7C15ull) >> 20) & (cap - 1);
            while (key[h] && key[h] != k) h = (h + 1) & (cap - 1);
            key[h] = k;
            net[h] += a < b ? 1 : -1;
        }
    for (int v : net)
        if (v) return false;
    return true;
} catch (const std::bad_alloc &) {
    return false;
}

int upload_colliders(const bbx_collider *list, int count, std::vector<DevCollider> &out) {
    if (count < 0 || count > kMaxColliders) return fail(BBX_E_RANGE, "collider count out of range (0..64)");
    if (count && !list) return fail(BBX_E_INVALID, "null collider list");
    out.resize((size_t)count);
    for (int i = 0; i < count; i++) BBX_CHECK(to_device(list[i], out[(size_t)i]));
    return BBX_OK;
}

}  // namespace

extern "C" {

int bbx_sdf_create(const int nodes[3], const double origin[3], const double spacing[3], const double *values,
                   bbx_sdf **out) {
    if (!out || !nodes || !origin || !spacing || !values) return fail(BBX_E_INVALID, "null argument");
    *out = nullptr;
    long long total = 1;
    for (int k = 0; k < 3; k++) {
        if (nodes[k] < 1 || nodes[k] > (1 << 15)) return fail(BBX_E_RANGE, "SDF node count out of range");
        if (!(spacing[k] > 0)) return fail(BBX_E_INVALID, "SDF spacing must be positive");
        total *= nodes[k];
    }
    if (total > (1LL << 31) - 1) return fail(BBX_E_RANGE, "SDF too large");
    bbx_sdf *s = new bbx_sdf();
    for (int k = 0; k < 3; k++) {
        s->nodes[k] = nodes[k];
        s->origin[k] = origin[k];
        s->spacing[k] = spacing[k];
    }
    std::vector<float> h((size_t)total);
    for (long long i = 0; i < total; i++) h[(size_t)i] = (float)values[i];
    hipError_t e = hipMalloc((void **)&s->field, sizeof(float) * (size_t)total);
    if (e == hipSuccess) e = hipMemcpy(s->field, h.data(), sizeof(float) * (size_t)total, hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        if (s->field) (void)hipFree(s->field);
        delete s;
        return fail(BBX_E_HIP, std::string("SDF upload: ") + hipGetErrorString(e));
    }
    *out = s;
    return BBX_OK;
}

int bbx_sdf_from_mesh(const double *vertices, int nvertices, const int *triangles, int ntriangles, double dx,
                      double margin, bbx_sdf **out) {
    if (!out) return fail(BBX_E_INVALID, "null output");
    *out = nullptr;
    if (!vertices || !triangles || nvertices < 3 || ntriangles < 1) return fail(BBX_E_INVALID, "empty mesh");
    if (!(dx > 0) || !(margin >= 0)) return fail(BBX_E_INVALID, "bad SDF spacing or margin");
    // bounds of the triangles' vertices (the mesh BVH root bound)
    double lo[3] = {DBL_MAX, DBL_MAX, DBL_MAX}, hi[3] = {-DBL_MAX, -DBL_MAX, -DBL_MAX};
    std::vector<double> tri((size_t)ntriangles * 9);
    for (int t = 0; t < ntriangles; t++)
        for (int c = 0; c < 3; c++) {
            const int v = triangles[3 * (size_t)t + c];
            if (v < 0 || v >= nvertices) return fail(BBX_E_INVALID, "triangle index out of range");
            for (int k = 0; k < 3; k++) {
                const double x = vertices[3 * (size_t)v + k];
                tri[9 * (size_t)t + 3 * c + k] = x;
                lo[k] = std::min(lo[k], x);
                hi[k] = std::max(hi[k], x);
            }
        }
    // GenerateShapeSDF (src/core/shape.cpp:478-505)
    double pmin[3], pmax[3];
    for (int k = 0; k < 3; k++) {
        const double scale = hi[k] - lo[k];
        pmin[k] = lo[k] - margin * scale;
        pmax[k] = hi[k] + margin * scale;
    }
    const double width = pmax[0] - pmin[0], height = pmax[1] - pmin[1], depth = pmax[2] - pmin[2];
    if (!(width > 0)) return fail(BBX_E_INVALID, "mesh has no extent along x");
    const double resd = std::ceil(width / dx);
    if (resd > 4096) return fail(BBX_E_RANGE, "SDF resolution above 4096 per axis");
    const int res = (int)resd;
    const double sp = width / (double)res;
    const int resy = (int)std::ceil(res * height / width);
    const int resz = (int)std::ceil(res * depth / width);
    if (resy > 4096 || resz > 4096) return fail(BBX_E_RANGE, "SDF resolution above 4096 per axis");
    if ((long long)(res + 1) * (resy + 1) * (resz + 1) > (1LL << 31) - 1) return fail(BBX_E_RANGE, "SDF too large");
    bbx_sdf *s = new bbx_sdf();
    s->nodes[0] = res + 1;
    s->nodes[1] = resy + 1;
    s->nodes[2] = resz + 1;
    for (int k = 0; k < 3; k++) {
        s->origin[k] = pmin[k];
        s->spacing[k] = sp;
    }
    const long long total = (long long)s->nodes[0] * s->nodes[1] * s->nodes[2];
    // triangles, then their bounding spheres
    double *dtri = nullptr;
    const size_t tri_bytes = (sizeof(double) * tri.size() + 255) / 256 * 256;
    const bool closed = closed_mesh(triangles, ntriangles);
    const float slack = (float)(1e-6 * (width + height + depth));
    hipError_t e = hipMalloc((void **)&s->field, sizeof(float) * (size_t)total);
    if (e == hipSuccess) e = hipMalloc((void **)&dtri, tri_bytes + sizeof(float4) * (size_t)ntriangles);
    if (e == hipSuccess) e = hipMemcpy(dtri, tri.data(), sizeof(double) * tri.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        float4 *sphere = (float4 *)((char *)dtri + tri_bytes);
        const bool direct = ntriangles <= kSdfFew || (ntriangles <= 2 * kSdfFew && total <= kSdfFewNodes);
        const int waves = ntriangles <= kSdfOneWave ? 1 : kSdfWaves;
        if (waves > 1)
            k_tri_spheres<<<(unsigned)((ntriangles + 255) / 256), 256>>>(dtri, ntriangles, pmin[0], pmin[1], pmin[2],
                                                                         slack, sphere);
        const long long bricks = (long long)((s->nodes[0] + 3) / 4) * ((s->nodes[1] + 3) / 4) * ((s->nodes[2] + 3) / 4);
        if (direct)
            k_sdf_all_pairs<<<(unsigned)((total + 63) / 64), 64>>>(dtri, ntriangles, s->nodes[0], s->nodes[1],
                                                                   s->nodes[2], pmin[0], pmin[1], pmin[2], sp, s->field);
        else
            (waves == 1 ? k_sdf_from_mesh<1> : k_sdf_from_mesh<kSdfWaves>)<<<(unsigned)bricks, 64 * waves>>>(
                dtri, sphere, ntriangles, s->nodes[0], s->nodes[1], s->nodes[2], pmin[0], pmin[1], pmin[2], sp, slack,
                closed ? 1 : 0, s->field);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipDeviceSynchronize();
    if (dtri) (void)hipFree(dtri);
    if (e != hipSuccess) {
        if (s->field) (void)hipFree(s->field);
        delete s;
        return fail(BBX_E_HIP, std::string("SDF from mesh: ") + hipGetErrorString(e));
    }
    *out = s;
    return BBX_OK;
}

int bbx_sdf_describe(const bbx_sdf *sdf, int nodes[3], double origin[3], double spacing[3]) {
    if (!sdf) return fail(BBX_E_INVALID, "null SDF");
    for (int k = 0; k < 3; k++) {
        if (nodes) nodes[k] = sdf->nodes[k];
        if (origin) origin[k] = sdf->origin[k];
        if (spacing) spacing[k] = sdf->spacing[k];
    }
    return BBX_OK;
}

int bbx_sdf_download(const bbx_sdf *sdf, double *values) {
    if (!sdf || !values) return fail(BBX_E_INVALID, "null argument");
    const size_t total = (size_t)sdf->nodes[0] * sdf->nodes[1] * sdf->nodes[2];
    std::vector<float> h(total);
    BBX_HIP_CHECK(hipMemcpy(h.data(), sdf->field, sizeof(float) * total, hipMemcpyDeviceToHost));
    for (size_t i = 0; i < total; i++) values[i] = h[i];
    return BBX_OK;
}

int bbx_sdf_sample(const bbx_sdf *sdf, const double *points, int n, double *values, double *gradients) {
    if (!sdf || (n > 0 && (!points || !values))) return fail(BBX_E_INVALID, "null argument");
    if (n <= 0) return BBX_OK;
    DevCollider c;
    std::memset(&c, 0, sizeof(c));
    c.kind = BBX_SHAPE_SDF;
    sdf_fields(sdf, c);
    std::vector<float4> hp((size_t)n), ho((size_t)n);
    for (int i = 0; i < n; i++)
        hp[(size_t)i] = make_float4((float)points[3 * (size_t)i], (float)points[3 * (size_t)i + 1],
                                    (float)points[3 * (size_t)i + 2], 0.f);
    float4 *dp = nullptr, *dout = nullptr;
    hipError_t e = hipMalloc((void **)&dp, sizeof(float4) * (size_t)n);
    if (e == hipSuccess) e = hipMalloc((void **)&dout, sizeof(float4) * (size_t)n);
    if (e == hipSuccess) e = hipMemcpy(dp, hp.data(), sizeof(float4) * (size_t)n, hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        k_sdf_sample<<<(unsigned)((n + 255) / 256), 256>>>(c, dp, n, dout);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpy(ho.data(), dout, sizeof(float4) * (size_t)n, hipMemcpyDeviceToHost);
    if (dp) (void)hipFree(dp);
    if (dout) (void)hipFree(dout);
    if (e != hipSuccess) return fail(BBX_E_HIP, std::string("SDF sample: ") + hipGetErrorString(e));
    for (int i = 0; i < n; i++) {
        values[i] = ho[(size_t)i].x;
        if (gradients) {
            gradients[3 * (size_t)i] = ho[(size_t)i].y;
            gradients[3 * (size_t)i + 1] = ho[(size_t)i].z;
            gradients[3 * (size_t)i + 2] = ho[(size_t)i].w;
        }
    }
    return BBX_OK;
}

void bbx_sdf_destroy(bbx_sdf *sdf) {
    if (!sdf) return;
    if (sdf->field) (void)hipFree(sdf->field);
    delete sdf;
}

int bbx_solver_set_colliders(bbx_solver *s, const bbx_collider *colliders, int count) {
    if (!s) return fail(BBX_E_INVALID, "null solver");
    std::vector<DevCollider> h;
    BBX_CHECK(upload_colliders(colliders, count, h));
    BBX_HIP_CHECK(hipStreamSynchronize(s->stream));  // kernels may still read the old list
    if (count == 0) {
        if (s->coll) (void)hipFree(s->coll);
        s->coll = nullptr;
        s->ncoll = 0;
        fill_sim_const(s);
        return BBX_OK;
    }
    if (!s->coll) {
        hipError_t e = hipMalloc((void **)&s->coll, sizeof(DevCollider) * kMaxColliders);
        if (e != hipSuccess) {
            s->coll = nullptr;
            return fail(BBX_E_NOMEM, std::string("collider list: ") + hipGetErrorString(e));
        }
    }
    BBX_HIP_CHECK(hipMemcpy(s->coll, h.data(), sizeof(DevCollider) * (size_t)count, hipMemcpyHostToDevice));
    s->ncoll = count;
    fill_sim_const(s);
    return BBX_OK;
}

int bbx_colliders_resolve(const bbx_collider *colliders, int count, double radius, double restitution,
                          double *pos, double *vel, int n, int *collided) {
    if (n < 0 || (n > 0 && (!pos || !vel))) return fail(BBX_E_INVALID, "bad point arrays");
    if (count < 1) return fail(BBX_E_INVALID, "no colliders");
    std::vector<DevCollider> h;
    BBX_CHECK(upload_colliders(colliders, count, h));
    if (n == 0) return BBX_OK;
    std::vector<float4> hp((size_t)n), hv((size_t)n);
    std::vector<int> hh((size_t)n);
    for (int i = 0; i < n; i++) {
        hp[(size_t)i] = make_float4((float)pos[3 * (size_t)i], (float)pos[3 * (size_t)i + 1],
                                    (float)pos[3 * (size_t)i + 2], 0.f);
        hv[(size_t)i] = make_float4((float)vel[3 * (size_t)i], (float)vel[3 * (size_t)i + 1],
                                    (float)vel[3 * (size_t)i + 2], 0.f);
    }
    DevCollider *dc = nullptr;
    float4 *dp = nullptr, *dv = nullptr;
    int *dh = nullptr;
    hipError_t e = hipMalloc((void **)&dc, sizeof(DevCollider) * (size_t)count);
    if (e == hipSuccess) e = hipMalloc((void **)&dp, sizeof(float4) * (size_t)n);
    if (e == hipSuccess) e = hipMalloc((void **)&dv, sizeof(float4) * (size_t)n);
    if (e == hipSuccess) e = hipMalloc((void **)&dh, sizeof(int) * (size_t)n);
    if (e == hipSuccess) e = hipMemcpy(dc, h.data(), sizeof(DevCollider) * (size_t)count, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(dp, hp.data(), sizeof(float4) * (size_t)n, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(dv, hv.data(), sizeof(float4) * (size_t)n, hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        k_resolve<<<(unsigned)((n + 255) / 256), 256>>>(dc, count, (float)radius, (float)restitution, dp, dv, dh,
                                                         n);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpy(hp.data(), dp, sizeof(float4) * (size_t)n, hipMemcpyDeviceToHost);
    if (e == hipSuccess) e = hipMemcpy(hv.data(), dv, sizeof(float4) * (size_t)n, hipMemcpyDeviceToHost);
    if (e == hipSuccess) e = hipMemcpy(hh.data(), dh, sizeof(int) * (size_t)n, hipMemcpyDeviceToHost);
    if (dc) (void)hipFree(dc);
    if (dp) (void)hipFree(dp);
    if (dv) (void)hipFree(dv);
    if (dh) (void)hipFree(dh);
    if (e != hipSuccess) return fail(BBX_E_HIP, std::string("collider resolve: ") + hipGetErrorString(e));
    for (int i = 0; i < n; i++) {
        pos[3 * (size_t)i] = hp[(size_t)i].x;
        pos[3 * (size_t)i + 1] = hp[(size_t)i].y;
        pos[3 * (size_t)i + 2] = hp[(size_t)i].z;
        vel[3 * (size_t)i] = hv[(size_t)i].x;
        vel[3 * (size_t)i + 1] = hv[(size_t)i].y;
        vel[3 * (size_t)i + 2] = hv[(size_t)i].z;
        if (collided) collided[i] = hh[(size_t)i];
    }
    return BBX_OK;
}

int bbx_colliders_resolve_noalloc(const bbx_collider *colliders, int count, double radius, double restitution,
                                  double *pos, double *vel, int n, int *collided) {
    if (n < 0 || (n > 0 && (!pos || !vel))) return fail(BBX_E_INVALID, "bad point arrays");
    if (n > BBX_NOALLOC_MAX_POINTS)
        return fail(BBX_E_RANGE, "bbx_colliders_resolve_noalloc takes at most " +
                                     std::to_string(BBX_NOALLOC_MAX_POINTS) + " points per call (got " +
                                     std::to_string(n) + ")");
    if (count < 1) return fail(BBX_E_INVALID, "no colliders");
    if (count > kMaxColliders) return fail(BBX_E_RANGE, "collider count out of range (0..64)");
    if (!colliders) return fail(BBX_E_INVALID, "null collider list");
    DevCollider table[kMaxColliders];
    for (int i = 0; i < count; i++) BBX_CHECK(to_device(colliders[i], table[i]));
    if (n == 0) return BBX_OK;
    unsigned char *base = nullptr;
    BBX_CHECK(scratch_for_current_device(&base));
    DevCollider *dc = (DevCollider *)base;
    double *dp = (double *)(base + kNoAllocCollBytes);
    double *dv = (double *)(base + kNoAllocCollBytes + kNoAllocVecBytes);
    int *dh = (int *)(base + kNoAllocCollBytes + 2 * kNoAllocVecBytes);
    const size_t vb = sizeof(double) * 3 * (size_t)n;
    hipError_t e = hipMemcpy(dc, table, sizeof(DevCollider) * (size_t)count, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(dp, pos, vb, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(dv, vel, vb, hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        k_resolve_f64<<<(unsigned)((n + 255) / 256), 256>>>(dc, count, (float)radius, (float)restitution, dp, dv,
                                                             dh, n);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpy(pos, dp, vb, hipMemcpyDeviceToHost);
    if (e == hipSuccess) e = hipMemcpy(vel, dv, vb, hipMemcpyDeviceToHost);
    if (e == hipSuccess && collided) e = hipMemcpy(collided, dh, sizeof(int) * (size_t)n, hipMemcpyDeviceToHost);
    if (e != hipSuccess) return fail(BBX_E_HIP, std::string("collider resolve (no-alloc): ") + hipGetErrorString(e));
    return BBX_OK;
}

}  // extern "C"
