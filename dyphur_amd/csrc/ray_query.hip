// ray_query.hip — closest-hit ray queries over the broadphase's LBVH for
// gfx950 (core/src/ray_query.cpp:12-195, core/include/core/ray_query.hpp).
//
// The reference walks the tree depth first, left subtree first, with the best
// hit so far (which fixes which of two equally distant hits is reported); node
// boxes are the 16-byte binary16 NodeBox records, leaves are tested exactly
// (oriented box slab test in the body frame, analytic sphere).  Arithmetic in
// the reference's operation order; compiled without contraction, so results
// are bit-equal to a CPU evaluation of the same steps.
#include "dy_internal.hpp"

namespace dy {

__device__ __forceinline__ void rq_slab(const float o[3], const float inv[3], const float mn[3], const float mx[3],
                                        float &tmin, float &tmax) {
    const float t1x = (mn[0] - o[0]) * inv[0], t2x = (mx[0] - o[0]) * inv[0];
    const float t1y = (mn[1] - o[1]) * inv[1], t2y = (mx[1] - o[1]) * inv[1];
    const float t1z = (mn[2] - o[2]) * inv[2], t2z = (mx[2] - o[2]) * inv[2];
    tmin = t1x < t2x ? t1x : t2x;
    tmax = t1x < t2x ? t2x : t1x;
    const float ylo = t1y < t2y ? t1y : t2y, yhi = t1y < t2y ? t2y : t1y;
    tmin = tmin > ylo ? tmin : ylo;
    tmax = tmax < yhi ? tmax : yhi;
    const float zlo = t1z < t2z ? t1z : t2z, zhi = t1z < t2z ? t2z : t1z;
    tmin = tmin > zlo ? tmin : zlo;
    tmax = tmax < zhi ? tmax : zhi;
}

// v rotated by the conjugate of q: t = 2 u x v, v + w t + u x t, u = -xyz
// (core/include/core/math/quat.hpp:31,39-42).
__device__ __forceinline__ void rq_rotate_inv(float w, float x, float y, float z, const float v[3], float o[3]) {
    const float ux = -x, uy = -y, uz = -z;
    const float tx = (uy * v[2] - uz * v[1]) * 2.f;
    const float ty = (uz * v[0] - ux * v[2]) * 2.f;
    const float tz = (ux * v[1] - uy * v[0]) * 2.f;
    o[0] = (v[0] + tx * w) + (uy * tz - uz * ty);
    o[1] = (v[1] + ty * w) + (uz * tx - ux * tz);
    o[2] = (v[2] + tz * w) + (ux * ty - uy * tx);
}

// A leaf's body as the exact test needs it.
struct RqBody {
    float p[3], q[4], h[3];  // position, orientation (w x y z), half extents (h[0]: a sphere's radius)
    uint32_t type, body;
};

__device__ __forceinline__ RqBody rq_body(const dy_bvh_view &bvh, const dy_body_view &bv, const dy_shape_view &sv,
                                          uint32_t leaf) {
    const uint32_t bi = bvh.n == 1u ? 0u : bvh.sorted_idx[leaf];
    const uint32_t sh = bv.shape[bi];
    return RqBody{{bv.pos_x[bi], bv.pos_y[bi], bv.pos_z[bi]},
                  {bv.rot_w[bi], bv.rot_x[bi], bv.rot_y[bi], bv.rot_z[bi]},
                  {sv.half_x[sh], sv.half_y[sh], sv.half_z[sh]},
                  sv.type[sh],
                  bi};
}

// Hit distance of the ray with a body, when it lies in [0, far); else negative.
__device__ __forceinline__ float rq_leaf(const RqBody &B, const float o[3], const float d[3], float far) {
    float t = -1.f;
    const float oc[3] = {o[0] - B.p[0], o[1] - B.p[1], o[2] - B.p[2]};
    if (B.type == kSphere) {
        const float r = B.h[0];
        const float a = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
        const float b = d[0] * oc[0] + d[1] * oc[1] + d[2] * oc[2];
        const float c = oc[0] * oc[0] + oc[1] * oc[1] + oc[2] * oc[2] - r * r;
        const float disc = b * b - a * c;
        if (disc >= 0.f) {
            const float sq = sqrtf(disc);
            t = (-b - sq) / a;
            if (t < 0.f) t = (-b + sq) / a;
            if (!(t >= 0.f && t < far)) t = -1.f;
        }
    } else {
        float lo[3], ld[3];
        rq_rotate_inv(B.q[0], B.q[1], B.q[2], B.q[3], oc, lo);
        rq_rotate_inv(B.q[0], B.q[1], B.q[2], B.q[3], d, ld);
        const float inv[3] = {1.f / ld[0], 1.f / ld[1], 1.f / ld[2]};
        const float mn[3] = {-B.h[0], -B.h[1], -B.h[2]};
        float tmin, tmax;
        rq_slab(lo, inv, mn, B.h, tmin, tmax);
        if (!(tmax < 0.f || tmin > tmax)) {
            t = tmin >= 0.f ? tmin : tmax;
            if (!(t >= 0.f && t < far)) t = -1.f;
        }
    }
    return t;
}

// The tree as the walk reads it: per internal node both children's boxes and
// numbers (2 x 16 B), per leaf its body (3 x 16 B).
struct RqRecords {
    uint4 *node;
    float4 *leaf;
};

// A node's box with its number.
__device__ __forceinline__ uint4 rq_child(const dy_bvh_view &bvh, int32_t c) {
    const uint4 nb = *reinterpret_cast<const uint4 *>(&bvh.aabb[c]);
    return make_uint4(nb.x, nb.y, nb.z, static_cast<uint32_t>(c));
}

__global__ __launch_bounds__(256) void ray_records(dy_bvh_view bvh, dy_body_view bv, dy_shape_view sv, RqRecords rec) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= bvh.n) return;
    if (k < bvh.n - 1u) {
        const uint4 l = rq_child(bvh, bvh.left[k]), r = rq_child(bvh, bvh.right[k]);
        rec.node[2 * static_cast<size_t>(k)] = l;
        rec.node[2 * static_cast<size_t>(k) + 1] = r;
    }
    const RqBody B = rq_body(bvh, bv, sv, k);
    float4 *f = rec.leaf + 3 * static_cast<size_t>(k);
    f[0] = make_float4(B.p[0], B.p[1], B.p[2], __uint_as_float(B.type));
    f[1] = make_float4(B.q[0], B.q[1], B.q[2], B.q[3]);
    f[2] = make_float4(B.h[0], B.h[1], B.h[2], __uint_as_float(B.body));
}

// True when the ray meets a node's box before best_t; entry distance in tmin.
// With `check`, `odd` is set when a slab distance is no number (an origin on
// the face's plane of a ray that runs along it, or infinite inputs): a box
// inside another then need not be entered later.
__device__ __forceinline__ bool rq_box(const uint4 &nb, const float o[3], const float inv[3], float best_t, float &tmin,
                                       bool check, bool &odd) {
    const float mn[3] = {f16_to_f32(static_cast<uint16_t>(nb.x & 0xffffu)),
                         f16_to_f32(static_cast<uint16_t>(nb.x >> 16)),
                         f16_to_f32(static_cast<uint16_t>(nb.y & 0xffffu))};
    const float mx[3] = {f16_to_f32(static_cast<uint16_t>(nb.y >> 16)),
                         f16_to_f32(static_cast<uint16_t>(nb.z & 0xffffu)),
                         f16_to_f32(static_cast<uint16_t>(nb.z >> 16))};
    float tmax;
    rq_slab(o, inv, mn, mx, tmin, tmax);
    if (check) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const float a = (mn[k] - o[k]) * inv[k], b = (mx[k] - o[k]) * inv[k];
            odd = odd || a != a || b != b;
        }
    }
    return tmax >= 0.f && tmax >= tmin && tmin < best_t;
}

// One ray's walk as the reference does it, by one lane, from the view's arrays.
__device__ __forceinline__ dy_ray_hit rq_walk(const dy_bvh_view &bvh, const dy_body_view &bv, const dy_shape_view &sv,
                                           const dy_ray &r) {
    const float o[3] = {r.ox, r.oy, r.oz}, d[3] = {r.dx, r.dy, r.dz};
    const float inv[3] = {1.f / r.dx, 1.f / r.dy, 1.f / r.dz};
    dy_ray_hit hit{r.t_max, 0xffffffffu};
    const uint32_t n = bvh.n;
    if (n == 0) return hit;
    int32_t stack[64];
    int top = 0;
    stack[top++] = n == 1 ? 0 : bvh.root[0];
    const uint32_t n_int = n - 1u;
    while (top > 0) {
        const int32_t node = stack[--top];
        float tmin;
        bool odd = false;
        if (n > 1 && !rq_box(rq_child(bvh, node), o, inv, hit.t, tmin, false, odd)) continue;
        if (static_cast<uint32_t>(node) >= n_int) {
            const RqBody B = rq_body(bvh, bv, sv, static_cast<uint32_t>(node) - n_int);
            const float t = rq_leaf(B, o, d, hit.t);
            if (t >= 0.f) hit = dy_ray_hit{t, B.body};
        } else if (top + 1 < 64) {
            stack[top++] = bvh.right[node];
            stack[top++] = bvh.left[node];
        }
    }
    return hit;
}

// The same out of line, for the rays that a team gives up.
__device__ __noinline__ dy_ray_hit rq_walk_apart(const dy_bvh_view &bvh, const dy_body_view &bv,
                                                 const dy_shape_view &sv, const dy_ray &r) {
    return rq_walk(bvh, bv, sv, r);
}

// One ray a lane: the form for many rays over few bodies (see ray_lanes).
__global__ __launch_bounds__(256) void ray_query_lanes(dy_bvh_view bvh, dy_body_view bv, dy_shape_view sv,
                                                       const dy_ray *__restrict__ rays, dy_ray_hit *__restrict__ hits,
                                                       uint32_t n_rays) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n_rays) hits[k] = rq_walk(bvh, bv, sv, rays[k]);
}

// A team of kRqTeam lanes walks one ray.  The reference's result is a fold over
// the leaves in order (left to right, leaf k is the k-th in Morton order):
// leaf k, entered at e_k and hit at t_k, replaces the best hit when
// m_k = max(e_k, t_k) lies before it.  (Its ancestors' boxes contain its box,
// so they are entered no later and pass whenever it does.)  So the team may
// visit the nodes in any order and fold the hits afterwards; and once leaf i is
// known, the best hit after it is at most m_i, so a subtree behind leaf i that
// is entered at m_i or later takes no part.  A body may reach out of its
// binary16 box, or have moved since the tree was built, so t_k may lie before
// e_k and the nearest hit is not always the one reported: the fold keeps the
// hits up to hits_reach, and a ray is walked by one lane if that turns out to
// reach a hit that had left the list.
//
// The team keeps a stack of internal nodes in LDS, the earliest in order on
// top; a step takes up to kRqTeam of them, tests both children of each, pushes
// the internal ones and collects the leaves, which are tested kRqTeam at a
// time.  Rays whose stack, leaves or hits outgrow the team's memory, and rays
// that met a slab distance that is no number, are walked by one lane.
//
// Bound by the rays' dependent loads: over a settled pile of 32 768 bodies a
// ray passes 206 internal nodes and 21 leaves on average and 1 274 and 342 at
// most, and one lane a ray waited for the longest of 64.  65 536 rays over it
// 1 247 -> 319 us, 500 rays over 40 000 bodies 1 016 -> 112 us, 200 000 rays over
// 5 000 bodies 612 -> 480 us.  Teams of 8 lanes: 379, 191 and 415 us; of 32: 504,
// 71 and 828.  A 64-entry stack sends enough rays to the walk by one lane to
// cost 628 us for the first.
constexpr uint32_t kRqTeam = 16, kRqTeams = 64u / kRqTeam;
constexpr uint32_t kRqStack = 128, kRqLeaves = 3u * kRqTeam, kRqHits = 2u * kRqTeam;

struct RqTeam {
    uint32_t node[kRqStack], first[kRqStack];  // internal node, its first leaf
    float enter[kRqStack];
    uint32_t leaf[kRqLeaves];
    float leaf_enter[kRqLeaves];
    float hit_m[kRqHits], hit_t[kRqHits];
    uint32_t hit_leaf[kRqHits], hit_body[kRqHits];
};

// A wavefront's LDS operations execute in program order; this holds the compiler to it.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Least value over the team's lanes.
__device__ __forceinline__ uint32_t team_min(uint32_t v) {
#pragma unroll
    for (uint32_t d = 1; d < kRqTeam; d <<= 1) {
        const uint32_t w = __shfl_xor(v, static_cast<int>(d), 64);
        v = w < v ? w : v;
    }
    return v;
}

// How far the hits reach that can decide the result: the least distance U, from
// the least m on, such that every hit at t <= U has m <= U.  Hits beyond U
// leave the best hit beyond U, which the others' m lie before, so they change
// nothing.  Two hits a lane (t infinite: none).
__device__ __forceinline__ float hits_reach(const float (&m)[2], const float (&t)[2], float least) {
    float reach = least;
    for (;;) {
        float far = reach;
#pragma unroll
        for (uint32_t q = 0; q < 2u; ++q)
            if (t[q] <= reach && m[q] > far) far = m[q];
#pragma unroll
        for (uint32_t d = 1; d < kRqTeam; d <<= 1) far = fmaxf(far, __shfl_xor(far, static_cast<int>(d), 64));
        const bool more = far > reach;
        reach = far;
        if (!__ballot(more)) return reach;
    }
}

template <bool RECORDS>
__global__ __launch_bounds__(64) void ray_query_kernel(dy_bvh_view bvh, dy_body_view bv, dy_shape_view sv, RqRecords rec,
                                                       const dy_ray *__restrict__ rays, dy_ray_hit *__restrict__ hits,
                                                       uint32_t n_rays) {
    __shared__ RqTeam teams[kRqTeams];
    const uint32_t lane = threadIdx.x, team = lane / kRqTeam, tl = lane % kRqTeam;
    const uint32_t k = blockIdx.x * kRqTeams + team;
    const uint32_t shift = team * kRqTeam;
    constexpr uint32_t kAll = kRqTeam == 32u ? ~0u : (1u << (kRqTeam & 31u)) - 1u;
    auto ballot = [&](bool p) { return static_cast<uint32_t>(__ballot(p) >> shift) & kAll; };
    RqTeam &S = teams[team];
    const bool mine = k < n_rays;
    const uint32_t n = bvh.n, n_int = n - 1u;
    dy_ray r{};
    if (mine) r = rays[k];
    const float o[3] = {r.ox, r.oy, r.oz}, d[3] = {r.dx, r.dy, r.dz};
    const float inv[3] = {1.f / r.dx, 1.f / r.dy, 1.f / r.dz};
    const float far = r.t_max;
    bool check = false;  // a slab distance may be no number
#pragma unroll
    for (int q = 0; q < 3; ++q) check = check || !(fabsf(inv[q]) <= 3.4e38f) || !(fabsf(o[q]) <= 3.4e38f);
    bool odd = n < 2u;
    uint32_t top = 0, n_leaf = 0, n_hit = 0;  // the same on every lane of the team
    float bound_m = far, dropped = INFINITY;  // least m so far; nearest hit that left the list
    uint32_t bound_leaf = 0xffffffffu;  // of the lane's own hits, then the team's
    if (mine && n > 1u) {
        float t0;
        const uint32_t root = static_cast<uint32_t>(bvh.root[0]);
        if (rq_box(rq_child(bvh, bvh.root[0]), o, inv, far, t0, check, odd)) {
            if (tl == 0) {
                S.node[0] = root;
                S.first[0] = 0u;
                S.enter[0] = t0;
            }
            top = 1;
        }
    }
    odd = ballot(odd) != 0u;
    const uint32_t above = kAll & ~((2u << tl) - 1u), below = (1u << tl) - 1u;  // the team's later, earlier lanes
    while (__ballot(!odd && (top | n_leaf))) {
        wave_sync();
        const bool run = !odd && (top | n_leaf) != 0u;
        const bool leaves = run && (n_leaf >= kRqTeam || top == 0u);
        const bool nodes = run && !leaves;
        // nodes: both children of up to kRqTeam entries
        bool pl = false, pr = false, ll = false, lr = false, over = false;
        uint32_t first = 0, lc = 0, rc = 0;
        float tl_ = 0.f, tr_ = 0.f;
        const uint32_t take = nodes ? (top < kRqTeam ? top : kRqTeam) : 0u;
        if (tl < take) {
            const uint32_t at = top - 1u - tl;
            const uint32_t node = S.node[at];
            first = S.first[at];
            if (!(first > bound_leaf && S.enter[at] >= bound_m)) {
                uint4 l, rt;
                if (RECORDS) {
                    l = rec.node[2 * static_cast<size_t>(node)];
                    rt = rec.node[2 * static_cast<size_t>(node) + 1];
                } else {
                    const int32_t li = bvh.left[node], ri = bvh.right[node];
                    l = rq_child(bvh, li);
                    rt = rq_child(bvh, ri);
                }
                lc = l.w;
                rc = rt.w;
                const bool hl = rq_box(l, o, inv, far, tl_, check, over), hr = rq_box(rt, o, inv, far, tr_, check, over);
                const uint32_t first_r = rc >= n_int ? rc - n_int : rc;  // an internal right child starts at its number
                pl = hl && lc < n_int;
                ll = hl && lc >= n_int;
                const bool cut = first_r > bound_leaf && tr_ >= bound_m;
                pr = hr && !cut && rc < n_int;
                lr = hr && !cut && rc >= n_int;
            }
        }
        top -= take;
        {
            // later lanes' entries go below earlier ones', right below left
            const uint32_t ml = ballot(pl), mr = ballot(pr);
            const uint32_t at = top + __popc(ml & above) + __popc(mr & above);
            const uint32_t grown = top + __popc(ml) + __popc(mr);
            if (grown > kRqStack) {
                over = true;
            } else {
                if (pr) {
                    S.node[at] = rc;
                    S.first[at] = rc;
                    S.enter[at] = tr_;
                }
                if (pl) {
                    const uint32_t q = at + (pr ? 1u : 0u);
                    S.node[q] = lc;
                    S.first[q] = first;
                    S.enter[q] = tl_;
                }
                top = grown;
            }
            const uint32_t kl = ballot(ll), kr = ballot(lr);
            const uint32_t lat = n_leaf + __popc(kl & below) + __popc(kr & below);
            if (n_leaf + __popc(kl) + __popc(kr) > kRqLeaves) {
                over = true;
            } else {
                if (ll) {
                    S.leaf[lat] = lc - n_int;
                    S.leaf_enter[lat] = tl_;
                }
                if (lr) {
                    S.leaf[lat + (ll ? 1u : 0u)] = rc - n_int;
                    S.leaf_enter[lat + (ll ? 1u : 0u)] = tr_;
                }
                if (nodes) n_leaf += __popc(kl) + __popc(kr);
            }
        }
        wave_sync();
        // leaves: up to kRqTeam exact tests
        const uint32_t give = leaves ? (n_leaf < kRqTeam ? n_leaf : kRqTeam) : 0u;
        bool hit = false;
        float t = -1.f, m = 0.f;
        uint32_t leaf = 0, body = 0;
        if (tl < give) {
            leaf = S.leaf[n_leaf - 1u - tl];
            const float e = S.leaf_enter[n_leaf - 1u - tl];
            if (!(leaf > bound_leaf && e >= bound_m)) {
                RqBody B;
                if (RECORDS) {
                    const float4 *f = rec.leaf + 3 * static_cast<size_t>(leaf);
                    const float4 f0 = f[0], f1 = f[1], f2 = f[2];
                    B = RqBody{{f0.x, f0.y, f0.z}, {f1.x, f1.y, f1.z, f1.w}, {f2.x, f2.y, f2.z},
                               __float_as_uint(f0.w), __float_as_uint(f2.w)};
                } else {
                    B = rq_body(bvh, bv, sv, leaf);
                }
                t = rq_leaf(B, o, d, far);
                m = e > t ? e : t;
                body = B.body;
                hit = t >= 0.f && !(leaf > bound_leaf && m >= bound_m);
            }
        }
        n_leaf -= give;
        const bool full = leaves && n_hit > kRqHits - kRqTeam;
        if (__ballot(full)) {
            // make room: hits beyond what the nearest ones reach leave
            float cm[2], ct[2];
            uint32_t cl[2], cb[2];
#pragma unroll
            for (uint32_t q = 0; q < 2u; ++q) {
                const uint32_t at = q * kRqTeam + tl;
                const bool v = full && at < n_hit;
                cm[q] = v ? S.hit_m[at] : 0.f;
                ct[q] = v ? S.hit_t[at] : INFINITY;
                cl[q] = S.hit_leaf[at];
                cb[q] = S.hit_body[at];
            }
            const float reach = hits_reach(cm, ct, bound_m);
            bool keep[2];
            float gone = INFINITY;
#pragma unroll
            for (uint32_t q = 0; q < 2u; ++q) {
                keep[q] = full && q * kRqTeam + tl < n_hit && ct[q] <= reach;
                if (full && q * kRqTeam + tl < n_hit && !keep[q] && ct[q] < gone) gone = ct[q];
            }
            gone = __uint_as_float(team_min(__float_as_uint(gone)));  // distances >= 0: their bits order as they do
            const uint32_t k0 = ballot(keep[0]), k1 = ballot(keep[1]);
            wave_sync();
#pragma unroll
            for (uint32_t q = 0; q < 2u; ++q)
                if (keep[q]) {
                    const uint32_t at = q ? __popc(k0) + __popc(k1 & below) : __popc(k0 & below);
                    S.hit_m[at] = cm[q];
                    S.hit_t[at] = ct[q];
                    S.hit_leaf[at] = cl[q];
                    S.hit_body[at] = cb[q];
                }
            if (full) {
                n_hit = __popc(k0) + __popc(k1);
                dropped = gone < dropped ? gone : dropped;
            }
            wave_sync();
        }
        const uint32_t mh = ballot(hit);
        if (n_hit + __popc(mh) > kRqHits) {
            over = true;
        } else if (hit) {
            const uint32_t at = n_hit + __popc(mh & below);
            S.hit_m[at] = m;
            S.hit_t[at] = t;
            S.hit_leaf[at] = leaf;
            S.hit_body[at] = body;
        }
        if (__ballot(hit)) {
            if (mh) {
                n_hit += __popc(mh);
                // the bound: the least m of the team (m >= 0, so its bits order as its value)
                const uint32_t b = team_min(hit ? __float_as_uint(m) : 0x7f800000u);
                const uint32_t who = ballot(hit && __float_as_uint(m) == b);
                const uint32_t src = shift + (who ? static_cast<uint32_t>(__ffs(who)) - 1u : 0u);
                const uint32_t bl = __shfl(leaf, static_cast<int>(src), 64);
                if (who && __uint_as_float(b) < bound_m) {
                    bound_m = __uint_as_float(b);
                    bound_leaf = bl;
                }
            }
        }
        odd = odd || ballot(over) != 0u;
    }
    // The fold: again and again the earliest leaf behind the last one taken that lies before the best hit.
    float best = far;
    uint32_t best_body = 0xffffffffu, next = 0;
    float hm[2], ht[2];
    uint32_t hl[2], hb[2];
    wave_sync();
#pragma unroll
    for (uint32_t q = 0; q < 2u; ++q) {
        const uint32_t at = q * kRqTeam + tl;
        const bool v = at < n_hit;
        hm[q] = v ? S.hit_m[at] : 0.f;
        ht[q] = v ? S.hit_t[at] : INFINITY;
        hl[q] = v ? S.hit_leaf[at] : 0xffffffffu;
        hb[q] = v ? S.hit_body[at] : 0u;
    }
    odd = odd || (n_hit != 0u && hits_reach(hm, ht, bound_m) >= dropped);
    for (;;) {
        uint32_t c = 0xffffffffu, q_mine = 0;
#pragma unroll
        for (uint32_t q = 0; q < 2u; ++q)
            if (hl[q] != 0xffffffffu && hl[q] >= next && hm[q] < best && hl[q] < c) {
                c = hl[q];
                q_mine = q;
            }
        const uint32_t least = team_min(c);
        if (!__ballot(least != 0xffffffffu)) break;
        const uint32_t who = ballot(c == least);
        const int src = static_cast<int>(shift + static_cast<uint32_t>(__ffs(who)) - 1u);
        const float tt = __shfl(q_mine ? ht[1] : ht[0], src, 64);
        const uint32_t bb = __shfl(q_mine ? hb[1] : hb[0], src, 64);
        if (least != 0xffffffffu) {
            best = tt;
            best_body = bb;
            next = least + 1u;
        }
    }
    if (mine && tl == 0) hits[k] = odd ? rq_walk_apart(bvh, bv, sv, r) : dy_ray_hit{best, best_body};
}

// One lane a ray (ray_query_lanes) or a team?  The lanes take as long as the
// longest walk however few the rays (20 us over 10 bodies, 300 over 1 000), and
// beyond a full chip 0.05 ns a ray over 10 bodies and 3 over 30 000; teams start
// at a tenth of that, and take 0.9 to 2.8 ns.  So many rays over few bodies are
// the lanes'.  Teams / lanes over a pile: 10 bodies 3 000 rays 16 / 19 us, 10 000
// rays 29 / 20; 100 bodies 30 000 rays 60 / 75, 200 000 rays 254 / 94; 1 000 bodies
// 100 000 rays 195 / 308, 200 000 rays 353 / 313; 8 000 bodies 400 000 rays
// 916 / 973, 800 000 rays 1 754 / 1 508; 30 000 bodies 2 000 000 rays 5 680 / 6 530.
// The lines follow the counts at which both took the same time.
static bool ray_lanes(uint32_t n, uint32_t n_rays) {
    const uint64_t m = n_rays;
    if (n <= 4u || m >= 550ull * n) return true;
    return n <= 16384u && m >= 60ull * n && m * m >= 5400ull * 5400ull * n;
}

// Rays of one launch: 16 threads each stay below the 2^32 threads that a grid may have.
constexpr uint32_t kRqLaunch = 1u << 27;

// launch(first, count) for the rays in runs that one grid can take.
template <class F>
static int ray_launches(uint32_t n_rays, F &&launch) {
    for (uint64_t k = 0; k < n_rays; k += kRqLaunch) {
        const uint64_t left = n_rays - k;
        launch(static_cast<size_t>(k), static_cast<uint32_t>(left < kRqLaunch ? left : kRqLaunch));
        DY_LAUNCH_CHECK();
    }
    return DY_OK;
}

}  // namespace dy

using namespace dy;

extern "C" {

int dy_ray_query(dy_stream_t s, const dy_bvh_view *bvh, const dy_body_view *bodies, const dy_shape_view *shapes,
                 const dy_ray *d_rays, dy_ray_hit *d_hits, uint32_t n_rays) {
    if (!bvh || !bodies || !shapes || (n_rays && (!d_rays || !d_hits))) return DY_ERR_INVALID_ARG;
    if (n_rays == 0) return DY_OK;
    if (bvh->n > bodies->n) return DY_ERR_INVALID_ARG;
    const uint32_t n = bvh->n;
    if (ray_lanes(n, n_rays))
        return ray_launches(n_rays, [&](size_t k, uint32_t m) {
            ray_query_lanes<<<ceil_div(m, 256), 256, 0, hs(s)>>>(*bvh, *bodies, *shapes, d_rays + k, d_hits + k, m);
        });
    const auto teams = [&](const RqRecords *rec) {
        return ray_launches(n_rays, [&](size_t k, uint32_t m) {
            const uint32_t blocks = ceil_div(m, kRqTeams);
            if (rec)
                ray_query_kernel<true><<<blocks, 64, 0, hs(s)>>>(*bvh, *bodies, *shapes, *rec, d_rays + k, d_hits + k, m);
            else
                ray_query_kernel<false><<<blocks, 64, 0, hs(s)>>>(*bvh, *bodies, *shapes, RqRecords{}, d_rays + k,
                                                                  d_hits + k, m);
        });
    };
    // Records are made for the call where enough rays read them (they cost an
    // allocation and a launch, about 33 us of a small call): 40 000 bodies with
    // 500 rays 117 us with and 112 without, 5 000 rays 153 / 182, 20 000 rays
    // 203 / 263; 1 000 bodies with 500 rays 67 / 34, 20 000 rays 73 / 83.  Not
    // under capture, where nothing is allocated, nor where memory is short.
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    const bool many = n_rays >= 4096u && n_rays >= n / 16u;
    if (many) DY_TRY(hipStreamIsCapturing(hs(s), &capture));
    if (!many || capture != hipStreamCaptureStatusNone) return teams(nullptr);
    uint4 *p = nullptr;
    if (hipMallocAsync(reinterpret_cast<void **>(&p), 5 * static_cast<size_t>(n) * sizeof(uint4), hs(s)) != hipSuccess) {
        (void)hipGetLastError();  // no room: the view's arrays will do
        return teams(nullptr);
    }
    const RqRecords rec{p, reinterpret_cast<float4 *>(p + 2 * static_cast<size_t>(n))};
    ray_records<<<ceil_div(n, 256), 256, 0, hs(s)>>>(*bvh, *bodies, *shapes, rec);
    const int st = teams(&rec);
    DY_TRY(hipFreeAsync(p, hs(s)));
    return st;
}

}  // extern "C"
