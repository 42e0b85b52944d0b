// rb_quad.h -- rays walked by quads of lanes: the parts of the traversal that the
// trace kernels (rb_trace.hip) and kernels that trace rays of their own
// (rb_bdpt.h) share.
#pragma once
#include "rb_device.h"

namespace rb {

// Global-memory pointer types.  A pointer read from memory (the LDS batch
// table) is generic to the compiler and loads through it become flat loads,
// which wait on both the vector-memory and the LDS counters; the scene and
// ray pointers of a lane are held in these types so every access is a
// global one.
// Plain clang vectors (no constructors) so the same loads compile in the
// host pass of the source.
typedef float V4f __attribute__((ext_vector_type(4)));
typedef int V4i __attribute__((ext_vector_type(4)));
typedef int V2i __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(1))) const V4f* GF4;
typedef __attribute__((address_space(1))) const V4i* GI4;
typedef __attribute__((address_space(1))) const uint32_t* GU32;
typedef __attribute__((address_space(1))) V2i* GI2;

// 1/x rounded to nearest even, equal to the IEEE division 1.0f / x: the
// hardware reciprocal refined by one fused Newton step, r + r * (1 - x * r).
// Wherever the refined value is a normal number it is the correctly rounded
// quotient (checked against the division for every one of the 2^32
// single-precision inputs on gfx950: 4,227,858,434 take this path, none
// differs).  Zero, subnormal, infinite and NaN inputs and |x| > 2^126 give a
// non-normal refined value and take the division.  5 instructions instead of
// the division's 11 on the common path.
__device__ __forceinline__ float rcp_rn(float x) {
    const float r = __builtin_amdgcn_rcpf(x);
    const float y = fmaf(fmaf(-x, r, 1.0f), r, r);
    if (__builtin_expect(__builtin_isnormal(y), 1)) return y;
    return 1.0f / x;
}

// Slab-span min / max as single instructions.  fminf / fmaxf on values that
// come from another basic block (the ray's tmin and the current hit
// distance) are preceded by a quieting copy of those operands on every node
// visit (IEEE mode: minNum must not see a signalling NaN); both operands
// here are quiet by construction (fused products, and tmin / hit distance
// quieted once per ray), so the instructions give what fminf / fmaxf give.
__device__ __forceinline__ float vmin_(float a, float b) {
    float r;
    asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ float vmax_(float a, float b) {
    float r;
    asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ float vmin3_(float a, float b, float c) {
    float r;
    asm("v_min3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
__device__ __forceinline__ float vmax3_(float a, float b, float c) {
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

// Distance of one plane of one of a wide record's children: its 8-bit step,
// picked from the lo and hi words by the selector into the low half, which as a
// half-precision number is q * 2^-24 (subnormal), goes straight into a
// mixed-precision fused multiply-add, q s + b (the record holds s * 2^24).
__device__ __forceinline__ float walk_plane(uint32_t lo, uint32_t hi, uint32_t sel, float s, float b) {
    typedef _Float16 H2 __attribute__((ext_vector_type(2)));
    const H2 p = __builtin_bit_cast(H2, __builtin_amdgcn_perm(hi, lo, sel));
    return fmaf((float)p.x, s, b);
}

// A value of another lane of the quad (lanes 4q..4q+3): of its lane 0 or 1,
// of the other lane of the pair, of the same lane of the other pair.
constexpr int kQuad0 = 0x00, kQuad1 = 0x55, kQuadXor1 = 0xB1, kQuadXor2 = 0x4E;
template <int PERM>
__device__ __forceinline__ int quad(int x) {
    return __builtin_amdgcn_mov_dpp(x, PERM, 0xF, 0xF, true);
}

// A ray in registers.
struct RayRegs {
    float ox, oy, oz, dx, dy, dz, tmin;
    float idx, idy, idz;     // reciprocal direction
    float oodx, oody, oodz;  // origin * reciprocal direction
};
__device__ __forceinline__ RayRegs ray_regs(V4f o, V4f d) {
    RayRegs r;
    r.ox = o.x, r.oy = o.y, r.oz = o.z;
    r.dx = d.x, r.dy = d.y, r.dz = d.z;
    // a quiet copy for the slab max (comparisons treat every NaN alike)
    r.tmin = __builtin_canonicalizef(o.w);
    const float ooeps = 0x1p-80f;
    r.idx = rcp_rn(fabsf(r.dx) > ooeps ? r.dx : copysignf(ooeps, r.dx));
    r.idy = rcp_rn(fabsf(r.dy) > ooeps ? r.dy : copysignf(ooeps, r.dy));
    r.idz = rcp_rn(fabsf(r.dz) > ooeps ? r.dz : copysignf(ooeps, r.dz));
    r.oodx = r.ox * r.idx;
    r.oody = r.oy * r.idy;
    r.oodz = r.oz * r.idz;
    return r;
}

// Whether a hit on reference `ref`, found over wide records, counts (leaf_boxes):
// its leaf's box passes the slab test.
__device__ __forceinline__ bool leaf_box_passes(GF4 boxes, uint32_t ref, float tmin, float idx, float idy, float idz,
                                                float oodx, float oody, float oodz) {
    const V4f a = boxes[2 * (size_t)ref], b = boxes[2 * (size_t)ref + 1];
    const float lox = fmaf(a.x, idx, -oodx), hix = fmaf(a.y, idx, -oodx);
    const float loy = fmaf(a.z, idy, -oody), hiy = fmaf(a.w, idy, -oody);
    const float loz = fmaf(b.x, idz, -oodz), hiz = fmaf(b.y, idz, -oodz);
    const float near = vmax3_(vmin_(lox, hix), vmin_(loy, hiy), vmax_(vmin_(loz, hiz), tmin));
    const float far = vmin3_(vmax_(lox, hix), vmax_(loy, hiy), vmax_(loz, hiz));
    return far >= near;
}
__device__ __forceinline__ bool leaf_box_passes(GF4 boxes, uint32_t ref, const RayRegs& r) {
    return leaf_box_passes(boxes, ref, r.tmin, r.idx, r.idy, r.idz, r.oodx, r.oody, r.oodz);
}

// What a walk over wide records has found: the hit, and the reference it lies
// on.
struct QuadHit {
    float t;
    int id, ref;
    bool strict;  // a hit counts only if its leaf's box passes: the ray is walked a second time
};

// One step of every quad of the wave: four lanes per ray, each testing one
// child of a record (two of them over the binary records) or one triangle of
// a leaf.  No lane branches: the wave skips the node or the triangle half when
// no lane is in it, and a lane with nothing to push stores to `spare`.  Steps
// and arithmetic of a ray and the order of its stack are trace_steps', so its
// result does not depend on which lanes took it.
// at_entry(e): where the quad keeps stack entry e (room entries).
template <bool WIDE, typename Entry>
__device__ __forceinline__ void quad_step(GF4 nodes, GF4 tris, const RayRegs& ray, bool an, int j, Entry at_entry,
                                          int room, int* spare, GF4 boxes, int& cur, int& sp, QuadHit& h, bool& full) {
    const float ox = ray.ox, oy = ray.oy, oz = ray.oz, dx = ray.dx, dy = ray.dy, dz = ray.dz, tmin = ray.tmin;
    const float idx_ = ray.idx, idy_ = ray.idy, idz_ = ray.idz;
    const float oodx = ray.oodx, oody = ray.oody, oodz = ray.oodz;
    const float hitT = h.t;
    const int hitId = h.id;
    const bool at_tri = cur < 0;
    const bool at_node = (uint32_t)cur < (uint32_t)kSentinel;
    const uint32_t l = ~(uint32_t)cur, cnt = l & 31u;
    const bool there = at_tri & ((uint32_t)j < cnt);
    // the node's record, or the lane's triangle
    const uint32_t rec = at_tri ? (l >> 5) + (there ? (uint32_t)j : 0u) : at_node ? (uint32_t)cur : 0u;
    const GF4 p = (at_tri ? tris : nodes) + 4 * (size_t)rec;
    const V4f r0 = p[0], r1 = p[1], r2 = p[2], r3 = p[3];
    // the entry that a pop at the end of this step takes
    const int upper = *at_entry(sp > 0 ? sp - 1 : 0);
    asm volatile("" ::"v"(r0.x), "v"(r1.x), "v"(r2.x), "v"(r3.x));

    bool pop = false;
    int next = cur;
    if (__ballot(at_tri) != 0) {  // (a branch of the wave: no lane is masked out)
        const float Oz = fmaf(-oz, r0.z, fmaf(-oy, r0.y, fmaf(-ox, r0.x, r0.w)));
        const float t = Oz * rcp_rn(fmaf(dz, r0.z, fmaf(dy, r0.y, dx * r0.x)));
        const float Ox = fmaf(oz, r1.z, fmaf(oy, r1.y, fmaf(ox, r1.x, r1.w)));
        const float Dx = fmaf(dz, r1.z, fmaf(dy, r1.y, dx * r1.x));
        const float u = fmaf(t, Dx, Ox);
        const float Oy = fmaf(oz, r2.z, fmaf(oy, r2.y, fmaf(ox, r2.x, r2.w)));
        const float Dy = fmaf(dz, r2.z, fmaf(dy, r2.y, dx * r2.x));
        const float v = fmaf(t, Dy, Oy);
        const int id = __float_as_int(r3.x);
        const float uv = u + v;
        bool hit = there & (t > tmin) & ((t < hitT) | ((t == hitT) & (id < hitId))) & (u >= 0.0f) & (v >= 0.0f) &
                   (uv <= 1.0f);
        bool found = false;
        if (__ballot(hit) != 0) {
            if (WIDE && __ballot(hit & h.strict) != 0)
                hit = hit & (!h.strict | leaf_box_passes(boxes, hit ? rec : 0u, ray));
            // one after the other the triangles would leave the nearest
            // hit (the lowest id on ties), or the first for any hit
            float tn = hit ? t : __builtin_inff();
            tn = vmin_(tn, __int_as_float(quad<kQuadXor1>(__float_as_int(tn))));
            tn = vmin_(tn, __int_as_float(quad<kQuadXor2>(__float_as_int(tn))));
            const int own = (hit & (an | (t == tn))) ? (an ? j : id) : 0x7FFFFFFF;
            const int o1 = quad<kQuadXor1>(own), p1 = o1 < own ? o1 : own;
            const int o2 = quad<kQuadXor2>(p1), best = o2 < p1 ? o2 : p1;
            found = best != 0x7FFFFFFF;
            const bool take = found & (own == best);
            int tb = take ? __float_as_int(t) : 0, ib = take ? id : 0;
            int rb = 0;
            if (WIDE) {
                rb = take ? (int)rec : 0;
                rb |= quad<kQuadXor1>(rb);
                rb |= quad<kQuadXor2>(rb);
            }
            tb |= quad<kQuadXor1>(tb);
            ib |= quad<kQuadXor1>(ib);
            tb |= quad<kQuadXor2>(tb);
            ib |= quad<kQuadXor2>(ib);
            h.t = found ? __int_as_float(tb) : h.t;
            h.id = found ? ib : h.id;
            h.ref = found ? rb : h.ref;
        }
        const bool over = found & an;
        pop = at_tri & (cnt <= 4) & !over;
        next = over ? kSentinel : at_tri ? (int)~(l + 124u) : cur;  // first + 4, count - 4
    }
    if (__ballot(at_node) != 0) {
        int link, first_link, top, at;
        bool push, none;
        if (WIDE) {
            const uint32_t lox = __float_as_uint(r1.z), hix = __float_as_uint(r1.w), loy = __float_as_uint(r2.x),
                           hiy = __float_as_uint(r2.y), loz = __float_as_uint(r2.z), hiz = __float_as_uint(r2.w);
            const float sx = r0.w * idx_, sy = r1.x * idy_, sz = r1.y * idz_;
            const float bx = fmaf(sx, 0.0f, fmaf(r0.x, idx_, -oodx));
            const float by = fmaf(sy, 0.0f, fmaf(r0.y, idy_, -oody));
            const float bz = fmaf(sz, 0.0f, fmaf(r0.z, idz_, -oodz));
            const uint32_t selx = 0x0C0C0C00u | ((idx_ < 0.0f ? 4 : 0) + j);
            const uint32_t sely = 0x0C0C0C00u | ((idy_ < 0.0f ? 4 : 0) + j);
            const uint32_t selz = 0x0C0C0C00u | ((idz_ < 0.0f ? 4 : 0) + j);
            const float nx = walk_plane(lox, hix, selx, sx, bx), fx = walk_plane(lox, hix, selx ^ 4, sx, bx);
            const float ny = walk_plane(loy, hiy, sely, sy, by), fy = walk_plane(loy, hiy, sely ^ 4, sy, by);
            const float nz = walk_plane(loz, hiz, selz, sz, bz), fz = walk_plane(loz, hiz, selz ^ 4, sz, bz);
            const int l01 = __float_as_int((j & 1) ? r3.y : r3.x), l23 = __float_as_int((j & 1) ? r3.w : r3.z);
            link = j < 2 ? l01 : l23;
            const float near = vmax3_(nx, ny, vmax_(nz, tmin));
            const float far = vmin3_(fx, fy, vmin_(fz, hitT));
            constexpr int kMiss = 0x7FFFFFFF;
            const int key = fmaf(fabsf(far), 0x1p-22f, far) >= near ? __float_as_int(near) : kMiss;
            // the three exchanges of trace_steps: (0, 1), (2, 3), then the
            // winners of both (the lower child on ties)
            const int kp = quad<kQuadXor1>(key);
            const bool won = (j & 1) ? key < kp : key <= kp;
            const int wk = key < kp ? key : kp, lk = key < kp ? kp : key;  // winner and loser of the pair
            const int ow = quad<kQuadXor2>(wk), ol = quad<kQuadXor2>(lk);
            const bool first = won & (j < 2 ? wk <= ow : wk < ow);
            const int lose_a = (j < 2 ? lk : ol) != kMiss, lose_b = (j < 2 ? ol : lk) != kMiss;
            // pushed: loser of (2, 3), loser of (0, 1), second winner
            push = (key != kMiss) & !first;
            at = sp + (won ? lose_a + lose_b : j < 2 ? lose_b : 0);
            top = sp + lose_a + lose_b + ((wk < ow ? ow : wk) != kMiss);
            first_link = first ? link : 0;
            first_link |= quad<kQuadXor1>(first_link);
            first_link |= quad<kQuadXor2>(first_link);
            none = (wk == kMiss) & (ow == kMiss);
        } else {
            const bool c = (j & 1) != 0;
            const float lx = c ? r1.x : r0.x, hx = c ? r1.y : r0.y, ly = c ? r1.z : r0.z, hy = c ? r1.w : r0.w;
            const float lz = c ? r2.z : r2.x, hz = c ? r2.w : r2.y;
            const int l0 = __float_as_int(r3.x), l1 = __float_as_int(r3.y);
            const float clox = fmaf(lx, idx_, -oodx), chix = fmaf(hx, idx_, -oodx);
            const float cloy = fmaf(ly, idy_, -oody), chiy = fmaf(hy, idy_, -oody);
            const float cloz = fmaf(lz, idz_, -oodz), chiz = fmaf(hz, idz_, -oodz);
            const float cmin = vmax3_(vmin_(clox, chix), vmin_(cloy, chiy), vmax_(vmin_(cloz, chiz), tmin));
            const float cmax = vmin3_(vmax_(clox, chix), vmax_(cloy, chiy), vmin_(vmax_(cloz, chiz), hitT));
            const int h = cmax >= cmin ? 1 : 0, m = __float_as_int(cmin);
            const bool t0 = quad<kQuad0>(h) != 0, t1 = quad<kQuad1>(h) != 0;
            const bool far_first =
                t1 & (!t0 | (__int_as_float(quad<kQuad1>(m)) < __int_as_float(quad<kQuad0>(m))));
            push = t0 & t1 & (j == 0);
            link = far_first ? l0 : l1;  // the farther one
            at = sp;
            top = sp + (t0 & t1);
            none = !t0 & !t1;
            first_link = far_first ? l1 : l0;
        }
        push = push & at_node;
        // (the upload refuses trees deep enough to fill the stack: a
        // launch that still did so is flagged, nothing written past it)
        full = full | (push & (at >= room));
        *((push & (at < room)) ? at_entry(at) : spare) = link;
        pop = at_node ? none : pop;
        next = at_node ? first_link : next;
        sp = at_node ? (top < room ? top : room) : sp;
    }
    cur = pop ? (sp == 0 ? kSentinel : upper) : next;
    sp -= pop & (sp > 0);
}

// Rows of four entries that a ray's stack can need.
inline uint32_t stack_rows(rb_bvh_t bvh, bool wide) { return ((wide ? bvh->wide_stack : bvh->stack) + 3) / 4; }
// LDS of a wave whose quads walk with such stacks.
inline size_t quad_lds(uint32_t rows) { return (rows + 1) * 64 * sizeof(int); }

// The walk of one ray per quad of the wave: cur is 0 for a quad whose ray
// starts and kSentinel for one whose ray has ended (or that has none); the
// result is h (h.id -1: a miss).  Steps are made while more than `until` quads
// have a ray under way.
// stack: quad_lds(rows) bytes; a quad's entry e lies in row e / 4, column e % 4
// of its four words, and the row behind the last takes the stores of lanes that
// have nothing to push.
template <bool WIDE>
__device__ __forceinline__ void quad_walk(GF4 nodes, GF4 tris, GF4 boxes, const RayRegs& r, bool an, int* stack,
                                          uint32_t rows, uint32_t until, int& cur, int& sp, QuadHit& h, bool& full) {
    const int lane = (int)__lane_id(), j = lane & 3;
    int* const own = stack + (lane & ~3);
    auto at_entry = [&](int e) -> int* { return own + (e >> 2) * 64 + (e & 3); };
    while ((uint32_t)__popcll(__ballot(cur != kSentinel)) > 4 * until)
        quad_step<WIDE>(nodes, tris, r, an, j, at_entry, 4 * (int)rows, stack + rows * 64 + lane, boxes, cur, sp, h,
                        full);
}

// Whether an ended walk over wide records has to be made again, strictly: the
// box of its hit's leaf does not pass.
__device__ __forceinline__ bool walk_again(GF4 boxes, const RayRegs& r, const QuadHit& h) {
    return h.id >= 0 && !h.strict && !leaf_box_passes(boxes, (uint32_t)h.ref, r);
}

}  // namespace rb
