// rb_trace.hip -- persistent while-while BVH traversal for gfx950 (wave64).
//
// The Aila-Laine persistent "while-while" kernel of renderbox2
// (src/accelerators/sbvh/kepler_dynamic_fetch.h:67-363) redesigned for CDNA4:
//  * work fetch: one ballot per wave, one atomic per `chunk` rays from the
//    wave's leader lane, rays handed to terminated lanes by ballot rank
//    (the reference does one atomic per warp refill, :99-153);
//  * traversal stack: entry 0..S-1 of each lane in LDS (lane-interleaved,
//    conflict-free), deeper entries in per-lane private memory (the
//    reference keeps all 64 entries in local memory, :62-71);
//  * nodes: the MI355X layout (4 x 16-byte loads per node, leaf size in the
//    32-bit link, no terminator rows);
//  * ties at equal t go to the lowest original triangle id; the reference
//    keeps the first one found (:264);
//  * the work counter lives in a per-launch slot that the last block resets
//    (the reference copies a zero into a global symbol before each launch,
//    cudatracer.cu:164-165), so concurrent launches and graph replays work;
//  * step loop: in one iteration every lane of a wave does one step of its
//    own ray, a node record or one triangle (trace_steps); records come in
//    through LDS, 64 bytes per cache access (stage_records); launches of few
//    rays give each ray four lanes (trace_quads);
//  * leaf order: a lane tests a leaf as soon as it reaches one, so every ray
//    visits nodes and leaves in the same order whatever the other rays of its
//    wave do -- the order of the single-ray restatement -- and results are
//    the same run to run.  SPEC = the reference's speculative form
//    (trace_spec: a lane holding a leaf keeps walking inner nodes until the
//    whole wave holds leaves, kepler_dynamic_fetch.h:222-243): the leaf order
//    then depends on the wave, and where a slab test rounds a box entry past
//    a hit inside it, which hit survives culling can change with it (rare;
//    ids and t may then differ);
//  * batched mode: one launch serves up to kMaxBatch ray batches against
//    different resident BVHs; every lane carries the batch its current ray
//    belongs to and that scene's pointers, so a wave can mix rays of several
//    scenes while it refills;
//  * paired mode: two queued ray sets of one BVH (an any-hit or closest-hit
//    set, then a closest-hit set) in one launch, so a render bounce pays
//    one launch's ramp-up and tail instead of two;
//  * top of the tree in LDS (speculative form): each block copies the first
//    lds_nodes node records (the layout stores them breadth-first) into LDS
//    at start and reads them from there.
// Arithmetic (fp32, explicit fmaf, reciprocals equal to the IEEE division)
// matches the oracle's restatement bit for bit.
#include <algorithm>

#include "rb_quad.h"

namespace rb {

struct TraceArgs {
    const float4* __restrict__ nodes;
    const float4* __restrict__ tris;  // 3 rows per reference (speculative walk), or 4 with the id (step loop)
    const uint32_t* __restrict__ index;
    const float4* __restrict__ rays;
    const uint8_t* __restrict__ mask;
    int2* __restrict__ hits;
    uint32_t* __restrict__ counts;
    uint32_t* counter;
    uint32_t* errors;  // RB_TRACE_ERR_* flags (device word), set on a traversal-stack overflow
    uint32_t n;
    const uint32_t* n_dev;  // when set, the ray count is read from device memory
    // paired launch: a second ray set (closest hit) after the first (any hit
    // when any0 is set, else closest hit)
    const float4* __restrict__ rays2;
    int2* __restrict__ hits2;
    const uint32_t* n_dev2;
    uint32_t any0;
    uint32_t chunk;
    uint32_t threshold;
    uint32_t leaf_gate;  // non-speculative: leave the inner-node phase once <= this many lanes still search
    uint32_t top_nodes;  // node records 0..top_nodes-1 are read from a copy in LDS
    uint32_t few;         // a launch of at most so many rays, known to the kernel only, gives each a quad
    uint32_t stack_rows;  // a ray's stack needs at most four times as many entries
    const float4* boxes;  // wide records: leaf_boxes
};

constexpr uint32_t kMaxBatch = 64;

struct BatchDesc {
    const float4* nodes;
    const float4* tris;
    const uint32_t* index;
    const float4* rays;
    int2* hits;
    const uint8_t* mask;    // rays with mask 0 report a miss untraced (NULL: none)
    const uint32_t* n_dev;  // ray count in device memory (NULL: n)
    uint32_t n;             // ray count, or the bound of *n_dev
    uint32_t start;         // first global ray index of the batch (set by the kernel)
    uint32_t any;           // 1: terminate on the first hit
    const float4* boxes;    // wide records: leaf_boxes
};

struct BatchTable {
    uint32_t nb;
    BatchDesc d[kMaxBatch];
};

// Distances of one plane of two of a wide record's children: their 8-bit
// steps, picked from the lo and hi words by the selector and spread by one
// byte permute to the two halves 0x00qq, which as half-precision numbers are
// q * 2^-24 (subnormal), go straight into a mixed-precision fused
// multiply-add each, q s + b (the record holds s * 2^24).
__device__ __forceinline__ void walk_planes(uint32_t lo, uint32_t hi, uint32_t sel, float s, float b, float t[2]) {
    typedef _Float16 H2 __attribute__((ext_vector_type(2)));
    const H2 p = __builtin_bit_cast(H2, __builtin_amdgcn_perm(hi, lo, sel));
    t[0] = fmaf((float)p.x, s, b);
    t[1] = fmaf((float)p.y, s, b);
}

// Every single-precision bit pattern through rcp_rn's fast path and through
// rcp_rn itself, against the division: out[0] += inputs whose refined
// reciprocal is taken, out[1] += inputs where either differs from 1.0f / x
// (NaN results count as equal whatever their payload).
__global__ __launch_bounds__(256) void k_rcp_check(unsigned long long* out) {
    __shared__ unsigned long long s_fast, s_bad;
    if (threadIdx.x == 0) {
        s_fast = 0;
        s_bad = 0;
    }
    __syncthreads();
    unsigned long long fast = 0, bad = 0;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t x = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; x < (1ull << 32); x += stride) {
        const float f = __uint_as_float((uint32_t)x);
        const float q = 1.0f / f;
        const float r = __builtin_amdgcn_rcpf(f);
        const float y = fmaf(fmaf(-f, r, 1.0f), r, r);
        if (__builtin_isnormal(y)) {
            fast++;
            if (__float_as_uint(y) != __float_as_uint(q)) bad++;
        }
        const float z = rcp_rn(f);
        if (!(__float_as_uint(z) == __float_as_uint(q) || (z != z && q != q))) bad++;
    }
    atomicAdd(&s_fast, fast);
    atomicAdd(&s_bad, bad);
    __syncthreads();
    if (threadIdx.x == 0) {
        atomicAdd(&out[0], s_fast);
        atomicAdd(&out[1], s_bad);
    }
}

// The last block out resets the launch's counters.
template <bool MULTI>
__device__ __forceinline__ void end_launch(const TraceArgs& a) {
    __syncthreads();
    if (threadIdx.x == 0) {
        __threadfence();
        if (atomicAdd(a.counter + 1, 1u) == gridDim.x - 1) {
            atomicExch(a.counter + 1, 0u);
            if (MULTI) {
                atomicExch(a.counter + 0, 0u);
            } else {
                // unrolled: as a loop it took the batched kernel from 71 to
                // 81 VGPRs (7 -> 5 waves per SIMD)
#pragma unroll
                for (uint32_t b = 0; b < kRayBands; b++) atomicExch(a.counter + kBandStride * (b + 1), 0u);
            }
        }
    }
}

// The traversal stack of a lane: entries 0..S-1 in LDS (lstack), deeper ones
// in private memory (spill).  The upload refuses trees deep enough to fill
// it, so the else branch of a push is unreachable for a library BVH; it
// flags the launch instead of writing past the stack.
#define RB_PUSH(v)                                            \
    do {                                                      \
        if (sp + 1 < kMaxStack) {                             \
            ++sp;                                             \
            if (sp < S)                                       \
                lstack[sp * BLOCK + tid] = (v);               \
            else                                              \
                spill[sp - S] = (v);                          \
        } else {                                              \
            atomicOr(a.errors, (uint32_t)RB_TRACE_ERR_STACK); \
        }                                                     \
    } while (0)
// Pops happen only at sp >= 0 (the sentinel at entry 0 ends the ray).  The
// LDS read is unconditional (the empty asm takes its value, so it cannot be
// folded away) and the spill read a separate branch: a select between the
// two arrays would become one generic (flat) load, which waits on both the
// vector-memory and the LDS counters.
#define RB_POP(dst)                                          \
    do {                                                     \
        int v_ = lstack[(sp < S ? sp : S - 1) * BLOCK + tid]; \
        asm volatile("" : "+v"(v_));                         \
        if (sp >= S) v_ = spill[sp - S];                     \
        (dst) = v_;                                          \
        --sp;                                                \
    } while (0)

// Claims of a wave on the launch's rays (wave-uniform).  The rays go to
// kRayBands bands in turn, kRunClaims claims at a time: a wave claims from the
// band of its XCD until that runs out, then from the next band in turn, so
// every ray is claimed exactly once.  Rays are traced nearly in order, so that
// a batched launch works on one or two of its scenes at a time (with eight
// contiguous bands, on up to eight, more than the Infinity Cache holds: 2.97
// against 3.48 Grays/s on four large scenes), neighbouring rays meet in one
// XCD's L2, and the claims spread over eight counters.  Measured against one
// counter for a batched launch, 1741 -> 1487 us on 64 batches of four scenes,
// 1397 -> 1340 on 32 of scenes of 1M triangles; and against eight contiguous
// bands for the others, whose last rays came from few of them: ambient
// occlusion 512x512 356 -> 345 us, 401x299 588 -> 575, 1920x1080 camera rays 402
// -> 398; a path-traced frame 18.8 ms with both, and 18.95 with a claim at a
// time.
constexpr uint32_t kRunClaims = 16;
struct RayPool {
    uint32_t next = 0, end = 0;  // claimed rays not handed out yet
    uint32_t band = 0;
    bool drained = false;  // nothing left to claim
    __device__ __forceinline__ void init() {
        asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(band));
        band &= kRayBands - 1;
    }
    // Hands rays to the lanes of mask m by rank; *mine is this lane's ray.
    // Returns whether this lane got one (lanes outside m: false).
    __device__ __forceinline__ bool take(const TraceArgs& a, uint32_t nrays, uint64_t m, uint32_t* mine) {
        const uint32_t lane = __lane_id();
        const uint32_t rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
        const uint32_t want = __popcll(m);
        const uint32_t avail = end - next;
        uint32_t base = next;  // lanes past the claimed ones: base + rank
        uint32_t got = want;
        *mine = base + rank;
        if (avail < want) {
            const int leader = __builtin_ctzll(m);
            base = nrays;  // every band claimed: nothing for the lanes past `avail`
            uint32_t lim = nrays;
            if ((int)lane == leader) {
                for (uint32_t t = 0; t < kRayBands; t++) {
                    const uint32_t o = atomicAdd(a.counter + kBandStride * (band + 1), a.chunk);
                    // (a run is whole claims, so a claim lies within one)
                    const uint32_t run = kRunClaims * a.chunk;
                    const uint32_t at = (o / run * kRayBands + band) * run + o % run;
                    if (o < nrays / kRayBands + run && at < nrays) {
                        base = at;
                        break;
                    }
                    band = (band + 1) % kRayBands;
                }
            }
            base = __builtin_amdgcn_readlane(base, leader);
            band = __builtin_amdgcn_readlane(band, leader);
            drained = base >= nrays;
            if (nrays - base > a.chunk) lim = base + a.chunk;
            const uint32_t more = want - avail < lim - base ? want - avail : lim - base;
            if (rank >= avail) *mine = base + (rank - avail);
            got = avail + more;
            next = base + more;
            end = lim;
        } else {
            next += want;
        }
        return ((m >> lane) & 1u) && rank < got;
    }
};

// One 64-byte record per lane (rec, 64-byte aligned) into the wave's 4 KB of
// LDS: load k brings the records of lane k of every quad, its quad's lanes
// 16 bytes each, row (j ^ k) of it at 16-byte slot j of the quad's 64 bytes,
// so the lanes of a quad read one row of theirs from different banks.  The L1
// cache serves a record with one 64-byte access this way; 16 bytes per lane of
// 64 records are 64 accesses per load, and their rate bound large launches:
// 340 M -> 130 M accesses on 2 Mi diffuse rays at 1M triangles, 745 -> 684 us,
// and a path-traced frame of 2M triangles 24.1 -> 19.3 ms.
__device__ __forceinline__ void stage_records(const V4f* rec, uint32_t lane, V4f* stage) {
    const uint64_t p = (uint64_t)rec;
    const int lo = (int)(uint32_t)p, hi = (int)(uint32_t)(p >> 32);
    const uint32_t row = (lane & 3) * 16;
#define RB_STAGE(k)                                                                                            \
    do {                                                                                                       \
        const uint32_t l_ = (uint32_t)__builtin_amdgcn_mov_dpp(lo, 0x55 * (k), 0xF, 0xF, true) | (row ^ (16 * (k))); \
        const uint32_t h_ = (uint32_t)__builtin_amdgcn_mov_dpp(hi, 0x55 * (k), 0xF, 0xF, true);                 \
        const uint64_t q_ = (uint64_t)h_ << 32 | l_;                                                           \
        __builtin_amdgcn_global_load_lds((__attribute__((address_space(1))) void*)q_,                          \
                                         (__attribute__((address_space(3))) void*)(stage + 64 * (k)), 16, 0, 0); \
    } while (0)
    RB_STAGE(0);
    RB_STAGE(1);
    RB_STAGE(2);
    RB_STAGE(3);
#undef RB_STAGE
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// The step loop for launches of few rays: four lanes per ray from the start,
// sixteen rays per one-wave block, no refill and so no work counters.
//
// With a lane per ray such a launch takes as long as its longest ray, whose
// steps wait for each other: 0.78 us a step, the chain of its instructions
// (8-10 cycles for each that needs the one before, 80 for each branch that
// part of the lanes take) and a record from L2 (240).  With a quad per ray a
// leaf of four triangles is one step and no lane branches: 0.37 us a step.
// Two children per record leave half of the quad idle, but keep the latency.
//
// Measured, a lane per ray throughout -> a quad for each wave's last rays
// (trace_steps) -> quads throughout (us), rays from surfaces among 1M
// triangles: 64 rays 109 -> 83 -> 54, 16 Ki 173 -> 132 -> 95, 64 Ki 196 -> 153
// -> 129, 128 Ki 226 -> 178 -> 186, 256 Ki 281 -> 226 -> 282; first camera rays
// of 200k triangles: 32 Ki 30 -> 22 -> 9, 128 Ki 50 -> 51 -> 24, 256 Ki 106 ->
// 97 -> 66; 4099 rays of 20k triangles 107 -> 83 -> 48.  Any hit over the
// binary records: 128 Ki 322 -> 262 -> 252, 192 Ki 346 -> 286 -> 336.  (Quads
// are bound by VALU issue from about 100k rays on: a node step is 105
// instructions for 16 rays, in the other loop 115 for up to 64.)  Rows of the
// stack for what the tree can need, not for the most any tree may: 4 KB a wave
// for 1M triangles, so that eight waves fit a SIMD (256 Ki rays 292 -> 282).
template <bool ANY_T, bool MULTI, bool PAIR, bool WIDE>
__device__ __forceinline__ void trace_quads(const TraceArgs& a, const BatchDesc* tab, uint32_t nb, uint32_t nrays,
                                            uint32_t n0, int* lstack, uint32_t group) {
    const int lane = (int)__lane_id(), j = lane & 3;
    uint32_t mine = group * 16 + ((uint32_t)lane >> 2);
    const bool live = mine < nrays;
    mine = live ? mine : 0u;
    uint32_t batch = 0;
    if (MULTI) {  // the last batch starting at or before `mine` (empty batches share their successor's start)
        uint32_t lo = 0, hi = nb;
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) >> 1;
            if (tab[mid].start <= mine) lo = mid;
            else hi = mid;
        }
        batch = lo;
    }
    const bool second = PAIR && mine >= n0;
    const bool an = MULTI ? tab[batch].any != 0 : PAIR ? !second && a.any0 != 0 : ANY_T;
    const GF4 nodes = MULTI ? (GF4)tab[batch].nodes : (GF4)a.nodes;
    const GF4 tris = MULTI ? (GF4)tab[batch].tris : (GF4)a.tris;
    const GF4 rays = MULTI ? (GF4)tab[batch].rays : second ? (GF4)a.rays2 : (GF4)a.rays;
    const uint8_t* const mk = MULTI ? tab[batch].mask : a.mask;
    const size_t ray = MULTI ? mine - tab[batch].start : second ? mine - n0 : mine;
    const V4f o = rays[2 * ray], d = rays[2 * ray + 1];
    const RayRegs r = ray_regs(o, d);
    const float hitT = __builtin_canonicalizef(d.w);
    const GF4 boxes = MULTI ? (GF4)tab[batch].boxes : (GF4)a.boxes;
    int cur = live && !(mk && mk[ray] == 0) ? 0 : kSentinel, sp = 0;
    QuadHit hit = {hitT, -1, 0, false};
    bool full = false;
    while (true) {
        quad_walk<WIDE>(nodes, tris, boxes, r, an, lstack, a.stack_rows, 0, cur, sp, hit, full);
        const bool again = WIDE && walk_again(boxes, r, hit);
        if (__ballot(again) == 0) break;
        if (again) {
            hit = {hitT, -1, 0, true};
            sp = 0;
            cur = 0;
        }
    }
    if (full) atomicOr(a.errors, (uint32_t)RB_TRACE_ERR_STACK);
    if (live && j == 0) {
        V2i h;
        h.x = hit.id;
        // a miss reports the caller's tmax, bit for bit
        h.y = hit.id < 0 ? __float_as_int(((const __attribute__((address_space(1))) float*)(rays + 2 * ray + 1))[3])
                         : __float_as_int(hit.t);
        const GI2 hits = MULTI ? (GI2)tab[batch].hits : second ? (GI2)a.hits2 : (GI2)a.hits;
        hits[ray] = h;
    }
}

// One traversal body for every launch form but the speculative one.
// PAIR: rays [0, n0) are the first set (a.rays / a.hits; any hit when
// a.any0), rays [n0, nrays) the closest-hit set (a.rays2 / a.hits2).
// WIDE: a.nodes holds wide (4-child) records; for closest hit, whose (id, t)
// does not depend on the visit order, and for occlusion sets (any hit read
// only as hit / miss).
//
// A step loop: in one iteration every lane of the wave does one step of its
// own ray, a node record or one triangle of a leaf, and the records of both
// kinds are loaded together before either kind of step runs.  The launch is
// bound by VALU issue (2 Mi diffuse rays, 1M triangles: 85% of the issue
// slots; 337 M instructions per launch), with the drain of the last rays
// behind it, so what counts is instructions per step and the lanes each
// instruction serves.  Measured on that launch against a node loop and a leaf
// loop in turn over power-of-two records (lanes that reached a leaf waited
// for the rest, lanes without one for the longest leaf): 504 M instructions
// and 36% of their lanes at work before, 0.935 -> 0.684 ms; 1920x1080 camera
// rays of 200k triangles 0.486 -> 0.410 ms; a 1024x1024x8-spp path-traced
// frame of 2M triangles 21.9 -> 19.3 ms.  Tried and left out: the top of the
// tree in LDS (a branch per step, more than it saved), and waves of a
// workgroup joining their last rays in one of them (720 against 684 us: the
// drain waits for the longest ray's steps, not for issue slots).  So once no
// rays are left to claim and sixteen or fewer of the wave's are under way, each
// of those gets a quad of lanes (quad_step), whose steps are half as long: 2 Mi
// diffuse rays 671 -> 610 us, as any hit 559 -> 501, 512 Ki of them 349 -> 280,
// the camera rays 402 -> 389, the path-traced frame 18.8 -> 18.5 ms.  A ray
// still tests its nodes and leaves in its own order, whatever the other rays
// of its wave do, so results are the same run to run and launch shape to
// launch shape.
template <bool ANY_T, bool COUNT, int S, int BLOCK, bool MULTI, bool PAIR, bool WIDE>
__device__ __forceinline__ void trace_steps(const TraceArgs& a, const BatchDesc* tab, uint32_t nb, uint32_t n_rays,
                                            uint32_t n0 = 0) {
    // the stack: S - 1 entries of each lane in LDS, lane-interleaved, deeper
    // ones in private memory; empty, it gives the sentinel that ends the ray.
    // (With S = 12, a lane in most waves is past the straight-line stores of
    // a push and the wave goes through the branches of the deep ones; 15 rows
    // are the most that keep 20 waves on a CU, which 16 did not: 671 us on 2
    // Mi diffuse rays against 684 with 12 and 720 with 16)
    constexpr int R = S - 1;
    constexpr int kLds = (16 + R) * BLOCK;  // words
    __shared__ V4f staged[kLds / 4];
    int* const lds = (int*)staged;
    int* const lstack = lds + 16 * BLOCK;
    int spill[kMaxStack - 1 - R];
    constexpr int kDeep = 48;  // a quad's entries past those, once a wave has given its last rays a quad each
    const int tid = threadIdx.x;
    const uint32_t lane = __lane_id();
    // this wave's 64 staged records (wave-uniform), and where this lane's lies
    V4f* const stage = staged + 256 * __builtin_amdgcn_readfirstlane(tid >> 6);
    const V4f* const mine_staged = stage + 64 * (lane & 3) + 4 * (lane >> 2);

    const uint32_t nrays = __builtin_amdgcn_readfirstlane(n_rays);
    if (!COUNT && (MULTI || PAIR) && nrays <= a.few) {
        const uint32_t wave = blockIdx.x * (BLOCK / 64) + (uint32_t)__builtin_amdgcn_readfirstlane(tid >> 6);
        for (uint32_t g = wave; g * 16 < nrays; g += gridDim.x * (BLOCK / 64))
            trace_quads<ANY_T, MULTI, PAIR, WIDE>(a, tab, nb, nrays, n0, lds + (tid >> 6) * (kLds / (BLOCK / 64)), g);
        return;
    }
    RayPool pool;
    pool.init();
    // cur: the ray's next step -- an inner record (>= 0), a leaf's remaining
    // triangles ~(first << 5 | count), or kSentinel when the ray is done
    int cur = kSentinel, sp = 0, hitId = -1;
    int hitRef = 0;       // WIDE: as QuadHit's
    bool strict = false;  // WIDE: likewise
    bool live = false;  // the lane holds a ray whose result is not stored yet
    uint32_t mine = 0;  // the ray's index in the launch
    uint32_t batch = 0;  // MULTI: its batch
    float ox = 0.f, oy = 0.f, oz = 0.f, tmin = 0.f, dx = 0.f, dy = 0.f, dz = 0.f, hitT = 0.f;
    float idx_ = 0.f, idy_ = 0.f, idz_ = 0.f, oodx = 0.f, oody = 0.f, oodz = 0.f;
    // byte selectors of a wide record's near and far planes by the sign of the
    // direction (walk_planes): per axis near of children 0 and 1, of 2 and 3,
    // far of both.  Set per ray: twelve registers for fifteen instructions
    // less per record
    uint32_t sel[3][4] = {};
    uint32_t c_inner = 0, c_tri = 0, c_leaf = 0;
    // scene of the lane's current ray (uniform in single-batch mode); a lane
    // that has had no ray yet still loads a record with its quad, the first
    // scene's root
    GF4 nodes = MULTI ? (GF4)tab[0].nodes : (GF4)a.nodes;
    GF4 tris = MULTI ? (GF4)tab[0].tris : (GF4)a.tris;
    // where the lane's ray came from: looked up again at its rare uses
    // instead of carried in registers through every step
    auto second = [&]() -> bool { return PAIR && mine >= n0; };
    auto any = [&]() -> bool { return MULTI ? tab[batch].any != 0 : PAIR ? !second() && a.any0 != 0 : ANY_T; };
    auto rayidx = [&]() -> uint32_t { return MULTI ? mine - tab[batch].start : second() ? mine - n0 : mine; };
    auto rays = [&]() -> GF4 { return MULTI ? (GF4)tab[batch].rays : second() ? (GF4)a.rays2 : (GF4)a.rays; };
    auto boxes = [&]() -> GF4 { return MULTI ? (GF4)tab[batch].boxes : (GF4)a.boxes; };
    auto hits = [&]() -> GI2 { return MULTI ? (GI2)tab[batch].hits : second() ? (GI2)a.hits2 : (GI2)a.hits; };

    // The upload refuses trees deep enough to fill the stack, so the last
    // branch is unreachable for a library BVH; it flags the launch instead of
    // writing past the stack.
    auto push = [&](int v) {
        if (sp < R)
            lstack[sp++ * BLOCK + tid] = v;
        else if (sp < kMaxStack - 1)
            spill[sp++ - R] = v;
        else
            atomicOr(a.errors, (uint32_t)RB_TRACE_ERR_STACK);
    };
    // The LDS read is unconditional (the empty asm takes its value, so it
    // cannot be folded away) and the spill read a separate branch: a select
    // between the two arrays would become one generic (flat) load, which
    // waits on both the vector-memory and the LDS counters.
    auto pop_entry = [&]() -> int {
        --sp;
        int v = lstack[((uint32_t)sp < (uint32_t)R ? sp : R - 1) * BLOCK + tid];
        asm volatile("" : "+v"(v));
        if (sp >= R) v = spill[sp - R];
        return sp < 0 ? kSentinel : v;
    };

    // the finished ray's result
    auto store = [&]() {
        const size_t i = rayidx();
        V2i r;
        if (hitId < 0) {  // a miss reports the caller's tmax, bit for bit
            r.x = -1;
            r.y = __float_as_int(((const __attribute__((address_space(1))) float*)(rays() + 2 * i + 1))[3]);
        } else {
            r.x = hitId;
            r.y = __float_as_int(hitT);
        }
        hits()[i] = r;
        if (COUNT) {
            a.counts[3 * i + 0] = c_inner;
            a.counts[3 * i + 1] = c_tri;
            a.counts[3 * i + 2] = c_leaf;
        }
        live = false;
    };

    uint32_t left = 0;  // rays that the loop leaves to the wave's quads
    const uint32_t tail = COUNT || 4 * a.stack_rows > (uint32_t)(R + kDeep) ? 0 : 16;
    while (true) {
        // ---- refill (wave-uniform control): results of the finished rays
        // out, new rays in, once too few lanes are busy ----
        const uint64_t tm = __ballot(cur == kSentinel);
        const uint32_t busy = 64 - __popcll(tm);
        if (busy == 0 || (pool.drained ? busy <= tail : busy < a.threshold)) {
            if (WIDE) {
                // hits that may not count (leaf_boxes): those rays again
                bool again = false;
                if (cur == kSentinel && live && hitId >= 0 && !strict)
                    again = !leaf_box_passes(boxes(), (uint32_t)hitRef, tmin, idx_, idy_, idz_, oodx, oody, oodz);
                if (__ballot(again) != 0) {
                    if (again) {
                        hitT = __builtin_canonicalizef(
                            ((const __attribute__((address_space(1))) float*)(rays() + 2 * (size_t)rayidx() + 1))[3]);
                        hitId = -1;
                        strict = true;
                        sp = 0;
                        cur = 0;
                    }
                    continue;
                }
            }
            if (cur == kSentinel && live) store();
            uint32_t done = pool.drained;
            if (!COUNT && done && busy) {
                // what is left of the wave's rays to LDS, for the quads below.
                // (The value below is opaque so that this stays in the loop:
                // used on the way out, every register of the ray would be
                // copied twice per step)
                asm volatile("" ::: "memory");
                const uint32_t rank =
                    __builtin_amdgcn_mbcnt_hi((uint32_t)(~tm >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)~tm, 0u));
                if (cur != kSentinel) {
                    V4f* const to = stage + 16 * rank;
                    to[0] = V4f{ox, oy, oz, tmin};
                    to[1] = V4f{dx, dy, dz, hitT};
                    to[2] = __builtin_bit_cast(V4f, V4i{hitId, cur, sp, (int)mine});
                    to[3] = __builtin_bit_cast(V4f, V4i{(int)batch, (int)lane, hitRef, strict ? 1 : 0});
                    for (int e = R; e < sp; e++) ((int*)to)[16 + e - R] = spill[e - R];
                }
                asm volatile("" ::: "memory");
            }
            asm volatile("" : "+s"(done));
            if (done) {
                left = busy;
                break;
            }
            uint32_t ray;
            if (pool.take(a, nrays, tm, &ray)) {
                mine = ray;
                const uint8_t* mk = a.mask;
                if (MULTI) {
                    // the last batch starting at or before `mine` (empty
                    // batches share their successor's start)
                    uint32_t lo = 0, hi = nb;
                    while (hi - lo > 1) {
                        const uint32_t mid = (lo + hi) >> 1;
                        if (tab[mid].start <= mine) lo = mid;
                        else hi = mid;
                    }
                    batch = lo;
                    nodes = (GF4)tab[lo].nodes;
                    tris = (GF4)tab[lo].tris;
                    mk = tab[lo].mask;
                }
                const uint32_t i = rayidx();
                const V4f o = rays()[2 * (size_t)i];
                const V4f d = rays()[2 * (size_t)i + 1];
                ox = o.x; oy = o.y; oz = o.z;
                dx = d.x; dy = d.y; dz = d.z;
                // quiet copies for the slab min / max (comparisons treat every
                // NaN alike)
                tmin = __builtin_canonicalizef(o.w);
                hitT = __builtin_canonicalizef(d.w);
                const float ooeps = 0x1p-80f;
                idx_ = rcp_rn(fabsf(dx) > ooeps ? dx : copysignf(ooeps, dx));
                idy_ = rcp_rn(fabsf(dy) > ooeps ? dy : copysignf(ooeps, dy));
                idz_ = rcp_rn(fabsf(dz) > ooeps ? dz : copysignf(ooeps, dz));
                oodx = ox * idx_;
                oody = oy * idy_;
                oodz = oz * idz_;
                if (WIDE) {
                    const float dir[3] = {idx_, idy_, idz_};
#pragma unroll
                    for (int c = 0; c < 3; c++) {
                        const bool neg = dir[c] < 0.0f;
                        sel[c][0] = neg ? 0x0C050C04u : 0x0C010C00u;
                        sel[c][1] = neg ? 0x0C070C06u : 0x0C030C02u;
                        sel[c][2] = neg ? 0x0C010C00u : 0x0C050C04u;
                        sel[c][3] = neg ? 0x0C030C02u : 0x0C070C06u;
                    }
                }
                sp = 0;
                hitId = -1;
                strict = false;
                live = true;
                cur = (mk && mk[i] == 0) ? kSentinel : 0;
                if (COUNT) { c_inner = 0; c_tri = 0; c_leaf = 0; }
            }
            continue;
        }

        // ---- one step of every busy lane's ray ----
        const bool at_node = (uint32_t)cur < (uint32_t)kSentinel;
        // triangles wait until few enough lanes are at a node
        const bool tri_now = __popcll(__ballot(at_node)) <= a.leaf_gate;
        const bool at_tri = tri_now && cur < 0;
        const V4f* const rec = (const V4f*)(at_tri ? tris + 4 * (size_t)(~(uint32_t)cur >> 5)
                                                   : nodes + 4 * (size_t)(at_node ? cur : 0));
        stage_records(rec, lane, stage);
        const V4f r0 = mine_staged[0 ^ (lane & 3)], r1 = mine_staged[1 ^ (lane & 3)], r2 = mine_staged[2 ^ (lane & 3)],
                  r3 = mine_staged[3 ^ (lane & 3)];
        asm volatile("" ::"v"(r0.x), "v"(r1.x), "v"(r2.x), "v"(r3.x) : "memory");
        bool pop = false;
        if (at_node) {
            if (COUNT) c_inner++;
            const V4i lk4 = __builtin_bit_cast(V4i, r3);
            if (WIDE) {
                // the four children's slab tests, then the nearest hit child
                // next and the others pushed
                const V4i q1 = __builtin_bit_cast(V4i, r1), q2 = __builtin_bit_cast(V4i, r2);
                const float sx = r0.w * idx_, sy = r1.x * idy_, sz = r1.y * idz_;
                // (a step that overflows, a scene past 4e9 units and a ray
                // along an axis plane, makes its axis NaN, which the min and
                // max below leave out: the box is not culled by that axis)
                const float bx = fmaf(sx, 0.0f, fmaf(r0.x, idx_, -oodx));
                const float by = fmaf(sy, 0.0f, fmaf(r0.y, idy_, -oody));
                const float bz = fmaf(sz, 0.0f, fmaf(r0.z, idz_, -oodz));
                int lnk[4] = {lk4.x, lk4.y, lk4.z, lk4.w};
                int key[4];  // entry distance as an integer (in order from 0 up), kMiss past every float
                constexpr int kMiss = 0x7FFFFFFF;
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    float nx[2], ny[2], nz[2], fx[2], fy[2], fz[2];
                    walk_planes(q1.z, q1.w, sel[0][h], sx, bx, nx);
                    walk_planes(q2.x, q2.y, sel[1][h], sy, by, ny);
                    walk_planes(q2.z, q2.w, sel[2][h], sz, bz, nz);
                    walk_planes(q1.z, q1.w, sel[0][2 + h], sx, bx, fx);
                    walk_planes(q2.x, q2.y, sel[1][2 + h], sy, by, fy);
                    walk_planes(q2.z, q2.w, sel[2][2 + h], sz, bz, fz);
#pragma unroll
                    for (int c = 0; c < 2; c++) {
                        const float near = vmax3_(nx[c], ny[c], vmax_(nz[c], tmin));
                        const float far = vmin3_(fx[c], fy[c], vmin_(fz[c], hitT));
                        key[2 * h + c] = fmaf(fabsf(far), 0x1p-22f, far) >= near ? __float_as_int(near) : kMiss;
                    }
                    // two children at a time: all four at once take 89
                    // registers, past the 80 that six waves per SIMD leave
                    __builtin_amdgcn_sched_barrier(0);
                }
                // the nearest to slot 0, the next candidate to slot 2: the
                // full sort (two more exchanges) reads 1.5-2% fewer records,
                // less than its instructions cost
#define RB_CS(i, j)                 \
    if (key[j] < key[i]) {          \
        const int tk = key[i];      \
        key[i] = key[j];            \
        key[j] = tk;                \
        const int tl = lnk[i];      \
        lnk[i] = lnk[j];            \
        lnk[j] = tl;                \
    }
                RB_CS(0, 1) RB_CS(2, 3) RB_CS(0, 2)
#undef RB_CS
                if (key[0] == kMiss) {
                    pop = true;
                } else {
                    cur = lnk[0];
                    if (sp + 3 <= R) {
                        // straight-line stores: one of a missed child is
                        // above the new top and overwritten by the next
                        lstack[sp * BLOCK + tid] = lnk[3];
                        sp += key[3] != kMiss;
                        lstack[sp * BLOCK + tid] = lnk[1];
                        sp += key[1] != kMiss;
                        lstack[sp * BLOCK + tid] = lnk[2];
                        sp += key[2] != kMiss;
                    } else {
                        if (key[3] != kMiss) push(lnk[3]);
                        if (key[1] != kMiss) push(lnk[1]);
                        if (key[2] != kMiss) push(lnk[2]);
                    }
                }
            } else {
                const float c0lox = fmaf(r0.x, idx_, -oodx), c0hix = fmaf(r0.y, idx_, -oodx);
                const float c0loy = fmaf(r0.z, idy_, -oody), c0hiy = fmaf(r0.w, idy_, -oody);
                const float c0loz = fmaf(r2.x, idz_, -oodz), c0hiz = fmaf(r2.y, idz_, -oodz);
                const float c1loz = fmaf(r2.z, idz_, -oodz), c1hiz = fmaf(r2.w, idz_, -oodz);
                const float c1lox = fmaf(r1.x, idx_, -oodx), c1hix = fmaf(r1.y, idx_, -oodx);
                const float c1loy = fmaf(r1.z, idy_, -oody), c1hiy = fmaf(r1.w, idy_, -oody);
                const float c0min = vmax3_(vmin_(c0lox, c0hix), vmin_(c0loy, c0hiy), vmax_(vmin_(c0loz, c0hiz), tmin));
                const float c0max = vmin3_(vmax_(c0lox, c0hix), vmax_(c0loy, c0hiy), vmin_(vmax_(c0loz, c0hiz), hitT));
                const float c1min = vmax3_(vmin_(c1lox, c1hix), vmin_(c1loy, c1hiy), vmax_(vmin_(c1loz, c1hiz), tmin));
                const float c1max = vmin3_(vmax_(c1lox, c1hix), vmax_(c1loy, c1hiy), vmin_(vmax_(c1loz, c1hiz), hitT));
                const bool swp = c1min < c0min;
                const bool t0 = c0max >= c0min;
                const bool t1 = c1max >= c1min;
                if (!t0 && !t1) {
                    pop = true;
                } else {
                    const bool second = t1 && (!t0 || swp);
                    cur = second ? lk4.y : lk4.x;
                    if (t0 && t1) push(second ? lk4.x : lk4.y);
                }
            }
            if (COUNT && !pop && cur < 0) c_leaf++;
        }
        if (at_tri) {
            const uint32_t l = ~(uint32_t)cur;
            const int id = __float_as_int(r3.x);
            // (binary records may link an empty leaf: count 0; its record is the
            // next leaf's first, or the zero one)
            bool done = (l & 31u) <= 1u;
            cur = (int)~(l + 31u);  // first + 1, count - 1
            if (WIDE || (l & 31u) != 0u) {
                if (COUNT) c_tri++;
                const float Oz = fmaf(-oz, r0.z, fmaf(-oy, r0.y, fmaf(-ox, r0.x, r0.w)));
                const float invDz = rcp_rn(fmaf(dz, r0.z, fmaf(dy, r0.y, dx * r0.x)));
                const float t = Oz * invDz;
                const float Ox = fmaf(oz, r1.z, fmaf(oy, r1.y, fmaf(ox, r1.x, r1.w)));
                const float Dx = fmaf(dz, r1.z, fmaf(dy, r1.y, dx * r1.x));
                const float u = fmaf(t, Dx, Ox);
                const float Oy = fmaf(oz, r2.z, fmaf(oy, r2.y, fmaf(ox, r2.x, r2.w)));
                const float Dy = fmaf(dz, r2.z, fmaf(dy, r2.y, dx * r2.x));
                const float v = fmaf(t, Dy, Oy);
                // ties at equal t go to the lowest id
                const bool nearer = t < hitT || (t == hitT && id < hitId);
                const float uv = u + v;
                if (t > tmin && nearer && u >= 0.0f && v >= 0.0f && uv <= 1.0f &&
                    (!WIDE || !strict || leaf_box_passes(boxes(), l >> 5, tmin, idx_, idy_, idz_, oodx, oody, oodz))) {
                    hitT = t;
                    hitId = id;
                    if (WIDE) hitRef = (int)(l >> 5);
                    if (any()) {
                        cur = kSentinel;
                        done = false;
                    }
                }
            }
            pop |= done;
        }
        if (pop) {
            cur = pop_entry();
            if (COUNT && cur < 0) c_leaf++;
        }
    }
    if (!COUNT && left) {
        // ---- the wave's last rays: a quad each ----
        const int q = (int)(lane >> 2), j = (int)(lane & 3);
        const bool has = (uint32_t)q < left;
        const V4f* const was = stage + 16 * (has ? q : 0);
        const V4f o = was[0], d = was[1];
        const V4i w = __builtin_bit_cast(V4i, was[2]), x = __builtin_bit_cast(V4i, was[3]);
        cur = has ? w.y : kSentinel;
        sp = w.z;
        mine = (uint32_t)w.w;
        batch = (uint32_t)x.x;
        QuadHit h = {d.w, w.x, x.z, x.w != 0};
        if (MULTI) {
            nodes = (GF4)tab[batch].nodes;
            tris = (GF4)tab[batch].tris;
        }
        const RayRegs r = ray_regs(o, d);
        const bool an = any();
        int* const column = lstack + (tid & ~63) + x.y;
        int* const deep = (int*)(stage + 16 * q) + 16;
        int* const spare = (int*)(stage + 16 * q) + j;
        auto at_entry = [&](int e) -> int* { return e < R ? column + e * BLOCK : deep + (e - R); };
        bool full = false;
        while (true) {
            while (__ballot(cur != kSentinel) != 0)
                quad_step<WIDE>(nodes, tris, r, an, j, at_entry, R + kDeep, spare, boxes(), cur, sp, h, full);
            const bool again = WIDE && has && walk_again(boxes(), r, h);
            if (__ballot(again) == 0) break;
            if (again) {
                h = {__builtin_canonicalizef(
                         ((const __attribute__((address_space(1))) float*)(rays() + 2 * (size_t)rayidx() + 1))[3]),
                     -1, 0, true};
                sp = 0;
                cur = 0;
            }
        }
        if (full) atomicOr(a.errors, (uint32_t)RB_TRACE_ERR_STACK);
        hitT = h.t;
        hitId = h.id;
        if (has && j == 0) store();
    }
    end_launch<false>(a);
}

// The reference's speculative order over the binary records (rb_trace_config
// .speculative): a lane that holds a leaf keeps walking inner nodes until the
// whole wave holds leaves.
template <bool ANY_T, bool COUNT, int S, int BLOCK, bool MULTI>
__device__ __forceinline__ void trace_spec(const TraceArgs& a, const BatchDesc* tab, uint32_t nb, uint32_t nrays) {
    __shared__ int lstack[S * BLOCK];
    int spill[kMaxStack - S];
    const int tid = threadIdx.x;
    const uint32_t lane = __lane_id();
    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));

    lstack[tid] = kSentinel;
    // top of the tree (the layout's first records, breadth-first) in LDS
    extern __shared__ V4f lnodes[];
    const uint32_t top = MULTI ? 0u : a.top_nodes;
    if (top) {
        const GF4 src = (GF4)a.nodes;
        for (uint32_t i = tid; i < 4 * top; i += BLOCK) lnodes[i] = src[i];
        __syncthreads();
    }
    uint32_t pool_next = 0, pool_end = 0;
    const uint32_t band_len = MULTI ? 0u : ((nrays + kRayBands - 1) / kRayBands + a.chunk - 1) / a.chunk * a.chunk;
    uint32_t band = 0;
    if (!MULTI) {
        asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(band));
        band &= kRayBands - 1;
    }
    int nodeAddr = kSentinel, leafAddr = 0, sp = 0, hitIndex = -1;
    uint32_t rayidx = 0;
    float ox = 0.f, oy = 0.f, oz = 0.f, tmin = 0.f, dx = 0.f, dy = 0.f, dz = 0.f, hitT = 0.f, tmax_in = 0.f;
    float idx_ = 0.f, idy_ = 0.f, idz_ = 0.f, oodx = 0.f, oody = 0.f, oodz = 0.f;
    uint32_t c_inner = 0, c_tri = 0, c_leaf = 0;
    // scene of the lane's current ray (uniform in single-batch mode)
    GF4 nodes = (GF4)a.nodes;
    GF4 tris = (GF4)a.tris;
    GU32 index = (GU32)a.index;
    GI2 hits = (GI2)a.hits;
    bool any = ANY_T;

    while (true) {
        // ---- fetch rays for terminated lanes (wave-uniform control) ----
        const bool term = nodeAddr == kSentinel;
        const uint64_t m = __ballot(term);
        if (m) {
            const uint32_t nterm = __popcll(m);
            const uint32_t rank = __popcll(m & lt_mask);
            const uint32_t avail = pool_end - pool_next;
            uint32_t mine;
            if (avail >= nterm) {
                mine = pool_next + rank;
                pool_next += nterm;
            } else {
                const int leader = __builtin_ctzll(m);
                uint32_t base = 0;
                if (MULTI) {
                    if ((int)lane == leader) base = atomicAdd(a.counter, a.chunk);
                } else {
                    if ((int)lane == leader) {
                        base = nrays;  // every band claimed: the lanes finish
                        for (uint32_t t = 0; t < kRayBands; t++) {
                            const uint32_t o = atomicAdd(a.counter + kBandStride * (band + 1), a.chunk);
                            if (o < band_len && band * band_len + o < nrays) {  // the last band ends at nrays
                                base = band * band_len + o;
                                break;
                            }
                            band = (band + 1) & (kRayBands - 1);
                        }
                    }
                    band = __shfl(band, leader);
                }
                base = __shfl(base, leader);
                mine = rank < avail ? pool_next + rank : base + (rank - avail);
                pool_next = base + (nterm - avail);
                pool_end = base + a.chunk;
            }
            if (term) {
                if (mine >= nrays) break;
                GF4 rays = (GF4)a.rays;
                rayidx = mine;
                const uint8_t* mk = a.mask;
                if (MULTI) {
                    // the last batch starting at or before `mine` (empty
                    // batches share their successor's start)
                    uint32_t lo = 0, hi = nb;
                    while (hi - lo > 1) {
                        const uint32_t mid = (lo + hi) >> 1;
                        if (tab[mid].start <= mine) lo = mid;
                        else hi = mid;
                    }
                    const BatchDesc& B = tab[lo];
                    nodes = (GF4)B.nodes;
                    tris = (GF4)B.tris;
                    index = (GU32)B.index;
                    hits = (GI2)B.hits;
                    rays = (GF4)B.rays;
                    any = B.any != 0;
                    rayidx = mine - B.start;
                    mk = B.mask;
                }
                const V4f o = rays[2 * (size_t)rayidx];
                const V4f d = rays[2 * (size_t)rayidx + 1];
                ox = o.x; oy = o.y; oz = o.z;
                dx = d.x; dy = d.y; dz = d.z;
                // quiet copies for the slab min / max (comparisons treat every
                // NaN alike); a miss reports the caller's tmax bits unchanged
                tmin = __builtin_canonicalizef(o.w);
                hitT = __builtin_canonicalizef(d.w);
                tmax_in = d.w;
                const float ooeps = 0x1p-80f;
                idx_ = rcp_rn(fabsf(dx) > ooeps ? dx : copysignf(ooeps, dx));
                idy_ = rcp_rn(fabsf(dy) > ooeps ? dy : copysignf(ooeps, dy));
                idz_ = rcp_rn(fabsf(dz) > ooeps ? dz : copysignf(ooeps, dz));
                oodx = ox * idx_;
                oody = oy * idy_;
                oodz = oz * idz_;
                sp = 0;
                leafAddr = 0;
                hitIndex = -1;
                nodeAddr = (mk && mk[rayidx] == 0) ? kSentinel : 0;
                if (COUNT) { c_inner = 0; c_tri = 0; c_leaf = 0; }
            }
        }

        // ---- traversal ----
        while (nodeAddr != kSentinel) {
            while ((uint32_t)nodeAddr < (uint32_t)kSentinel) {
                V4f n0, n1, nz;
                V4i lk;
                if ((uint32_t)nodeAddr < top) {
                    const V4f* ln = lnodes + 4 * nodeAddr;
                    n0 = ln[0];
                    n1 = ln[1];
                    nz = ln[2];
                    lk = __builtin_bit_cast(V4i, ln[3]);
                } else {
                    const GF4 np = nodes + 4 * (size_t)nodeAddr;
                    n0 = np[0];
                    n1 = np[1];
                    nz = np[2];
                    lk = *(GI4)(np + 3);
                    // All four loads of the record in flight at once: without
                    // this the compiler sinks the link load below the slab tests
                    // (it is only read when a child is hit), a second memory
                    // round trip per visited node.  The empty asm consumes every
                    // loaded value.
                    asm volatile("" ::"v"(n0.x), "v"(n0.y), "v"(n0.z), "v"(n0.w), "v"(n1.x), "v"(n1.y), "v"(n1.z),
                                 "v"(n1.w), "v"(nz.x), "v"(nz.y), "v"(nz.z), "v"(nz.w), "v"(lk.x), "v"(lk.y));
                }
                if (COUNT) c_inner++;
                const float c0lox = fmaf(n0.x, idx_, -oodx), c0hix = fmaf(n0.y, idx_, -oodx);
                const float c0loy = fmaf(n0.z, idy_, -oody), c0hiy = fmaf(n0.w, idy_, -oody);
                const float c0loz = fmaf(nz.x, idz_, -oodz), c0hiz = fmaf(nz.y, idz_, -oodz);
                const float c1loz = fmaf(nz.z, idz_, -oodz), c1hiz = fmaf(nz.w, idz_, -oodz);
                const float c1lox = fmaf(n1.x, idx_, -oodx), c1hix = fmaf(n1.y, idx_, -oodx);
                const float c1loy = fmaf(n1.z, idy_, -oody), c1hiy = fmaf(n1.w, idy_, -oody);
                const float c0min = vmax3_(vmin_(c0lox, c0hix), vmin_(c0loy, c0hiy), vmax_(vmin_(c0loz, c0hiz), tmin));
                const float c0max = vmin3_(vmax_(c0lox, c0hix), vmax_(c0loy, c0hiy), vmin_(vmax_(c0loz, c0hiz), hitT));
                const float c1min = vmax3_(vmin_(c1lox, c1hix), vmin_(c1loy, c1hiy), vmax_(vmin_(c1loz, c1hiz), tmin));
                const float c1max = vmin3_(vmax_(c1lox, c1hix), vmax_(c1loy, c1hiy), vmin_(vmax_(c1loz, c1hiz), hitT));
                const bool swp = c1min < c0min;
                const bool t0 = c0max >= c0min;
                const bool t1 = c1max >= c1min;
                int far = lk.y;
                if (!t0 && !t1) {
                    RB_POP(nodeAddr);
                } else {
                    nodeAddr = t0 ? lk.x : lk.y;
                    if (t0 && t1) {
                        if (swp) {
                            const int tmp = nodeAddr;
                            nodeAddr = far;
                            far = tmp;
                        }
                        RB_PUSH(far);
                    }
                }
                if (nodeAddr < 0 && leafAddr >= 0) {
                    leafAddr = nodeAddr;
                    RB_POP(nodeAddr);
                }
                if (!__any(leafAddr >= 0)) break;
            }

            while (leafAddr < 0) {
                const uint32_t l = ~(uint32_t)leafAddr;
                const uint32_t first = l >> 5;
                const uint32_t cnt = l & 31u;
                if (COUNT) c_leaf++;
                for (uint32_t k = 0; k < cnt; k++) {
                    const GF4 w = tris + 3 * (size_t)(first + k);
                    const V4f v0 = w[0];
                    const V4f v1 = w[1];
                    const V4f v2 = w[2];
                    if (COUNT) c_tri++;
                    const float Oz = fmaf(-oz, v0.z, fmaf(-oy, v0.y, fmaf(-ox, v0.x, v0.w)));
                    const float invDz = rcp_rn(fmaf(dz, v0.z, fmaf(dy, v0.y, dx * v0.x)));
                    const float t = Oz * invDz;
                    if (t > tmin && (t < hitT || (hitIndex != -1 && t == hitT))) {
                        const float Ox = fmaf(oz, v1.z, fmaf(oy, v1.y, fmaf(ox, v1.x, v1.w)));
                        const float Dx = fmaf(dz, v1.z, fmaf(dy, v1.y, dx * v1.x));
                        const float u = fmaf(t, Dx, Ox);
                        if (u >= 0.0f) {
                            const float Oy = fmaf(oz, v2.z, fmaf(oy, v2.y, fmaf(ox, v2.x, v2.w)));
                            const float Dy = fmaf(dz, v2.z, fmaf(dy, v2.y, dx * v2.x));
                            const float v = fmaf(t, Dy, Oy);
                            if (v >= 0.0f && u + v <= 1.0f) {
                                bool take = t < hitT;
                                if (!take) take = index[first + k] < index[hitIndex];
                                if (take) {
                                    hitT = t;
                                    hitIndex = (int)(first + k);
                                    if (any) {
                                        nodeAddr = kSentinel;
                                        break;
                                    }
                                }
                            }
                        }
                    }
                }
                leafAddr = nodeAddr;
                if (nodeAddr < 0) RB_POP(nodeAddr);
            }

            // Dynamic fetch: refill when too few lanes are still busy.
            if (__popcll(__ballot(1)) < a.threshold) break;
        }

        if (nodeAddr == kSentinel) {
            V2i r;
            r.x = hitIndex < 0 ? -1 : (int)index[hitIndex];
            r.y = __float_as_int(hitIndex < 0 ? tmax_in : hitT);
            hits[rayidx] = r;
            if (COUNT) {
                a.counts[3 * (size_t)rayidx + 0] = c_inner;
                a.counts[3 * (size_t)rayidx + 1] = c_tri;
                a.counts[3 * (size_t)rayidx + 2] = c_leaf;
            }
        }
    }
    end_launch<MULTI>(a);
}

#undef RB_PUSH
#undef RB_POP

template <bool ANY, bool COUNT, int S, int BLOCK, bool SPEC>
__global__ __launch_bounds__(BLOCK) void k_trace(TraceArgs a) {
    const uint32_t nrays = a.n_dev ? __builtin_nontemporal_load(a.n_dev) : a.n;
    if (SPEC)
        trace_spec<ANY, COUNT, S, BLOCK, false>(a, nullptr, 0, nrays);
    else
        trace_steps<ANY, COUNT, S, BLOCK, false, false, false>(a, nullptr, 0, nrays);
}

// Closest hit, or occlusion (ANY), over the wide records (COUNT: inner =
// wide records visited).
template <bool ANY, bool COUNT, int S, int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_trace_wide(TraceArgs a) {
    const uint32_t nrays = a.n_dev ? __builtin_nontemporal_load(a.n_dev) : a.n;
    trace_steps<ANY, COUNT, S, BLOCK, false, false, true>(a, nullptr, 0, nrays);
}

template <int S, int BLOCK, bool WIDE>
__global__ __launch_bounds__(BLOCK) void k_trace_pair(TraceArgs a) {
    const uint32_t n0 = __builtin_nontemporal_load(a.n_dev);
    const uint32_t n1 = __builtin_nontemporal_load(a.n_dev2);
    trace_steps<true, false, S, BLOCK, false, true, WIDE>(a, nullptr, 0, n0 + n1, n0);
}

// The launch's batch table in LDS, with each batch's first global ray.
__device__ __forceinline__ void batch_table(const BatchTable& t, BatchDesc* tab, uint32_t* total) {
    for (uint32_t i = threadIdx.x; i < t.nb; i += blockDim.x) tab[i] = t.d[i];
    __syncthreads();
    if (threadIdx.x == 0) {  // batch starts from the counts (device counts were final before the launch)
        uint32_t sum = 0;
        for (uint32_t i = 0; i < t.nb; i++) {
            uint32_t n = tab[i].n;
            if (tab[i].n_dev) {
                const uint32_t c = __builtin_nontemporal_load(tab[i].n_dev);
                n = c < n ? c : n;
            }
            tab[i].start = sum;
            sum += n;
        }
        *total = sum;
    }
    __syncthreads();
}

template <int S, int BLOCK, bool SPEC, bool WIDE>
__global__ __launch_bounds__(BLOCK) void k_trace_batch(TraceArgs a, BatchTable t) {
    __shared__ BatchDesc tab[kMaxBatch];
    __shared__ uint32_t s_total;
    batch_table(t, tab, &s_total);
    if (SPEC)
        trace_spec<false, false, S, BLOCK, true>(a, tab, t.nb, s_total);
    else
        trace_steps<false, false, S, BLOCK, true, false, WIDE>(a, tab, t.nb, s_total);
}

template <bool ANY, bool WIDE>
__global__ __launch_bounds__(64) void k_trace_few(TraceArgs a) {
    const uint32_t nrays = a.n_dev ? __builtin_nontemporal_load(a.n_dev) : a.n;
    extern __shared__ int lstack[];
    if (blockIdx.x * 16 < nrays) trace_quads<ANY, false, false, WIDE>(a, nullptr, 0, nrays, 0, lstack, blockIdx.x);
}

template <bool WIDE>
__global__ __launch_bounds__(64) void k_trace_few_pair(TraceArgs a) {
    const uint32_t n0 = __builtin_nontemporal_load(a.n_dev);
    const uint32_t n1 = __builtin_nontemporal_load(a.n_dev2);
    extern __shared__ int lstack[];
    if (blockIdx.x * 16 < n0 + n1)
        trace_quads<true, false, true, WIDE>(a, nullptr, 0, n0 + n1, n0, lstack, blockIdx.x);
}

template <bool WIDE>
__global__ __launch_bounds__(64) void k_trace_few_batch(TraceArgs a, BatchTable t) {
    __shared__ BatchDesc tab[kMaxBatch];
    __shared__ uint32_t s_total;
    batch_table(t, tab, &s_total);
    extern __shared__ int lstack[];
    if (blockIdx.x * 16 < s_total)
        trace_quads<false, true, false, WIDE>(a, tab, t.nb, s_total, 0, lstack, blockIdx.x);
}

// ---------------------------------------------------------------- launch --

typedef void (*TraceKernel)(TraceArgs);
typedef void (*BatchKernel)(TraceArgs, BatchTable);

#define RB_FOR_CONFIGS(X)                                                        \
    X(8, 64) X(8, 128) X(8, 256) X(8, 512) X(8, 1024) X(12, 64) X(12, 128)       \
    X(12, 256) X(12, 512) X(12, 1024) X(16, 64) X(16, 128) X(16, 256) X(16, 512) \
    X(20, 64) X(20, 128) X(20, 256) X(24, 64) X(24, 128) X(24, 256)

template <bool ANY, bool COUNT>
static TraceKernel pick(const rb_trace_config& c) {
#define RB_K(s, b)                             \
    if (c.lds_stack == s && c.block == b)      \
        return c.speculative ? k_trace<ANY, COUNT, s, b, true> : k_trace<ANY, COUNT, s, b, false>;
    RB_FOR_CONFIGS(RB_K)
#undef RB_K
    return nullptr;
}

template <bool ANY, bool COUNT>
static TraceKernel pick_wide(const rb_trace_config& c) {
#define RB_K(s, b) \
    if (c.lds_stack == s && c.block == b) return k_trace_wide<ANY, COUNT, s, b>;
    RB_FOR_CONFIGS(RB_K)
#undef RB_K
    return nullptr;
}

template <bool WIDE>
static TraceKernel pick_pair(const rb_trace_config& c) {
#define RB_K(s, b) \
    if (c.lds_stack == s && c.block == b) return k_trace_pair<s, b, WIDE>;
    RB_FOR_CONFIGS(RB_K)
#undef RB_K
    return nullptr;
}

static BatchKernel pick_batch(const rb_trace_config& c, bool wide) {
#define RB_K(s, b)                                                                    \
    if (c.lds_stack == s && c.block == b)                                             \
        return c.speculative ? k_trace_batch<s, b, true, false>                       \
                             : wide ? k_trace_batch<s, b, false, true> : k_trace_batch<s, b, false, false>;
    RB_FOR_CONFIGS(RB_K)
#undef RB_K
    return nullptr;
}

// Whether a set may walk the wide records: closest hit, or an any-hit set
// read only as hit / miss (kOcclusion), under a non-speculative config with
// the wide walk on, over a BVH that has wide records.
static bool wide_walk(const rb_trace_config& cfg, rb_bvh_t bvh, uint32_t flags) {
    return cfg.wide && !cfg.speculative && bvh->wnodes && (!(flags & RB_ANY) || (flags & kOcclusion));
}

// Launches of up to this many rays per CU take trace_quads: where both loops are
// level on rays that scatter (the figures are at trace_quads), over the wide and
// the binary records alike.  Three times as many camera rays, whose quads share
// their lines and branches (384 Ki: 148 us in trace_steps, 115 in trace_quads;
// 512 Ki: 171 and 161).
constexpr uint32_t kFewPerCu = 512, kFewCoherentPerCu = 1536;
static bool few_rays(const rb_trace_config& cfg, uint64_t n, bool coherent = false) {
    return !cfg.speculative && n <= (uint64_t)dev().num_cus * (coherent ? kFewCoherentPerCu : kFewPerCu);
}
// The same for a launch with a larger bound whose ray counts only the kernel
// knows, where a wave's LDS holds the quads' stacks.  (The later bounces of a
// path-traced frame, whose bound is two rays per path: 24 served tiles 11.1 ->
// 9.8 ms, a 512x512x4 BDPT frame 6.79 -> 6.74, a 1024x1024x8 path-traced one 17.99
// -> 17.88.)
static uint32_t few_known_late(const rb_trace_config& cfg, uint32_t rows) {
    return rows + 1 <= cfg.lds_stack + 15 ? dev().num_cus * kFewPerCu : 0;
}
static uint32_t few_blocks(uint64_t n) { return (uint32_t)((n + 15) / 16); }

// Static LDS of a trace block: the stack and, in the step loop, a staged
// 64-byte record per lane.
static size_t trace_lds(const rb_trace_config& cfg) {
    return (size_t)cfg.block * (4 * cfg.lds_stack + (cfg.speculative ? 0 : 64));
}

static uint32_t persistent_blocks(const rb_trace_config& cfg, uint64_t n) {
    const uint32_t waves = dev().num_cus * cfg.waves_per_cu;
    uint32_t blocks = waves * 64 / cfg.block;
    const uint64_t need = (n + cfg.block - 1) / cfg.block;
    if (blocks > need) blocks = (uint32_t)need;
    return blocks ? blocks : 1;
}

rb_status launch_trace(rb_bvh_t bvh, const rb_ray* rays, uint32_t n, uint32_t flags, const uint8_t* mask,
                       rb_hit* hits, uint32_t* counts, hipStream_t stream, const rb_trace_config& cfg,
                       const uint32_t* n_dev, uint32_t* counter) {
    if (n == 0) return RB_OK;
    if (!bvh || !rays || !hits) return fail(RB_ERR_INVALID, "NULL bvh, rays or hits");
    if (n > 0x7FFFFFFFu) return fail(RB_ERR_INVALID, "too many rays in one call (%u)", n);
    if ((flags & RB_MASKED) && !mask) return fail(RB_ERR_INVALID, "RB_MASKED without a mask");
    const bool any = (flags & RB_ANY) != 0;
    // Closest hit and occlusion walk the wide records (leaf_boxes: whose hits
    // they are); visit counts follow the binary walk unless RB_WIDE_COUNTS asks for the
    // wide one.
    const bool wide_counts = (flags & RB_WIDE_COUNTS) != 0;
    if (wide_counts && (!counts || any || cfg.speculative))
        return fail(RB_ERR_INVALID, "RB_WIDE_COUNTS: visit counts of a closest-hit, non-speculative trace only");
    if (wide_counts && !bvh->wnodes)
        return fail(RB_ERR_UNSUPPORTED, "RB_WIDE_COUNTS: this BVH has no wide records (the upload kept the binary walk)");
    const bool wide = wide_counts || (!counts && wide_walk(cfg, bvh, flags));
    TraceKernel k = wide ? (counts ? pick_wide<false, true>(cfg) : any ? pick_wide<true, false>(cfg)
                                                                       : pick_wide<false, false>(cfg))
                  : counts ? (any ? pick<true, true>(cfg) : pick<false, true>(cfg))
                           : (any ? pick<true, false>(cfg) : pick<false, false>(cfg));
    if (!k) return fail(RB_ERR_INVALID, "unsupported trace config (lds_stack %u, block %u)", cfg.lds_stack, cfg.block);
    TraceArgs a;
    std::memset(&a, 0, sizeof(a));
    a.nodes = bvh->nodes;
    a.tris = cfg.speculative ? bvh->tris : bvh->tris4;
    a.index = bvh->index;
    a.rays = reinterpret_cast<const float4*>(rays);
    a.mask = (flags & RB_MASKED) ? mask : nullptr;
    a.hits = reinterpret_cast<int2*>(hits);
    a.counts = counts;
    a.errors = dev().errors;
    a.n = n;
    a.n_dev = n_dev;
    a.chunk = cfg.chunk;
    a.threshold = cfg.fetch_threshold;
    a.leaf_gate = cfg.leaf_gate;
    if (wide) a.nodes = bvh->wnodes;
    a.stack_rows = stack_rows(bvh, wide);
    a.boxes = bvh->wnodes + 4 * (size_t)bvh->n_wnodes;
    // top-of-tree records in LDS: the speculative walk only
    a.top_nodes = !cfg.speculative ? 0 : cfg.lds_nodes < bvh->n_nodes ? cfg.lds_nodes : bvh->n_nodes;
    const size_t top_bytes = (size_t)a.top_nodes * 64;
    const size_t lds = trace_lds(cfg) + top_bytes;
    if (lds > dev().lds_per_block)
        return fail(RB_ERR_INVALID, "trace config needs %zu bytes of LDS per block (stack %u x %u lanes + %u node records); "
                    "the device allows %zu", lds, cfg.lds_stack, cfg.block, a.top_nodes, dev().lds_per_block);
    if (!counts && few_rays(cfg, n, (flags & kCoherent) != 0)) {
        TraceKernel q = wide ? (any ? k_trace_few<true, true> : k_trace_few<false, true>)
                             : (any ? k_trace_few<true, false> : k_trace_few<false, false>);
        hipLaunchKernelGGL(q, dim3(few_blocks(n)), dim3(64), quad_lds(a.stack_rows), stream, a);
        const hipError_t e = hipGetLastError();
        return e != hipSuccess ? hip_fail(e, "trace launch") : RB_OK;
    }
    SlotLease L;
    if (counter) {
        L.counter = counter;
    } else {
        L = take_counter_slot(stream);
        if (L.st != RB_OK) return L.st;
        if (!L.counter) return fail(RB_ERR_INVALID, "render graph: out of work-counter slots");
    }
    a.counter = L.counter;
    hipLaunchKernelGGL(k, dim3(persistent_blocks(cfg, n)), dim3(cfg.block), top_bytes, stream, a);
    const hipError_t e = hipGetLastError();
    release_counter_slot(L, stream);
    if (e != hipSuccess) return hip_fail(e, "trace launch");
    return RB_OK;
}

rb_status launch_trace_pair(rb_bvh_t bvh, const rb_ray* rays0, uint32_t cap0, const uint32_t* n0_dev, rb_hit* hits0,
                            uint32_t flags0, const rb_ray* rays1, uint32_t cap1, const uint32_t* n1_dev, rb_hit* hits1,
                            hipStream_t stream, const rb_trace_config& cfg) {
    if (!bvh) return fail(RB_ERR_INVALID, "paired trace: NULL bvh");
    // both sets walk the wide records when set 0 may (set 1 is closest hit)
    const bool wide = wide_walk(cfg, bvh, flags0);
    TraceKernel k = cfg.speculative ? nullptr : wide ? pick_pair<true>(cfg) : pick_pair<false>(cfg);
    // the speculative order, or more rays than one counter range takes: two launches
    if (!k || (uint64_t)cap0 + cap1 > 0x7FFFFFFFull) {
        rb_status st = launch_trace(bvh, rays0, cap0, flags0 & (RB_ANY | kOcclusion), nullptr, hits0, nullptr, stream,
                                    cfg, n0_dev);
        if (st != RB_OK) return st;
        return launch_trace(bvh, rays1, cap1, RB_CLOSEST, nullptr, hits1, nullptr, stream, cfg, n1_dev);
    }
    if (cap0 + cap1 == 0) return RB_OK;
    if (!rays0 || !rays1 || !hits0 || !hits1 || !n0_dev || !n1_dev)
        return fail(RB_ERR_INVALID, "paired trace: NULL argument");
    TraceArgs a;
    std::memset(&a, 0, sizeof(a));
    a.nodes = wide ? bvh->wnodes : bvh->nodes;
    a.stack_rows = stack_rows(bvh, wide);
    a.boxes = bvh->wnodes + 4 * (size_t)bvh->n_wnodes;
    a.tris = bvh->tris4;
    a.index = bvh->index;
    a.rays = reinterpret_cast<const float4*>(rays0);
    a.hits = reinterpret_cast<int2*>(hits0);
    a.n_dev = n0_dev;
    a.rays2 = reinterpret_cast<const float4*>(rays1);
    a.hits2 = reinterpret_cast<int2*>(hits1);
    a.n_dev2 = n1_dev;
    a.any0 = (flags0 & RB_ANY) ? 1u : 0u;
    a.errors = dev().errors;
    a.n = cap0 + cap1;
    a.chunk = cfg.chunk;
    a.threshold = cfg.fetch_threshold;
    a.leaf_gate = cfg.leaf_gate;
    a.few = few_known_late(cfg, a.stack_rows);
    const size_t lds = trace_lds(cfg);
    if (lds > dev().lds_per_block)
        return fail(RB_ERR_INVALID, "trace config needs %zu bytes of LDS per block; the device allows %zu", lds,
                    dev().lds_per_block);
    if (few_rays(cfg, a.n)) {
        TraceKernel q = wide ? k_trace_few_pair<true> : k_trace_few_pair<false>;
        hipLaunchKernelGGL(q, dim3(few_blocks(a.n)), dim3(64), quad_lds(a.stack_rows), stream, a);
        const hipError_t e = hipGetLastError();
        return e != hipSuccess ? hip_fail(e, "paired trace launch") : RB_OK;
    }
    const SlotLease L = take_counter_slot(stream);
    if (L.st != RB_OK) return L.st;
    if (!L.counter) return fail(RB_ERR_INVALID, "render graph: out of work-counter slots");
    a.counter = L.counter;
    hipLaunchKernelGGL(k, dim3(persistent_blocks(cfg, a.n)), dim3(cfg.block), 0, stream, a);
    const hipError_t e = hipGetLastError();
    release_counter_slot(L, stream);
    if (e != hipSuccess) return hip_fail(e, "paired trace launch");
    return RB_OK;
}

static rb_status launch_trace_sets_pass(const BatchSet* b, uint32_t nb, hipStream_t stream, const rb_trace_config& cfg,
                                        bool wide);

// The sets that may walk the wide records go through launches of their own
// (pass 1), the rest through the binary kernel (pass 0).
rb_status launch_trace_sets(const BatchSet* b, uint32_t nb, hipStream_t stream, const rb_trace_config& cfg) {
    for (uint32_t i = 0; i < nb; i++) {
        if (b[i].n == 0) continue;
        if (!b[i].bvh || !b[i].rays || !b[i].hits) return fail(RB_ERR_INVALID, "batch %u: NULL bvh, rays or hits", i);
        if (b[i].n > 0x7FFFFFFFu) return fail(RB_ERR_INVALID, "batch %u: more than 2^31 - 1 rays", i);
    }
    for (int pass = 0; pass < 2; pass++) {
        const rb_status st = launch_trace_sets_pass(b, nb, stream, cfg, pass == 1);
        if (st != RB_OK) return st;
    }
    return RB_OK;
}

static rb_status launch_trace_sets_pass(const BatchSet* b, uint32_t nb, hipStream_t stream, const rb_trace_config& cfg,
                                        bool wide) {
    BatchKernel k = pick_batch(cfg, wide);
    if (!k) return fail(RB_ERR_INVALID, "unsupported trace config (lds_stack %u, block %u)", cfg.lds_stack, cfg.block);
    auto in_pass = [&](const BatchSet& x) {
        return wide_walk(cfg, x.bvh, (x.any ? RB_ANY : 0u) | (x.occlusion ? kOcclusion : 0u)) == wide;
    };
    for (uint32_t i0 = 0; i0 < nb;) {
        BatchTable t;
        std::memset(&t, 0, sizeof(t));
        uint64_t total = 0;  // bound of the launch's rays (sizes the grid)
        uint32_t rows = 0;
        uint32_t i = i0;
        for (; i < nb && t.nb < kMaxBatch; i++) {
            if (b[i].n == 0 || !in_pass(b[i])) continue;
            if (total + b[i].n > 0x7FFFFFFFull) break;  // the next launch takes it
            BatchDesc& d = t.d[t.nb++];
            d.nodes = wide ? b[i].bvh->wnodes : b[i].bvh->nodes;
            d.tris = cfg.speculative ? b[i].bvh->tris : b[i].bvh->tris4;
            d.index = b[i].bvh->index;
            d.rays = b[i].rays;
            d.hits = b[i].hits;
            d.mask = b[i].mask;
            d.n_dev = b[i].n_dev;
            d.n = b[i].n;
            d.any = b[i].any ? 1u : 0u;
            d.boxes = b[i].bvh->wnodes + 4 * (size_t)b[i].bvh->n_wnodes;
            rows = std::max(rows, stack_rows(b[i].bvh, wide));
            total += b[i].n;
        }
        i0 = i;
        if (t.nb == 0) continue;
        TraceArgs a;
        std::memset(&a, 0, sizeof(a));
        a.errors = dev().errors;
        a.n = (uint32_t)total;
        a.stack_rows = rows;
        a.chunk = cfg.chunk;
        a.threshold = cfg.fetch_threshold;
        a.leaf_gate = cfg.leaf_gate;
        a.few = few_known_late(cfg, a.stack_rows);
        if (few_rays(cfg, total)) {
            BatchKernel q = wide ? k_trace_few_batch<true> : k_trace_few_batch<false>;
            hipLaunchKernelGGL(q, dim3(few_blocks(total)), dim3(64), quad_lds(a.stack_rows), stream, a, t);
            const hipError_t e = hipGetLastError();
            if (e != hipSuccess) return hip_fail(e, "batched trace launch");
            continue;
        }
        const SlotLease L = take_counter_slot(stream);
        if (L.st != RB_OK) return L.st;
        if (!L.counter) return fail(RB_ERR_INVALID, "render graph: out of work-counter slots");
        a.counter = L.counter;
        hipLaunchKernelGGL(k, dim3(persistent_blocks(cfg, total)), dim3(cfg.block), 0, stream, a, t);
        const hipError_t e = hipGetLastError();
        release_counter_slot(L, stream);
        if (e != hipSuccess) return hip_fail(e, "batched trace launch");
    }
    return RB_OK;
}

rb_status launch_trace_batch(const rb_batch_desc* b, uint32_t nb, hipStream_t stream, const rb_trace_config& cfg) {
    uint64_t total = 0;
    std::vector<BatchSet> sets;
    try {
        sets.reserve(nb);
    } catch (...) {
        return fail(RB_ERR_OOM, "batch table (host allocation)");
    }
    for (uint32_t i = 0; i < nb; i++) {
        if (b[i].n == 0) continue;
        if (!b[i].bvh || !b[i].rays || !b[i].hits) return fail(RB_ERR_INVALID, "batch %u: NULL bvh, rays or hits", i);
        if (b[i].flags & RB_MASKED) return fail(RB_ERR_INVALID, "batch %u: masks are not supported in batches", i);
        if (b[i].flags & ~(uint32_t)RB_ANY) return fail(RB_ERR_INVALID, "batch %u: unknown trace flags 0x%x", i, b[i].flags);
        // the rays of one table of kMaxBatch batches go through one launch
        total = (sets.size() % kMaxBatch == 0 ? 0 : total) + b[i].n;
        if (total > 0x7FFFFFFFull) return fail(RB_ERR_INVALID, "more than 2^31 rays in one batched call");
        sets.push_back(BatchSet{b[i].bvh, reinterpret_cast<const float4*>(b[i].rays), reinterpret_cast<int2*>(b[i].hits),
                                b[i].n, nullptr, (b[i].flags & RB_ANY) != 0, nullptr});
    }
    return launch_trace_sets(sets.data(), (uint32_t)sets.size(), stream, cfg);
}

static rb_status check_cfg(const rb_trace_config& c) {
    if (c.block != 64 && c.block != 128 && c.block != 256 && c.block != 512 && c.block != 1024)
        return fail(RB_ERR_INVALID, "block must be 64/128/256/512/1024");
    if (!pick<false, false>(c))
        return fail(RB_ERR_INVALID, "no kernel for lds_stack %u at block %u (512: stack 8-16; 1024: stack 8-12)",
                    c.lds_stack, c.block);
    if (c.lds_stack < 8 || c.lds_stack > 24 || c.lds_stack % 4) return fail(RB_ERR_INVALID, "lds_stack must be 8..24, step 4");
    if (c.chunk < 64 || c.chunk % 64 || c.chunk > 65536) return fail(RB_ERR_INVALID, "chunk must be a multiple of 64 up to 65536");
    if (c.fetch_threshold > 64) return fail(RB_ERR_INVALID, "fetch_threshold must be <= 64");
    if (c.waves_per_cu < 1 || c.waves_per_cu > 64) return fail(RB_ERR_INVALID, "waves_per_cu must be 1..64");
    if (c.speculative > 1) return fail(RB_ERR_INVALID, "speculative must be 0 or 1");
    if (c.leaf_gate > 63) return fail(RB_ERR_INVALID, "leaf_gate must be 0..63");
    if (c.lds_nodes > 512 || c.lds_nodes % 64) return fail(RB_ERR_INVALID, "lds_nodes must be 0..512, step 64");
    if (c.wide > 1) return fail(RB_ERR_INVALID, "wide must be 0 or 1");
    return RB_OK;
}

}  // namespace rb

using namespace rb;

extern "C" {

rb_status rb_trace_get_config(rb_trace_config* c) {
    if (!c) return fail(RB_ERR_INVALID, "NULL config");
    rb_status st = ensure_device();
    if (st != RB_OK) return st;
    *c = dev().cfg;
    return RB_OK;
}

rb_status rb_trace_set_config(const rb_trace_config* c) {
    if (!c) return fail(RB_ERR_INVALID, "NULL config");
    rb_status st = ensure_device();
    if (st != RB_OK) return st;
    if ((st = check_cfg(*c)) != RB_OK) return st;
    dev().cfg = *c;
    return RB_OK;
}

rb_status rb_trace(rb_bvh_t bvh, const rb_ray* rays, uint32_t n, uint32_t flags, const uint8_t* mask, rb_hit* hits,
                   void* stream) {
    rb_status st = ensure_device();
    if (st != RB_OK) return st;
    if (flags & ~(uint32_t)(RB_ANY | RB_MASKED)) return fail(RB_ERR_INVALID, "unknown trace flags 0x%x", flags);
    return launch_trace(bvh, rays, n, flags, mask, hits, nullptr, stream ? (hipStream_t)stream : dev().stream,
                        dev().cfg);
}

rb_status rb_trace_batch(const rb_batch_desc* batches, uint32_t nb, void* stream) {
    rb_status st = ensure_device();
    if (st != RB_OK) return st;
    if (nb && !batches) return fail(RB_ERR_INVALID, "NULL batch table");
    return launch_trace_batch(batches, nb, stream ? (hipStream_t)stream : dev().stream, dev().cfg);
}

rb_status rb_trace_autotune(rb_bvh_t bvh, const rb_ray* rays, uint32_t n, uint32_t flags, rb_hit* hits,
                            uint32_t reps, rb_trace_config* best, float* best_ms, void* stream) {
    rb_status st = ensure_device();
    if (st != RB_OK) return st;
    if (!bvh || !rays || !hits || n == 0) return fail(RB_ERR_INVALID, "autotune needs a bvh and a non-empty ray batch");
    if (flags & RB_MASKED) return fail(RB_ERR_INVALID, "autotune takes unmasked batches");
    if (flags & ~(uint32_t)RB_ANY) return fail(RB_ERR_INVALID, "unknown trace flags 0x%x", flags);
    if (reps == 0) reps = 3;
    hipStream_t s = stream ? (hipStream_t)stream : dev().stream;
    hipEvent_t e0, e1;
    if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess)
        return fail(RB_ERR_DEVICE, "hipEventCreate failed");
    auto measure = [&](const rb_trace_config& c, float* ms) -> rb_status {
        rb_status r = launch_trace(bvh, rays, n, flags, nullptr, hits, nullptr, s, c);  // warm-up
        if (r != RB_OK) return r;
        hipError_t e = hipEventRecord(e0, s);
        if (e != hipSuccess) return hip_fail(e, "autotune event");
        for (uint32_t i = 0; i < reps; i++)
            if ((r = launch_trace(bvh, rays, n, flags, nullptr, hits, nullptr, s, c)) != RB_OK) return r;
        if ((e = hipEventRecord(e1, s)) != hipSuccess) return hip_fail(e, "autotune event");
        e = hipEventSynchronize(e1);
        if (e != hipSuccess) return hip_fail(e, "autotune sync");
        if ((e = hipEventElapsedTime(ms, e0, e1)) != hipSuccess) return hip_fail(e, "autotune timing");
        *ms /= (float)reps;
        return RB_OK;
    };
    rb_trace_config cur = dev().cfg;
    float cur_ms = 0.f;
    if ((st = measure(cur, &cur_ms)) != RB_OK) goto done;
    {
        const uint32_t blocks[] = {64, 128, 256, 512, 1024};
        const uint32_t stacks[] = {8, 12, 16, 20, 24};
        const uint32_t chunks[] = {64, 128, 256, 1024};
        const uint32_t thresholds[] = {0, 16, 32, 40, 48, 56, 60};
        const uint32_t waves[] = {8, 12, 16, 20, 24, 32};
        const uint32_t gates[] = {16, 24, 32, 40, 48, 56, 63};
        const uint32_t tops[] = {0, 64, 128, 192, 256, 384};
        // launches of few rays do not use the configuration: every candidate
        // would be the same launch, and the one that noise favours would be
        // installed for the large ones
        const int passes = few_rays(cur, n) ? 0 : 2;
        for (int pass = 0; pass < passes; pass++) {
            for (int dim = 0; dim < 7; dim++) {
                const uint32_t* vals;
                int nv;
                switch (dim) {
                    case 0: vals = blocks; nv = 5; break;
                    case 1: vals = stacks; nv = 5; break;
                    case 2: vals = chunks; nv = 4; break;
                    case 3: vals = thresholds; nv = 7; break;
                    case 4: vals = waves; nv = 6; break;
                    case 5: vals = gates; nv = 7; break;
                    default: vals = tops; nv = 6; break;
                }
                if (dim == 5 && cur.speculative) continue;   // the gate acts on the step loop,
                if (dim == 6 && !cur.speculative) continue;  // the records in LDS on the speculative walk
                for (int k = 0; k < nv; k++) {
                    rb_trace_config c = cur;
                    uint32_t* f = dim == 0 ? &c.block : dim == 1 ? &c.lds_stack : dim == 2 ? &c.chunk
                                : dim == 3 ? &c.fetch_threshold : dim == 4 ? &c.waves_per_cu
                                : dim == 5 ? &c.leaf_gate : &c.lds_nodes;
                    if (*f == vals[k]) continue;
                    *f = vals[k];
                    if (!pick<false, false>(c) ||
                        trace_lds(c) + (c.speculative ? (size_t)c.lds_nodes * 64 : 0) > dev().lds_per_block)
                        continue;  // no kernel for this shape, or more LDS than a block gets
                    float ms = 0.f;
                    if ((st = measure(c, &ms)) != RB_OK) goto done;
                    if (ms < cur_ms * 0.99f) {
                        cur = c;
                        cur_ms = ms;
                    }
                }
            }
        }
    }
    dev().cfg = cur;
    if (best) *best = cur;
    if (best_ms) *best_ms = cur_ms;
done:
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    return st;
}

rb_status rb_selftest_rcp(unsigned long long* fast_inputs, unsigned long long* mismatches) {
    rb_status st = ensure_device();
    if (st != RB_OK) return st;
    if (!fast_inputs || !mismatches) return fail(RB_ERR_INVALID, "NULL argument");
    unsigned long long* d = nullptr;
    if ((st = dalloc((void**)&d, 2 * sizeof(unsigned long long))) != RB_OK) return st;
    unsigned long long h[2] = {0, 0};
    const hipStream_t s = dev().stream;
    hipError_t e = hipMemsetAsync(d, 0, sizeof(h), s);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_rcp_check, dim3(4096), dim3(256), 0, s, d);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpyAsync(h, d, sizeof(h), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    dfree(d, 2 * sizeof(unsigned long long));
    if (e != hipSuccess) return hip_fail(e, "reciprocal self-test");
    *fast_inputs = h[0];
    *mismatches = h[1];
    return RB_OK;
}

rb_status rb_trace_errors(uint32_t* flags) {
    rb_status st = ensure_device();
    if (st != RB_OK) return st;
    if (!flags) return fail(RB_ERR_INVALID, "NULL flags");
    uint32_t h = 0;
    hipError_t e = hipDeviceSynchronize();
    if (e == hipSuccess) e = hipMemcpy(&h, dev().errors, 4, hipMemcpyDeviceToHost);
    if (e == hipSuccess && h) e = hipMemset(dev().errors, 0, 4);
    if (e != hipSuccess) return hip_fail(e, "trace error flags");
    *flags = h;
    if (h & RB_TRACE_ERR_STACK)
        return fail(RB_ERR_INVALID, "a traversal stack overflowed: hits of the launches since the last check may be wrong");
    if (h) return fail(RB_ERR_INVALID, "trace error flags 0x%x", h);
    return RB_OK;
}

rb_status rb_trace_counts(rb_bvh_t bvh, const rb_ray* rays, uint32_t n, uint32_t flags, rb_hit* hits,
                          uint32_t* counts, void* stream) {
    rb_status st = ensure_device();
    if (st != RB_OK) return st;
    if (!counts) return fail(RB_ERR_INVALID, "NULL counts");
    if (flags & ~(uint32_t)(RB_ANY | RB_MASKED | RB_WIDE_COUNTS))
        return fail(RB_ERR_INVALID, "unknown trace flags 0x%x", flags);
    return launch_trace(bvh, rays, n, flags & ~RB_MASKED, nullptr, hits, counts,
                        stream ? (hipStream_t)stream : dev().stream, dev().cfg);
}

}  // extern "C"
