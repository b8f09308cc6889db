// trace_quad.hpp — the tracer of batches too small to fill the chip with one
// lane per ray (included by trace_relaid.hip).
//
// A batch of a few thousand rays leaves most SIMDs with one wave or none, and
// lasts as long as its longest ray's chain of steps: what counts is the time
// of one step, not the work per ray. So a ray gets four lanes here (a quad):
// lanes 0, 1 and 2 hold the ray's x, y and z, and every per-axis operation of
// the step (sample, domain and leaf tests, split planes, midpoints, exit
// quotients) is one instruction for the three axes instead of three. The axes
// meet in the quad through DPP quad permutes (octant bits, the exit's minimum)
// and through s_wqm, which spreads a lane-mask bit over its quad (a test fails
// for the ray when it fails on any axis). A wave holds 16 rays (4 x 4 angular
// tiles), so it also waits less on its deepest descent and longest leaf run
// than one of 64.
//
// A wave is a workgroup and traces one unit, rays of one env: its scene's
// split planes are staged for that scene alone, no work queue is needed (the
// hardware dispatches units to SIMDs as they free up), and nothing is
// refilled. The per-ray results are the fast march's, whose operations these
// are lane by lane; a unit that the fast march does not cover (boxes beyond
// 2^100, records below 30 levels, negative leaves, planes off the uniform grid,
// a range of 1000 or more) takes quad_general, the general march in quads.
//
// What bounds it: the chain of one step, about 1400 cycles of which half are
// its four to five dependent reads (a cell table one level deeper saves one
// and 60 ns a step) and half its instructions (up to about 100 vector and 90
// scalar ones), which a lone wave issues one every four to five cycles. 43
// VGPRs, eight waves per SIMD. A pass with a lane per ray and with four: 1024 rays
// of a 64^3 room 48 and 32 us; 49 K rays of a 128^3 volume 120 and 68; 49 K rays of
// a 1024^3 volume with their observation 263 and 152. A per-ray cache of
// the last depth-8 cell's slot made no difference: a wave skips the reads only
// when all its rays hit.
#pragma once

namespace navi {

constexpr uint32_t kQuadPlanes = 8;  // split-plane depth: 3 x 258 planes of the unit's scene in LDS
constexpr uint32_t kQuadAxis = 260;  // floats per axis (a multiple of four: planes are written four at a time)

constexpr uint64_t kAxisLanes = 0x7777777777777777ull;  // lanes 0, 1 and 2 of every quad

// The value of the lane's neighbour in its quad: lanes swapped in pairs, and
// the pairs swapped.
__device__ __forceinline__ uint32_t quad_swap1(uint32_t x) {
    return static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(x), 0xb1, 0xf, 0xf, true));
}
__device__ __forceinline__ uint32_t quad_swap2(uint32_t x) {
    return static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(x), 0x4e, 0xf, 0xf, true));
}
__device__ __forceinline__ uint32_t quad_or(uint32_t x) {
    x |= quad_swap1(x);
    return x | quad_swap2(x);
}
__device__ __forceinline__ uint32_t quad_min(uint32_t x) {
    x = min(x, quad_swap1(x));
    return min(x, quad_swap2(x));
}

// The quads (every lane of them) with a set bit in m.
__device__ __forceinline__ uint64_t quad_any(uint64_t m) { return navi_s_wqm(m); }
// The quads with no set bit in m.
__device__ __forceinline__ uint64_t quad_none(uint64_t m) { return ~quad_any(m); }
// The quads whose axis lanes all have their bit set in m.
__device__ __forceinline__ uint64_t quad_all(uint64_t m) { return ~quad_any(~m & kAxisLanes); }

// Work index (of ray_of) of ray i of unit `unit`: units never cross an env,
// and cover a square of angular neighbours where the rays are in tiles.
// 0xffffffff past the env's last ray.
__device__ __forceinline__ uint32_t unit_ray(const RelaidParams& P, uint32_t unit, uint32_t i) {
    const uint32_t env_pos = fdiv(unit, P.div_units);
    const uint32_t w = unit - env_pos * P.env_units;
    uint32_t q;
    if (P.tile_el) {
        const uint32_t lx = (P.quad_shift + 1u) >> 1, ly = P.quad_shift >> 1;  // log2 of the patch's sides
        const uint32_t per = 6u - P.quad_shift;                              // log2 of the units in a tile
        const uint32_t sub = w & ((1u << per) - 1u);
        const uint32_t sx = sub & ((8u >> lx) - 1u), sy = sub >> (3u - lx);
        q = ((w >> per) << 6) | (sy << ly | i >> lx) << 3 | sx << lx | (i & ((1u << lx) - 1u));
    } else {
        q = (w << P.quad_shift) + i;
    }
    return q < P.rays_per_env ? env_pos * P.rays_per_env + q : 0xffffffffu;
}

// The unit of a workgroup. Workgroups go to the eight XCDs in turn; runs of 64
// units (1024 rays of 16 a unit: neighbouring tiles of one env) share an XCD,
// so that its L2 holds what they share of the scene (512^3 room grid, 393 K
// rays: 336 us, against 366 in order and 355 with an eighth of the batch per
// XCD; 16 scenes of 1024^3, 590 K rays: 422, 435 and 515 us).
__device__ __forceinline__ uint32_t unit_of_block(uint32_t block, uint32_t blocks) {
    return block < (blocks & ~511u) ? (block & ~511u) | (block & 7u) << 6 | (block >> 3 & 63u) : block;
}

// The split planes of 2^8 cells along the three axes of one box, nested
// midpoints as the descent computes them (kernel.cu:165-176): lane i splits
// its 64th of each axis off in registers, and its four planes follow.
__device__ __forceinline__ void stage_quad_planes(const float* lo3, const float* hi3, uint32_t lane, float* planes) {
#pragma unroll
    for (uint32_t a = 0; a < 3u; ++a) {
        float lo = lo3[a], hi = hi3[a];
        float* pl = planes + a * kQuadAxis;
        if (lane == 63u) pl[256] = hi, pl[257] = 0.0f;
#pragma unroll
        for (uint32_t b = 32u; b != 0u; b >>= 1) {
            const float m = (lo + hi) * 0.5f;
            const bool up = (lane & b) != 0u;
            lo = up ? m : lo;
            hi = up ? hi : m;
        }
        const float m = (lo + hi) * 0.5f;
        *reinterpret_cast<float4*>(pl + 4u * lane) = make_float4(lo, (lo + m) * 0.5f, m, (m + hi) * 0.5f);
    }
}

struct QuadResult {
    float t;
    int32_t step, sem;
};

// A ray's state as quad_march takes it, an axis a lane: the axis's plane lookup
// (planes, scale, offset), mirrored origin and |direction|, exit reciprocal
// (NaN on axes the exit leaves out), the faces ahead of the domain and of the
// cached leaf (NaN: outside, none cached), the prefix cell's upper face as a
// depth-8 plane index, and, the same in all four lanes, the cell table's first
// entry, the leaf's word, t and the step count. Lane 3's om, adm, scale and off
// are 0 and its dm and lf +inf.
struct QuadRay {
    const float* pl;
    float scale, off, om, adm, r, dm, lf;
    uint32_t pre, table, lf_slot;
    float t;
    int32_t step, sem;
};

// The fast march (march_fast, an axis a lane) of the rays of the quads in live
// (whole quads, as every mask below) to their ends; neg holds the mirrored
// axes. kLeaves: see march_fast.
template <int kDepth, bool kLeaves>
__device__ __forceinline__ void quad_march(const RelaidParams& P, uint64_t neg, uint64_t live, QuadRay& R) {
    constexpr uint32_t D = kDepth;
    constexpr uint32_t kUp = kQuadPlanes - D;  // levels between the table and the planes
    constexpr uint32_t kSh = kQuadPlanes - kPrefixDepth;
    constexpr uint32_t kCells = 1u << kQuadPlanes;
    constexpr float kInf = __builtin_inff();
    const float nan = __builtin_nanf("");
    const uint32_t axis = threadIdx.x & 3u;
    const uint32_t ax = axis == 3u ? 0u : axis;
    // lane 3's sample is -FLT_MAX (q' = 0 with the flip's bits): it lies below
    // every plane and midpoint, so it adds no index or octant bit
    const uint32_t flip = axis == 3u ? 0xff7fffffu : (lane_in(neg) ? 0x80000000u : 0u);
    const uint32_t face_keep = axis == 3u ? 0u : 0xffffffffu, face_flip = axis == 3u ? 0x7f800000u : flip;
    const uint32_t ahead_up = lane_in(neg) ? 0u : 1u;
    const __amdgpu_buffer_rsrc_t records = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint32_t*>(P.records), static_cast<short>(4), static_cast<int>(P.n_records * 8u), 0x00020000);
    const __amdgpu_buffer_rsrc_t tables = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint64_t*>(P.cell_table), static_cast<short>(8),
        static_cast<int>(static_cast<uint32_t>(P.n_scenes) << (3u * D)), 0x00020000);
    const float* const pl = R.pl;
    const float scale = R.scale, off = R.off, om = R.om, adm = R.adm, r = R.r, dm = R.dm;
    const uint32_t my_table = R.table;
    float lf = R.lf, t = R.t;
    uint32_t pre = R.pre, lf_slot = R.lf_slot;
    int32_t step = R.step, sem = 0;

    while (live != 0ull) {
        step = add_lane_bit(step, live);
        const float qa = __builtin_fmaf(t, adm, om);
        const uint64_t m_dom = quad_none(wave_mask(!(qa <= dm)));
        const uint64_t m_hit_lf = quad_none(wave_mask(!(qa <= lf))) & live;
        const uint64_t m_desc = live & m_dom & ~m_hit_lf;
        // (lanes that do not descend: void marker and a face at +inf, see march_fast)
        float h = kInf;
        uint32_t slot = kSlotVoid;
        if (lane_in(m_desc)) {
            const float p = __uint_as_float(__float_as_uint(qa) ^ flip);
            // ---- the depth-8 cell along the axis ----
            float lo, hi;
            uint32_t j = plane_cell(p, off, scale, pl, kCells, lo, hi);
            // ---- the prefix cell (kernel.cu:120-132), when p is on one of its upper faces ----
            const uint64_t m_face = wave_mask(j == pre) & wave_mask(p == lo);
            uint64_t m_pre = 0ull;
            if (m_face != 0ull) {  // rare
                const uint64_t m_in = wave_mask((j >> kSh) + 1u == (pre >> kSh));
                m_pre = quad_any(m_face) & quad_all(m_face | m_in);
                if (lane_in(m_pre & m_face)) {
                    j -= 1u;
                    hi = lo;
                    lo = pl[j];
                }
            }
            // ---- the axes' index bits gathered over the quad: the table index
            // (x, y, z fields of D bits), then three octant bits per level below it ----
            uint32_t w = (j >> kUp) << (D * ax);
#pragma unroll
            for (uint32_t l = 0; l < kUp; ++l)
                w |= ((j >> (kUp - 1u - l)) & 1u) << (3u * (D + l) + ax);
            w = quad_or(w);  // (lane 3's j is 0)
            const navi_u32x2 e = navi_struct_load_b64(
                tables, static_cast<int32_t>(my_table | (w & ((1u << (3u * D)) - 1u))), 0, 0, 0);
            slot = e[0];
            uint32_t depth = e[1];
#pragma unroll
            for (uint32_t l = 0; l < kUp; ++l) {
                if (slot < kSlotBadChild) {
                    const uint32_t oct = __builtin_amdgcn_ubfe(w, 3u * (D + l), 3u);
                    slot = navi_struct_load_b32(records, static_cast<int32_t>((slot << 3) | oct), 0, 0, 0);
                    depth = D + l + 1u;
                }
            }
            // kernel.cu:154-163: a fresh descent caches its depth-4 cell when the path goes below depth 4
            const uint64_t m_save = ~m_pre & wave_mask(depth > kPrefixDepth);
            pre = lane_in(m_save) ? ((j >> kSh) + 1u) << kSh : pre;
            if (depth < kQuadPlanes) {
                // a leaf / void / fault above depth 8: its face ahead from the planes
                const uint32_t up = kQuadPlanes - depth;
                h = pl[((j >> up) + ahead_up) << up];
            } else {
                // ---- below the planes: one 4-byte slot per level (kernel.cu:136-199) ----
                bool deeper = slot < kSlotBadChild;
                for (uint32_t trip = kQuadPlanes; deeper && trip < static_cast<uint32_t>(kMaxDepth); ++trip) {
                    const float m = (lo + hi) * 0.5f;
                    const bool g = p >= m;
                    lo = g ? m : lo;
                    hi = g ? hi : m;
                    const uint32_t oct = quad_or(g ? 1u << axis : 0u);
                    slot = navi_struct_load_b32(records, static_cast<int32_t>((slot << 3) | oct), 0, 0, 0);
                    deeper = slot < kSlotBadChild;
                }
                h = lane_in(neg) ? lo : hi;
            }
            h = __uint_as_float((__float_as_uint(h) & face_keep) ^ face_flip);  // mirrored
        }

        // ---- the query's outcome and the leaf cache ----
        const uint64_t m_new = wave_mask(static_cast<int32_t>(slot) < 0);
        const uint64_t m_leaf = m_hit_lf | m_new;
        lf = lane_in(m_new) ? h : lf;
        lf_slot = lane_in(m_new) ? slot : lf_slot;
        if (kLeaves && P.leaves != nullptr && lane_in(m_new)) lf_slot = table_leaf_word(slot, P.leaves, P.n_leaves);

        // ---- finish the step (kernel.cu:54-85, 297-308): an axis's quotient
        // clamped to [1e-5, 1000] (NaN to 1000) is a positive float, ordered as
        // its bits are, so the quad takes the least of them as integers ----
        const float e = fmaxf(fminf(markstein(h - qa, adm, r), kOutsideDomain), kVoidAdvanceEps);
        const float void_d = __uint_as_float(quad_min(__float_as_uint(e)));
        const float leaf_d = half_to_float(lf_slot & 0xffffu);
        const int32_t leaf_s = static_cast<int32_t>(__builtin_amdgcn_ubfe(lf_slot, 16u, P.sem_bits));
        const bool on_leaf = lane_in(m_leaf);
        const float dist = on_leaf ? leaf_d : (slot == kSlotVoid ? void_d : nan);
        const uint64_t m_hit = m_leaf & wave_mask(leaf_s != 0) & wave_mask(dist < P.hit_eps);
        const float t_next = t + dist;
        uint64_t m_fin = live & (wave_mask(slot == kSlotFault) | m_hit | wave_mask(t_next > P.max_distance) |
                                 wave_mask(step >= P.max_steps));
        t = lane_in(live & ~m_hit) ? t_next : t;
        sem = lane_in(m_fin & m_hit) ? leaf_s : sem;

        // ---- further steps that the leaf cache answers alone ----
        uint64_t m_run = live & ~m_fin & m_leaf;
        for (uint32_t k = 0; k < kQuadLeafRun; ++k) {
            m_run &= quad_none(wave_mask(!(__builtin_fmaf(t, adm, om) <= lf)));
            if (m_run == 0ull) break;
            step = add_lane_bit(step, m_run);
            t = lane_in(m_run) ? t + dist : t;
            const uint64_t m_fin2 = m_run & (wave_mask(t > P.max_distance) | wave_mask(step >= P.max_steps));
            m_fin |= m_fin2;
            m_run &= ~m_fin2;
        }
        live &= ~m_fin;
    }
    R.t = t;
    R.step = step;
    R.sem = sem;
}

// The fast march of a wave's rays (march_fast, an axis a lane): box [lo_a, hi_a]
// of scene S along the lane's axis with the plane lookup's scale and offset, the
// ray's origin o and direction d along it.
template <int kDepth>
__device__ __forceinline__ QuadResult quad_fast(const RelaidParams& P, const navi_relaid_scene& S, uint32_t scene,
                                                float lo_a, float hi_a, float scale, float off, float o, float d,
                                                bool has_ray, float* planes) {
    constexpr uint32_t D = kDepth;
    const uint32_t lane = threadIdx.x;
    const uint32_t axis = lane & 3u;
    const uint32_t ax = axis == 3u ? 0u : axis;
    stage_quad_planes(S.bbox_min, S.bbox_max, lane, planes);
    __syncthreads();
    const float nan = __builtin_nanf("");
    constexpr float kInf = __builtin_inff();
    const uint64_t neg = wave_mask(__float_as_int(d) < 0 && axis != 3u);  // the mirrored axes
    const bool inside = lane_in(quad_all(wave_mask(o >= lo_a && o <= hi_a)));
    const bool root_leaf = (S.root_slot & 0x80000000u) != 0u;  // a one-leaf DAG: its leaf is the domain
    QuadRay R;
    R.pl = planes + ax * kQuadAxis;
    R.scale = axis == 3u ? 0.f : scale;
    R.off = axis == 3u ? 0.f : off;
    R.om = axis == 3u ? 0.f : mirror(o, d);
    R.adm = axis == 3u ? 0.f : fabsf(d);
    R.r = (axis != 3u && (d > kDirEps || d < -kDirEps)) ? fabsf(1.0f / d) : nan;
    R.dm = axis == 3u ? kInf : (inside ? (lane_in(neg) ? -lo_a : hi_a) : nan);
    R.lf = root_leaf || axis == 3u ? R.dm : nan;
    R.lf_slot = (P.leaves != nullptr && root_leaf) ? table_leaf_word(S.root_slot, P.leaves, P.n_leaves) : S.root_slot;
    R.pre = 0xffffffffu;
    R.table = scene << (3u * D);
    R.t = 0.f;
    R.step = 0;
    quad_march<kDepth, true>(P, neg, wave_mask(has_ray), R);
    return {R.t, R.step, R.sem};
}

// The general march of a wave's rays (march in trace_relaid.hip, an axis a
// lane): any box, depth, leaf sign and range. Boxes come from splits, every
// cache of kernel.cu:236-247 is kept, and the exit divides.
template <int kDepth>
__device__ __forceinline__ QuadResult quad_general(const RelaidParams& P, const navi_relaid_scene& S, uint32_t scene,
                                                   float lo_a, float hi_a, float o, float d, bool has_ray) {
    constexpr uint32_t D = kDepth;
    const uint32_t axis = threadIdx.x & 3u;
    const uint32_t bit = axis == 3u ? 0u : 1u << axis;  // the axis's octant bit
    const float nan = __builtin_nanf("");
    const bool leaves_axis = axis != 3u && (d > kDirEps || d < -kDirEps);  // the exit uses the axis
    // a one-leaf DAG: its leaf is the domain (see march)
    const bool root_leaf = (S.root_slot & 0x80000000u) != 0u;
    float lf_lo = lo_a, lf_hi = hi_a, vd_lo = lo_a, vd_hi = hi_a, pre_lo = lo_a, pre_hi = hi_a;
    uint64_t lf_ok = root_leaf ? ~0ull : 0ull, vd_ok = 0ull, pre_ok = 0ull;
    uint32_t lf_slot = root_leaf ? (P.leaves != nullptr ? table_leaf_word(S.root_slot, P.leaves, P.n_leaves)
                                                        : S.root_slot) : 0u;
    uint32_t pre_j = 0u;  // the prefix cell's depth-4 index along the axis
    float t = 0.f, dist = 0.f;
    int32_t step = 0, sem = 0;
    // one split of [lo, hi] at its midpoint (kernel.cu:165-176), to the upper half where up
    auto split = [](float& lo, float& hi, float m, bool up) {
        lo = up ? m : lo;
        hi = up ? hi : m;
    };
    uint64_t live = wave_mask(has_ray);
    while (live != 0ull) {
        step = add_lane_bit(step, live);
        const float p = __builtin_fmaf(t, d, o);
        // kernel.cu:265-267, 108-118, as exclusive outcomes
        const uint64_t m_vd = live & vd_ok & quad_all(wave_mask(p > vd_lo) & wave_mask(p < vd_hi));
        const uint64_t m_in = quad_all(wave_mask(p >= lo_a) & wave_mask(p <= hi_a));
        const uint64_t m_out = live & ~m_vd & ~m_in;
        const uint64_t m_lf = live & ~m_vd & m_in & lf_ok & quad_all(wave_mask(p >= lf_lo) & wave_mask(p <= lf_hi));
        const uint64_t m_desc = live & ~(m_vd | m_out | m_lf);
        uint32_t slot = 0u;
        uint32_t depth = 0u;
        float lo = lo_a, hi = hi_a;
        bool save = false;  // per lane: a mask made where only some lanes run must not leave there
        uint32_t j = 0u;
        if (lane_in(m_desc)) {
            // the depth-D cell, from the prefix cell (kernel.cu:120-132) or the root
            const uint64_t m_pre = pre_ok & quad_all(wave_mask(p >= pre_lo) & wave_mask(p <= pre_hi));
            const bool use_pre = lane_in(m_pre);
            lo = use_pre ? pre_lo : lo_a;
            hi = use_pre ? pre_hi : hi_a;
            j = use_pre ? pre_j : 0u;
            if (!use_pre) {
                for (uint32_t l = 0; l < static_cast<uint32_t>(kPrefixDepth); ++l) {
                    const float m = (lo + hi) * 0.5f;
                    j = append_bit(j, p >= m);
                    split(lo, hi, m, p >= m);
                }
            }
            for (uint32_t l = kPrefixDepth; l < D; ++l) {
                const float m = (lo + hi) * 0.5f;
                j = append_bit(j, p >= m);
                split(lo, hi, m, p >= m);
            }
            const uint32_t idx = quad_or(axis == 3u ? 0u : j << (D * axis));
            const uint64_t e = P.cell_table[(scene << (3u * D)) | idx];
            slot = static_cast<uint32_t>(e);
            depth = static_cast<uint32_t>(e >> 32);
            if (depth < D) {
                lo = lo_a;
                hi = hi_a;
                for (uint32_t l = 0; l < depth; ++l) split(lo, hi, (lo + hi) * 0.5f, (j >> (D - 1u - l)) & 1u);
            }
            // kernel.cu:154-163
            save = !use_pre && (depth > kPrefixDepth || (depth == kPrefixDepth && slot < kSlotBadChild));
            if (save) {
                pre_j = j >> (D - kPrefixDepth);
                pre_lo = lo_a;
                pre_hi = hi_a;
                for (uint32_t l = 0; l < static_cast<uint32_t>(kPrefixDepth); ++l)
                    split(pre_lo, pre_hi, (pre_lo + pre_hi) * 0.5f, (pre_j >> (kPrefixDepth - 1u - l)) & 1u);
            }
            // below the table (kernel.cu:136-199); a record past the pool (a corrupt one) reads as slot 0
            while (slot < kSlotBadChild && depth < static_cast<uint32_t>(kMaxDepth)) {
                const float m = (lo + hi) * 0.5f;
                const uint32_t oct = quad_or(p >= m ? bit : 0u);
                split(lo, hi, m, p >= m);
                slot = slot < P.n_records ? P.records[8ull * slot + oct] : 0u;
                ++depth;
            }
            // a bad child index faults only where the reference examines the
            // child, above the 32-level limit; at depth 32 the result is stale
            slot = slot == kSlotBadChild && depth < static_cast<uint32_t>(kMaxDepth) ? kSlotFault : slot;
        }
        pre_ok |= wave_mask(save);
        // classify and update the caches (lanes that did not descend hold slot 0)
        const uint64_t m_new_leaf = wave_mask((slot & 0x80000000u) != 0u) & wave_mask(depth < static_cast<uint32_t>(kMaxDepth));
        const uint64_t m_new_void = wave_mask(slot == kSlotVoid);
        const uint64_t m_fault = wave_mask(slot == kSlotFault);
        if (lane_in(m_new_void)) {
            vd_lo = lo;
            vd_hi = hi;
        }
        if (lane_in(m_new_leaf)) {
            lf_lo = lo;
            lf_hi = hi;
            lf_slot = P.leaves != nullptr ? table_leaf_word(slot, P.leaves, P.n_leaves) : slot;
        }
        vd_ok |= m_new_void;
        lf_ok |= m_new_leaf;
        const uint64_t m_void = m_vd | m_new_void, m_leaf = m_lf | m_new_leaf;
        // kernel.cu:54-85 on the void box; see quad_fast for the minimum
        const float n = (d > 0.f ? vd_hi : vd_lo) - p;
        const float exit = leaves_axis ? n / d : kOutsideDomain;
        const float void_d = __uint_as_float(
            quad_min(__float_as_uint(fmaxf(fminf(exit, kOutsideDomain), kVoidAdvanceEps))));
        const float leaf_d = half_to_float(lf_slot & 0xffffu);
        const int32_t leaf_s = static_cast<int32_t>(__builtin_amdgcn_ubfe(lf_slot, 16u, P.sem_bits));
        // stale (32 levels without leaf or void): dist and sem keep their values
        const bool is_void = lane_in(m_void), is_leaf = lane_in(m_leaf), outside = lane_in(m_out);
        dist = is_void ? void_d : (is_leaf ? leaf_d : (outside ? kOutsideDomain : dist));
        sem = is_void ? 0 : (is_leaf ? leaf_s : (outside ? 0 : sem));
        // kernel.cu:297-308
        const uint64_t m_hit = live & ~m_fault & wave_mask(sem != 0) & wave_mask(dist < P.hit_eps);
        const float t_next = t + dist;
        const uint64_t m_fin = live & (m_fault | m_hit | wave_mask(t_next > P.max_distance) |
                                       wave_mask(step >= P.max_steps));
        t = lane_in(live & ~m_hit) ? t_next : t;
        t = lane_in(m_fin & m_fault) ? nan : t;
        sem = lane_in(m_fin & ~m_hit) ? 0 : sem;
        live &= ~m_fin;
    }
    return {t, step, sem};
}

// See the head of the file.
template <int kDepth, bool kPoses>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(8))) void trace_quad_kernel(RelaidParams P) {
    static_assert(kDepth >= 4 && kDepth <= 7, "cell tables of 4 to 7 levels");
    constexpr uint32_t kCells = 1u << kQuadPlanes;
    __shared__ __align__(16) float planes[3u * kQuadAxis];
    const uint32_t lane = threadIdx.x;
    const uint32_t unit = unit_of_block(blockIdx.x, gridDim.x);
    const uint32_t axis = lane & 3u;
    const uint32_t ax = axis == 3u ? 0u : axis;  // lane 3 of a quad loads what lane 0 loads and counts for nothing

    // ---- the unit's env and scene (uniform) ----
    const uint32_t env_pos = fdiv(unit, P.div_units);
    const int32_t env = P.env_order ? P.env_order[env_pos] : static_cast<int32_t>(env_pos);
    if (static_cast<uint32_t>(env) >= P.n_envs) return;
    const int32_t sc = P.env_scene ? P.env_scene[env] : 0;
    const uint32_t i = lane >> 2;
    const uint32_t q = i < (1u << P.quad_shift) ? unit_ray(P, unit, i) : 0xffffffffu;
    const bool has_ray = q != 0xffffffffu;
    int32_t env_again = 0;
    const uint32_t ray = has_ray ? ray_of(P, q, env_again) : 0u;
    if (sc < 0 || sc >= P.n_scenes) {
        // unknown scene: reported like a fault, no steps
        if (has_ray && axis == 0u) {
            store_distance(P, ray, __builtin_nanf(""));
            P.out_s[ray] = 0;
            if (P.out_steps) P.out_steps[ray] = 0;
        }
        return;
    }
    const navi_relaid_scene& S = P.scenes[sc];

    // ---- what the fast march needs of the scene (see stage_scenes and
    // stage_planes). With |off| <= 2^16 every plane lies within 2^-5 cell of
    // the uniform grid: a level's midpoint is off by at most half an ulp of the
    // largest coordinate, 2^-24 of (2^16 + 2^8) cells, which eight levels add
    // up, and the offset is exact to half of its ulp, 2^-8 cell: what plane_cell
    // allows is 0.2 cell and more. (The combined kernel's planes are 2^6, so its
    // 2^14 reaches as far: a 512^3 room grid 100 of its sides from the origin,
    // 49 K rays, takes 209 us, 324 in the general march.) ----
    const float lo_a = S.bbox_min[ax], hi_a = S.bbox_max[ax];
    const float extent = hi_a - lo_a;
    const float scale = static_cast<float>(kCells) / extent;
    const float off = __builtin_fmaf(-lo_a, scale, -0.25f);
    const double cw = (static_cast<double>(hi_a) - static_cast<double>(lo_a)) / kCells;
    const bool axis_ok = fabsf(lo_a) < 0x1p100f && fabsf(hi_a) < 0x1p100f && extent > 0.0f && scale > 0.0f &&
                         scale <= 0x1p127f && cw > 0.0 && fabs(static_cast<double>(scale) * cw - 1.0) <= 1e-6 &&
                         fabsf(off) <= 0x1p16f;
    const bool shallow = S.max_depth <= static_cast<uint32_t>(kMaxDepth - 2);
    const bool monotone = (S.flags & NAVI_SCENE_NONNEG_LEAVES) != 0u;
    const bool fast = shallow && monotone && P.small_tables != 0u && P.max_distance < kOutsideDomain &&
                      wave_mask(!axis_ok) == 0ull;

    // ---- the lane's axis of its ray: origin and direction ----
    float o = 0.f, d = 0.f;
    if (has_ray) {
        if (kPoses) {
            const uint32_t r = ray - static_cast<uint32_t>(env) * P.rays_per_env;
            const float c = P.env_rot[2 * env], s = P.env_rot[2 * env + 1];
            const float lx = P.local_dirs[3 * r + 0], ly = P.local_dirs[3 * r + 1], lz = P.local_dirs[3 * r + 2];
            const float dx = lx * c + lz * s;
            const float dz = (-lx) * s + lz * c;
            o = P.env_pos[3 * env + ax];
            d = ax == 0u ? dx : (ax == 1u ? ly : dz);
        } else {
            o = P.origins[3 * ray + ax];
            d = P.dirs[3 * ray + ax];
        }
    }
    QuadResult out;
    if (fast) {
        out = quad_fast<kDepth>(P, S, static_cast<uint32_t>(sc), lo_a, hi_a, scale, off, o, d, has_ray, planes);
    } else {
        out = quad_general<kDepth>(P, S, static_cast<uint32_t>(sc), lo_a, hi_a, o, d, has_ray);
    }
    if (has_ray && axis == 0u) {
        store_distance(P, ray, out.t);
        __builtin_nontemporal_store(out.sem, &P.out_s[ray]);
        if (P.out_steps) P.out_steps[ray] = out.step;
    }
}

}  // namespace navi
