// The solver of small worlds: one workgroup takes a world through everything that solver_prepare and
// solver_substeps launch kernel by kernel (block set-up, substeps, impulses back), with the rows'
// velocities, delta words, resolutions and poses in LDS. Included by world.hip inside its namespace.
//
// What bounds it: the latency of a few hundred barrier-separated phases, each a pass of the world's
// contacts or rows, against a launch and its gap (about 5 us) for each of them when launched. The
// blocks' deltas are the same fixed-point words, summed by LDS atomics in place of the rows' lists
// (integer sums, any order), and every expression is the launched passes' own function, so the results
// are the launched passes' bit for bit. The blocks are solved by quads (solve_block), and where there is
// a quad for each its block and bodies stay in registers through a substep's iterations: 24 mixed bodies
// (31 contacts) take 97 us a step, and 167 with a lane a block and everything read back each time.
#pragma once

// A world of a batch: its rows (simulated ones, then the others) and its colliders.
struct GroupWorld {
    uint32_t dynamic_base, dynamic_count, static_base, static_count, collider_base, collider_count;
    uint32_t pad[2];
};

// LDS words per row: what the row resolved (3), its block count and marks (1), then either the
// velocities (6) and their delta words (6) or the pose (7), the position words (3) and their count (1).
constexpr uint32_t kGroupRowWords = 16;
constexpr uint32_t kGroupListed = 1u << 31;  // the row has blocks and is not inert
constexpr uint32_t kGroupMarked = 1u << 30;  // an inert row that a position block touched
constexpr uint32_t kGroupCount = kGroupMarked - 1u;

struct GroupLds {
    uint32_t* at;
    uint32_t rows;
    GroupWorld g;

    __device__ __forceinline__ uint32_t local(uint32_t row) const {
        const uint32_t d = row - g.dynamic_base;
        return d < g.dynamic_count ? d : g.dynamic_count + (row - g.static_base);
    }
    __device__ __forceinline__ uint32_t global(uint32_t r) const {
        return r < g.dynamic_count ? g.dynamic_base + r : g.static_base + (r - g.dynamic_count);
    }
    __device__ __forceinline__ uint32_t& word(uint32_t k, uint32_t r) const { return at[k * rows + r]; }
    __device__ __forceinline__ float get(uint32_t k, uint32_t r) const { return __uint_as_float(at[k * rows + r]); }
    __device__ __forceinline__ void set(uint32_t k, uint32_t r, float v) const { at[k * rows + r] = __float_as_uint(v); }
    __device__ __forceinline__ v3 get3(uint32_t k, uint32_t r) const { return mk(get(k, r), get(k + 1u, r), get(k + 2u, r)); }
    __device__ __forceinline__ void set3(uint32_t k, uint32_t r, v3 v) const {
        set(k, r, v.x);
        set(k + 1u, r, v.y);
        set(k + 2u, r, v.z);
    }
};
// word offsets of a row
constexpr uint32_t kGrResolved = 0, kGrBlocks = 3, kGrVelocity = 4, kGrWords = 10, kGrPose = 4, kGrMove = 11, kGrSides = 14;

// Where a group's block deltas go: each non-inert side's words added to the row's words in LDS, three
// a lane.
struct GroupCommit {
    const GroupLds& l;
    uint32_t* linear;   // with `residual`: this thread's largest delta words
    uint32_t* angular;
    bool residual;
    __device__ __forceinline__ void operator()(uint32_t lane, uint32_t fb, uint32_t sb, bool fi, bool si, v3 da, v3 sa,
                                               v3 db, v3 sbv) const {
        const v3 part = quad_part(lane, da, sa, db, sbv);
        if (!(lane & 2u ? si : fi)) {
            const uint32_t r = l.local(lane & 2u ? sb : fb), k = kGrWords + 3u * (lane & 1u);
            const float scale = DYN_SOLVER_VELOCITY_SCALE;
            atomicAdd(&l.word(k, r), solver_word(part.x, scale));
            atomicAdd(&l.word(k + 1u, r), solver_word(part.y, scale));
            atomicAdd(&l.word(k + 2u, r), solver_word(part.z, scale));
        }
        if (!residual) return;
        *linear = max(*linear, solver_word(fmx(len3(da), len3(db)), DYN_SOLVER_VELOCITY_SCALE));
        *angular = max(*angular, solver_word(fmx(len3(sa), len3(sbv)), DYN_SOLVER_VELOCITY_SCALE));
    }
};

// A row's velocities. An inert row's never change, so its record's would do; LDS holds the same.
__device__ __forceinline__ void group_velocity(const GroupLds& l, uint32_t row, SolverBody* b) {
    const uint32_t r = l.local(row);
    b->v = l.get3(kGrVelocity, r);
    b->w = l.get3(kGrVelocity + 3u, r);
}

// The first contact whose collider a is at least `collider`: contacts are in (a, b) order, and a
// wave reads 64 places at once.
__device__ __forceinline__ uint32_t group_lower_bound(const uint2* keys, uint32_t count, uint32_t collider) {
    uint32_t lo = 0, hi = count;  // the answer lies in [lo, hi]
    const uint32_t lane = lane_id();
    while (hi - lo > static_cast<uint32_t>(kWave)) {
        const uint32_t step = (hi - lo) / kWave;
        const uint32_t less = static_cast<uint32_t>(__popcll(__ballot(keys[lo + (lane + 1u) * step - 1u].x < collider)));
        if (less < static_cast<uint32_t>(kWave)) hi = lo + (less + 1u) * step - 1u;
        lo += less * step;
    }
    const bool below = lo + lane < hi && keys[lo + lane].x < collider;
    return lo + static_cast<uint32_t>(__popcll(__ballot(below)));
}

// The rows' deltas of one velocity pass onto their velocities (k_apply), the words cleared.
template <uint32_t T>
__device__ __forceinline__ void group_apply(const GroupLds& l) {
    for (uint32_t r = threadIdx.x; r < l.rows; r += T) {
        if (!(l.word(kGrBlocks, r) & kGroupListed)) continue;
        uint32_t s[6];
#pragma unroll
        for (uint32_t k = 0; k < 6; ++k) s[k] = l.word(kGrWords + k, r);
        if ((s[0] | s[1] | s[2] | s[3] | s[4] | s[5]) == 0u) continue;
#pragma unroll
        for (uint32_t k = 0; k < 6; ++k) {
            l.word(kGrWords + k, r) = 0u;
            l.set(kGrVelocity + k, r, l.get(kGrVelocity + k, r) + solver_value(s[k], DYN_SOLVER_VELOCITY_SCALE));
        }
    }
}

// k_advance and the position iterations (k_position_block, k_position_apply) of a group whose rows'
// block words and resolutions are in LDS. A thread serves the same rows throughout, so only the
// blocks' passes need barriers around them.
template <uint32_t T>
__device__ __forceinline__ void group_position(const W& w, const GroupLds& l, uint32_t c0, uint32_t c1) {
    const uint32_t t = threadIdx.x;
    // the poses of the rows with blocks go into LDS for the iterations
    for (uint32_t r = t; r < l.rows; r += T) {
        const uint32_t row = l.global(r);
        if (r < l.g.dynamic_count) advance_at(w, row);
        if (l.word(kGrBlocks, r) == 0u) continue;
        const dyn_body_state& s = w.st[row];
        l.set3(kGrPose, r, ld3(s.position));
        const float4 q = ld4(s.orientation);
        l.set3(kGrPose + 3u, r, mk(q.x, q.y, q.z));
        l.set(kGrPose + 6u, r, q.w);
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) l.word(kGrMove + k, r) = 0u;  // the words and their count
    }
    // the first kHeld contacts of a thread stay in its registers through the iterations
    constexpr uint32_t kHeld = 4;
    PositionRow held[kHeld];
    uint32_t held_flags[kHeld], held_first[kHeld], held_second[kHeld];
#pragma unroll
    for (uint32_t k = 0; k < kHeld; ++k) {
        const uint32_t ci = c0 + t + k * T;
        held_flags[k] = held_first[k] = held_second[k] = 0u;
        held[k] = PositionRow{0.0f, 0.0f, zero3v(), make_float4(0.0f, 0.0f, 0.0f, 0.0f)};
        if (ci < c1) {
            const float4* prow = w.prows + 3u * ci;
            const float4 h0 = prow[0];
            held_flags[k] = __float_as_uint(h0.z);
            if (held_flags[k] & 7u) {
                held_first[k] = l.local(__float_as_uint(h0.x));
                held_second[k] = l.local(__float_as_uint(h0.y));
                held[k] = load_position_row(h0, prow);
            }
        }
    }
    auto correct = [&](uint32_t flags, const PositionRow& row, uint32_t f, uint32_t s) {
        v3 la, lb;
        if (!position_correction(w, row, flags & 7u, l.get3(kGrResolved, f), l.get3(kGrResolved, s), &la, &lb)) return;
        const float scale = DYN_SOLVER_POSITION_SCALE;
        if (flags & 8u) {  // inert rows get only the mark of one
            l.word(kGrSides, f) = 1u;
        } else {
            atomicAdd(&l.word(kGrSides, f), 1u);
            atomicAdd(&l.word(kGrMove, f), solver_word(la.x, scale));
            atomicAdd(&l.word(kGrMove + 1u, f), solver_word(la.y, scale));
            atomicAdd(&l.word(kGrMove + 2u, f), solver_word(la.z, scale));
        }
        if (flags & 16u) {
            l.word(kGrSides, s) = 1u;
        } else {
            atomicAdd(&l.word(kGrSides, s), 1u);
            atomicAdd(&l.word(kGrMove, s), solver_word(lb.x, scale));
            atomicAdd(&l.word(kGrMove + 1u, s), solver_word(lb.y, scale));
            atomicAdd(&l.word(kGrMove + 2u, s), solver_word(lb.z, scale));
        }
    };
    __syncthreads();
    for (uint32_t it = 0; it < w.p.position_iterations; ++it) {
#pragma unroll
        for (uint32_t k = 0; k < kHeld; ++k) {
            if (held_flags[k] & 7u) correct(held_flags[k], held[k], held_first[k], held_second[k]);
        }
        for (uint32_t ci = c0 + t + kHeld * T; ci < c1; ci += T) {
            const float4* prow = w.prows + 3u * ci;
            const float4 h0 = prow[0];
            const uint32_t flags = __float_as_uint(h0.z);
            if ((flags & 7u) == 0u) continue;
            correct(flags, load_position_row(h0, prow), l.local(__float_as_uint(h0.x)), l.local(__float_as_uint(h0.y)));
        }
        __syncthreads();
        for (uint32_t r = t; r < l.rows; r += T) {
            const uint32_t blocks = l.word(kGrBlocks, r);
            if (blocks == 0u) continue;
            const uint32_t sides = l.word(kGrSides, r);
            if (sides == 0u) continue;
            v3 p1, moved;
            float4 q1;
            const v3 q = l.get3(kGrPose + 3u, r);
            position_move(l.get3(kGrPose, r), make_float4(q.x, q.y, q.z, l.get(kGrPose + 6u, r)), l.word(kGrMove, r),
                          l.word(kGrMove + 1u, r), l.word(kGrMove + 2u, r), sides, &p1, &q1, &moved);
            l.set3(kGrPose, r, p1);
            l.set3(kGrPose + 3u, r, mk(q1.x, q1.y, q1.z));
            l.set(kGrPose + 6u, r, q1.w);
            l.set3(kGrResolved, r, add(l.get3(kGrResolved, r), moved));
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k) l.word(kGrMove + k, r) = 0u;
            if (!(blocks & kGroupListed)) l.word(kGrBlocks, r) = blocks | kGroupMarked;
        }
        __syncthreads();
    }
    for (uint32_t r = t; r < l.rows; r += T) {
        if (!(l.word(kGrBlocks, r) & (kGroupListed | kGroupMarked))) continue;
        dyn_body_state& s = w.st[l.global(r)];
        st3(s.position, l.get3(kGrPose, r));
        const v3 q = l.get3(kGrPose + 3u, r);
        st4(s.orientation, make_float4(q.x, q.y, q.z, l.get(kGrPose + 6u, r)));
    }
}

// The workgroup's world, its rows' LDS and its contacts, [range[0], range[1]) after a barrier.
// `worlds` null: one world of all rows and contacts.
__device__ __forceinline__ GroupLds group_begin(const W& w, const GroupWorld* worlds, uint32_t* lds, uint32_t* range) {
    const uint32_t t = threadIdx.x;
    GroupLds l;
    l.g = worlds ? worlds[blockIdx.x] : GroupWorld{0u, w.d, w.d, w.n - w.d, 0u, w.k, {0u, 0u}};
    l.at = lds;
    l.rows = l.g.dynamic_count + l.g.static_count;
    const uint32_t all = *w.ncontacts;
    if (worlds) {
        if (t < 2u * kWave) {
            const uint32_t end = t / kWave;
            const uint32_t at = group_lower_bound(w.ckeys, all, l.g.collider_base + (end ? l.g.collider_count : 0u));
            if (lane_id() == 0u) range[end] = at;
        }
    } else if (t == 0u) {
        range[0] = 0u;
        range[1] = all;
    }
    return l;
}

// A substep's advance and position iterations of worlds whose velocities were solved by the launched
// passes: one launch for 2 x position_iterations + 1 of them.
template <uint32_t T>
__global__ void __launch_bounds__(T) k_group_position(W w, const GroupWorld* worlds, uint32_t first, uint32_t last) {
    extern __shared__ uint32_t group_lds[];
    __shared__ uint32_t range[2];
    const GroupLds l = group_begin(w, worlds, group_lds, range);
    float4* resolution = reinterpret_cast<float4*>(w.resolution);
    for (uint32_t r = threadIdx.x; r < l.rows; r += T) {
        const uint32_t row = l.global(r);
        l.word(kGrBlocks, r) = w.block_counts[row] | (w.list_counts[row] != 0u ? kGroupListed : 0u);
        const float4 done = first ? make_float4(0.0f, 0.0f, 0.0f, 0.0f) : resolution[row];
        l.set3(kGrResolved, r, mk(done.x, done.y, done.z));
    }
    __syncthreads();
    group_position<T>(w, l, range[0], range[1]);
    if (last) return;
    for (uint32_t r = threadIdx.x; r < l.rows; r += T) {
        const v3 done = l.get3(kGrResolved, r);
        resolution[l.global(r)] = make_float4(done.x, done.y, done.z, 0.0f);
    }
}

template <uint32_t T>
__global__ void __launch_bounds__(T) k_group_solve(W w, const GroupWorld* worlds) {
    extern __shared__ uint32_t group_lds[];
    __shared__ uint32_t range[2], totals[2];
    const uint32_t t = threadIdx.x, lane = t % 4u;
    const GroupLds l = group_begin(w, worlds, group_lds, range);
    if (t < 2u) totals[t] = 0u;
    // SolverReset and the blocks (k_solver_reset, k_blocks, k_rows_count)
    uint32_t live = 0;
    for (uint32_t r = t; r < l.rows; r += T) {
        const uint32_t row = l.global(r);
        l.word(kGrBlocks, r) = 0u;
        l.set3(kGrResolved, r, zero3v());
        const Body b = load_body(w, row);
        if (row < w.d && body_is_active(b.s, b.d)) ++live;
        write_block_body(w, row, b);
    }
    __syncthreads();
    const uint32_t c0 = range[0], c1 = range[1];
    for (uint32_t ci = c0 + t; ci < c1; ci += T) {
        uint32_t fb, sb;
        bool fi, si;
        if (!write_block(w, ci, &fb, &sb, &fi, &si)) continue;
        uint32_t &nf = l.word(kGrBlocks, l.local(fb)), &ns = l.word(kGrBlocks, l.local(sb));
        if (fi) nf = 1u; else atomicAdd(&nf, 1u);
        if (si) ns = 1u; else atomicAdd(&ns, 1u);
    }
    __syncthreads();
    uint32_t claimed = 0;
    for (uint32_t r = t; r < l.rows; r += T) {
        const uint32_t blocks = l.word(kGrBlocks, r);
        if (blocks == 0u) continue;
        ++claimed;
        const uint32_t row = l.global(r);
        if (kind_simulates(w.de[row]) && w.st[row].sleeping == 0u) l.word(kGrBlocks, r) = blocks | kGroupListed;
    }
    live = wave_sum(live);
    claimed = wave_sum(claimed);
    if (lane_id() == 0u) {
        if (live) atomicAdd(&totals[0], live);
        if (claimed) atomicAdd(&totals[1], claimed);
    }
    __syncthreads();
    if (t == 0u && totals[0]) atomicAdd(cw(w.counters, DYN_COUNTER_LIVE), totals[0]);
    if (t == 0u && totals[1]) atomicAdd(cw(w.counters, DYN_COUNTER_SOLVER_ROWS), totals[1]);
    uint32_t linear = 0, angular = 0;
    for (uint32_t sub = 0; sub < w.p.substeps; ++sub) {
        // k_integrate
        for (uint32_t r = t; r < l.rows; r += T) {
            const uint32_t row = l.global(r);
            if (r < l.g.dynamic_count) integrate_at(w, row);
            const uint32_t blocks = l.word(kGrBlocks, r) & kGroupCount;
            if (blocks == 0u) continue;
            const Body b = write_solver_body(w, row, blocks);
            l.set3(kGrVelocity, r, ld3(b.s.velocity));
            l.set3(kGrVelocity + 3u, r, ld3(b.s.angular_velocity));
#pragma unroll
            for (uint32_t k = 0; k < 6; ++k) l.word(kGrWords + k, r) = 0u;
        }
        __syncthreads();
        for (uint32_t ci = c0 + t / 4u; ci < c1; ci += T / 4u) {
            solve_prep_at(w, ci, lane, sub == 0u ? 1u : 0u);
            if (sub == 0u) warm_block(w, ci, lane, GroupCommit{l, nullptr, nullptr, false});
        }
        __syncthreads();
        if (sub == 0u) {
            group_apply<T>(l);
            __syncthreads();
        }
        // a block for every quad: it stays in registers through the iterations
        const bool held = c1 - c0 <= T / 4u;
        BlockLane b{};
        SolverBody bf{}, bs{};
        for (uint32_t it = 0; it < w.p.solve_iterations; ++it) {
            const bool last = it + 1u == w.p.solve_iterations;
            const GroupCommit commit{l, &linear, &angular, sub == 0u && last};
            for (uint32_t ci = c0 + t / 4u; ci < c1; ci += T / 4u) {
                if (!held || it == 0u) {
                    b = load_block(w, ci, lane);
                    bf = load_solver_body(w, b.fb);  // row 0 for a block without rows
                    bs = load_solver_body(w, b.sb);
                }
                if (!(b.flags & kRowActive)) continue;
                group_velocity(l, b.fb, &bf);
                group_velocity(l, b.sb, &bs);
                solve_block(w, lane, b, bf, bs, commit);
                if (!held || last) store_impulses(w, ci, lane, b);
            }
            __syncthreads();
            group_apply<T>(l);
            __syncthreads();
        }
        // the velocities back to the states
        for (uint32_t r = t; r < l.rows; r += T) {
            if (!(l.word(kGrBlocks, r) & kGroupListed)) continue;
            dyn_body_state& s = w.st[l.global(r)];
            st3(s.velocity, l.get3(kGrVelocity, r));
            st3(s.angular_velocity, l.get3(kGrVelocity + 3u, r));
        }
        group_position<T>(w, l, c0, c1);
    }
    if (linear) atomicMax(cw(w.counters, DYN_COUNTER_SOLVE_LINEAR_RESIDUAL), linear);
    if (angular) atomicMax(cw(w.counters, DYN_COUNTER_SOLVE_ANGULAR_RESIDUAL), angular);
    for (uint32_t ci = c0 + t; ci < c1; ci += T) impulses_store_at(w, ci);
}
