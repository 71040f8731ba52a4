// sphk_walk.hip -- the two neighbour walks of the SPH step (density; forces + integration).
//
// Work item ("chunk"): up to 64 consecutive cell-sorted particles of one (x,y) column of
// the dense grid, one per lane of a 64-wide wavefront.  Within a column the sort order is
// ascending z cell, so a chunk covers z cells [zmin, zmax] and all of its candidate
// neighbours lie in the 3x3 neighbouring columns between z cells zmin-1 and zmax+1 (widened
// to +-2 on an axis when `axis_edge_flags` proves a pair two cells apart possible for some
// lane of the chunk).  Each column contributes one contiguous range of sorted slots.
//
// Phase 1 (test): the chunk's candidate words (32 consecutive slots of one column) are
//   visited in the cursor's order (parts, passes, columns: see kPasses), and each lane gets
//   one bit per candidate from the conservative integer filter: on the matrix cores
//   (filter_word, 32 candidates x 64 targets per word), or one candidate at a time for
//   the whole wave (push_quant) in the words that span too many z cells for them and, with the
//   candidate data through the scalar cache, in the force walk's re-test and the
//   neighbour-list export; the bits are the same.  `wj0[w]` is the sorted slot of the first
//   candidate of word w.  Segments hold up to kSeg - 1 words and never span two parts.
// Phase 2 (evaluate): every lane walks only its own set bits and evaluates the kernel for
//   those pairs (pairs the filter let through beyond the radius weigh exactly zero).
// The density pass stores the words of each chunk in HBM (masks, wj0, word count, part
// starts) and the force rows of each particle; the force pass reads them back instead of
// testing again.  Chunks with more words than the engine stores (StepConsts::max_words: 256,
// or 128 for engines whose word buffers would pass 16 GiB; pile-ups of thousands of particles
// per cell) are re-tested by the force pass.  The neighbour-list export walks the reference's
// (dx, dy, dz, id) order.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>

#include "sphk_walk_pairs.h"

namespace sphk {

// ---------------------------------------------------------------------------
// chunk list: per column, ceil(len/64) chunks of consecutive sorted slots
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_chunk_count(const uint32_t* __restrict__ cs,
                                                     StepConsts c,
                                                     const SceneGrid* __restrict__ scenes,
                                                     uint32_t* __restrict__ cnt) {
    const uint32_t col = blockIdx.x * blockDim.x + threadIdx.x;
    if (col > c.ncols) return;
    if (col == c.ncols) {
        cnt[col] = 0;
        return;
    }
    const SceneGrid g = scenes[scene_of_col(scenes, c.nscenes, col)];
    const uint32_t first = g.cell_base + (col - g.col_base) * (uint32_t)g.nz;
    const uint32_t a = cs[first], b = cs[first + (uint32_t)g.nz];
    cnt[col] = (b - a + 63u) / 64u;
}

constexpr uint32_t kLoneChunks = 1100;  // see lone_chunk

// The number of chunks and, from the density walk before this list (lone_chunk), whether the
// team walks of this step give every wavefront a chunk of its own.
__device__ __forceinline__ void publish_chunks(uint32_t* __restrict__ nitems, uint32_t total) {
    nitems[2] = 2u * nitems[1] > nitems[0] && total >= kLoneChunks ? 1u : 0u;
    nitems[1] = 0u;
    nitems[0] = total;
}

__global__ __launch_bounds__(256) void k_chunk_fill(const uint32_t* __restrict__ cs, StepConsts c,
                                                    const SceneGrid* __restrict__ scenes,
                                                    const uint32_t* __restrict__ offs,
                                                    uint32_t* __restrict__ items,
                                                    uint4* __restrict__ desc,
                                                    uint32_t* __restrict__ nitems) {
    const uint32_t col = blockIdx.x * blockDim.x + threadIdx.x;
    if (col == 0) publish_chunks(nitems, offs[c.ncols]);
    if (col >= c.ncols) return;
    const uint32_t scene = scene_of_col(scenes, c.nscenes, col);
    const SceneGrid g = scenes[scene];
    const uint32_t first = g.cell_base + (col - g.col_base) * (uint32_t)g.nz;
    column_items(make_uint2(cs[first], cs[first + (uint32_t)g.nz]), scene, g, col, offs[col],
                 items, desc);
}

// Every column may end with a part-filled chunk, and every chunk holds a particle.  (Without the
// second bound the launches of a sparse scene follow its columns: 97,000 particles on 755 x 755 of
// them step 476 -> 302 us, 10,600 369 -> 192.)
uint32_t max_chunks(uint32_t n, const StepConsts& c) {
    return std::min((n + 63u) / 64u + c.ncols, n);
}

// ---------------------------------------------------------------------------
// Launch shapes of the walks: words per LDS segment x wavefronts per workgroup.  Every
// wavefront works on its own chunk and the waves of a workgroup never synchronise, but for the
// team walks (the "_split" shapes, below), which give a chunk a workgroup.
// ---------------------------------------------------------------------------

// ---------------------------------------------------------------------------
// density: rho_i = m_i W(0) + sum_{j != i} m_j W(r_ij)   (compute_density,
// src/sph_engine.cpp:370-383).  The self pair is one of the words' bits (d = 0), so the sum
// runs over the set bits, self included.  Stores the neighbour words of every chunk and the
// force walk's neighbour rows of every particle.
// ---------------------------------------------------------------------------
// A value computed here, before whatever follows.  Pinning each pair's sum keeps it ahead of
// the next step's refill branch, so the row it used is dead when the row after it is requested
// and the two share registers; left to the compiler, the sums sink past the branches and the
// loop copies a row set at its back edge.  Measured on the 1M dam break: density walk 0.429
// -> 0.423 ms; at 10,000 particles the split shapes' walks (both pinned) 1-2 % faster.  The
// ping-pong force walk keeps its sums unpinned: its steps wait on row gathers, and pinned sums
// (which hold the next request back until they are formed) took it 0.581 -> 0.594 ms.
__device__ __forceinline__ float pinned(float x) {
    asm volatile("" : "+v"(x));
    return x;
}

// Neighbour positions are requested two steps ahead, in three rotating register sets.
template <bool kCut, int kSeg>
__device__ __forceinline__ float density_bits(BitWalk<kSeg>& bw, uint32_t steps,
                                              const uint32_t* __restrict__ lmask,
                                              const uint32_t* __restrict__ lwj0, uint32_t lane,
                                              const float4* __restrict__ spm, const float4& pi,
                                              const StepConsts& c, float acc) {
    if (steps == 0) return acc;
    const float hh = 0.5f * c.inv_h;
    float4 q0 = row_at(spm, bw.template next<4>(lmask, lwj0, lane));
    float4 q1 = row_at(spm, bw.template next<4>(lmask, lwj0, lane));
    uint32_t t = 0;
    for (; t + 3 <= steps; t += 3) {
        const float4 q2 = row_at(spm, bw.template next<4>(lmask, lwj0, lane));
        acc = pinned(density_pair<kCut>(pi, q0, c, hh, acc));
        q0 = row_at(spm, bw.template next<4>(lmask, lwj0, lane));
        acc = pinned(density_pair<kCut>(pi, q1, c, hh, acc));
        q1 = row_at(spm, bw.template next<4>(lmask, lwj0, lane));
        acc = pinned(density_pair<kCut>(pi, q2, c, hh, acc));
    }
    if (t < steps) acc = density_pair<kCut>(pi, q0, c, hh, acc);
    if (t + 1 < steps) acc = density_pair<kCut>(pi, q1, c, hh, acc);
    return acc;
}

// The same walk with kAhead rows in flight, for the split shapes, whose wavefronts are few
// (below one per SIMD at 10,000 particles) and hide little of each other's gather latency.
// Rows rotate through kAhead + 1 register sets, each refilled right after its row is used;
// the pairs are summed in the same order as above.  Measured at 10,000 particles: each walk
// ~1 us (2 %) faster than with two rows in flight, so the small-scene walks are not bound by
// gather latency either.
template <bool kCut, int kSeg, int kAhead>
__device__ __forceinline__ float density_bits_deep(BitWalk<kSeg>& bw, uint32_t steps,
                                                   const uint32_t* __restrict__ lmask,
                                                   const uint32_t* __restrict__ lwj0,
                                                   uint32_t lane, const float4* __restrict__ spm,
                                                   const float4& pi, const StepConsts& c,
                                                   float acc) {
    if (steps == 0) return acc;
    const float hh = 0.5f * c.inv_h;
    float4 q[kAhead + 1];
#pragma unroll
    for (int k = 0; k < kAhead; ++k) q[k] = row_at(spm, bw.template next<4>(lmask, lwj0, lane));
    uint32_t t = 0;
    for (; t + kAhead + 1 <= steps; t += kAhead + 1) {
#pragma unroll
        for (int k = 0; k <= kAhead; ++k) {
            q[(k + kAhead) % (kAhead + 1)] = row_at(spm, bw.template next<4>(lmask, lwj0, lane));
            acc = pinned(density_pair<kCut>(pi, q[k], c, hh, acc));
        }
    }
#pragma unroll
    for (int k = 0; k < kAhead; ++k)
        if (t + k < steps) acc = density_pair<kCut>(pi, q[k], c, hh, acc);
    return acc;
}

// Rows in flight per wavefront in the split shapes' walks, and per lane in the ping-pong force
// walk.  Measured on the 1M dam break (pp16_waves4): 2 rows 0.578 ms, 3 rows 0.574, 4 rows
// 0.566, 5 rows 0.561, 6 rows 0.560 (158 VGPRs: three wavefronts per SIMD where the LDS allows
// four), 8 rows 0.624 (two wavefronts per SIMD): the force walk is bound by its gathers'
// latency more than by wavefronts in flight.
constexpr int kDeepAhead = 5;
constexpr int kPPAhead = 6;

// The ping-pong shapes' walk, which goes on across calls: on entry and on return the rows of
// the lane's next two pairs are in flight in q0 and q1, and a call takes exactly `steps` bits
// and sums exactly `steps` pairs (the two in flight at a part's end are summed by the caller).
template <bool kCut, int kW>
__device__ __forceinline__ float density_run(BitWalk<kW>& bw, float4& q0, float4& q1,
                                             uint32_t steps, const uint32_t* __restrict__ lmask,
                                             const uint32_t* __restrict__ lwj0, uint32_t lane,
                                             const float4* __restrict__ spm, const float4& pi,
                                             const StepConsts& c, float acc) {
    const float hh = 0.5f * c.inv_h;
    uint32_t t = 0;
    for (; t + 3 <= steps; t += 3) {
        const float4 q2 = row_at(spm, bw.template next<4>(lmask, lwj0, lane));
        acc = pinned(density_pair<kCut>(pi, q0, c, hh, acc));
        q0 = row_at(spm, bw.template next<4>(lmask, lwj0, lane));
        acc = pinned(density_pair<kCut>(pi, q1, c, hh, acc));
        q1 = row_at(spm, bw.template next<4>(lmask, lwj0, lane));
        acc = pinned(density_pair<kCut>(pi, q2, c, hh, acc));
    }
    for (; t < steps; ++t) {
        const float4 q2 = row_at(spm, bw.template next<4>(lmask, lwj0, lane));
        acc = density_pair<kCut>(pi, q0, c, hh, acc);
        q0 = q1;
        q1 = q2;
    }
    return acc;
}

// The sum over a chunk's words by one wavefront, a segment of kSeg - 1 of them at a time; the
// parts' sums are folded as (p0 + p1) + p2.
template <class Shape, bool kCut, bool kFar>
__device__ __forceinline__ float density_segments(
    const Chunk& ch, const WordTable& wt, bool tab, MfmaFilter& mf, const float4* __restrict__ spm,
    const uint2* __restrict__ sq, const uint32_t* __restrict__ cs, const StepConsts& c, uint2 qi,
    bool active, const float4& pi, uint32_t* __restrict__ gm, uint32_t* __restrict__ gj,
    uint32_t* __restrict__ lmask, uint32_t* __restrict__ lwj0, uint32_t lane) {
    constexpr int kSeg = Shape::seg;
    Cursor cu;
    if (!tab) cursor_begin(cu, ch, cs, c);
    float total = 0.0f, cur = 0.0f;
    int cur_part = 0;
    int seg_base = wt.first;
    int ti = 0;  // next table entry
    for (;;) {
        SegLane sl;
        int seg_part;
        const int nw =
            tab ? phase1_table<kSeg, kFar>(wt, ti, sq, c, lmask, lwj0, gm, gj, lane, sl, seg_part,
                                           mf)
                : phase1_segment<kSeg, true, kFar>(cu, ch, sq, cs, c, qi, active, lmask, lwj0, lane,
                                                   sl, seg_part, &mf);
        if (nw == 0) break;
        for (; cur_part < seg_part; ++cur_part) {
            total = cur_part == 0 ? cur : total + cur;
            cur = 0.0f;
        }
        wave_sync();
        if (!tab) store_words(c.max_words, seg_base, nw, lmask, lwj0, gm, gj, lane);
        BitWalk<kSeg> bw;
        bw.begin(sl.nonempty, lmask, lwj0, lane);
        const uint32_t steps = wave_max(sl.count);
        cur = density_bits<kCut>(bw, steps, lmask, lwj0, lane, spm, pi, c, cur);
        seg_base += nw;
        wave_sync();
        if (tab ? ti >= wt.n : cu.done) break;
    }
    for (; cur_part < kParts; ++cur_part) {
        total = cur_part == 0 ? cur : total + cur;
        cur = 0.0f;
    }
    return total;
}

// Density pass over one chunk by one wavefront.  As many wavefronts per SIMD as the LDS
// allows (six with 24-word segments): the walk is VALU-bound (a few spills outside the walk
// loops).  The ping-pong shapes aim at what their LDS
// allows (6 with two 12-word buffers, 4 with two 16-word ones).
template <class Shape, bool kCut, bool kFar>
__global__ __launch_bounds__(Shape::threads) __attribute__((amdgpu_waves_per_eu(Shape::density_waves, 8))) void k_density_walk(
    const uint32_t* __restrict__ items, const uint4* __restrict__ desc,
    const uint32_t* __restrict__ nitems,
    const float4* __restrict__ spm, const uint2* __restrict__ sq, float4* __restrict__ svr,
    ForceRow* __restrict__ rows, const uint32_t* __restrict__ skey,
    const uint32_t* __restrict__ cs, StepConsts c, const SceneGrid* __restrict__ scenes,
    uint32_t* __restrict__ gmask, uint32_t* __restrict__ gwj0, uint32_t* __restrict__ gnw,
    uint32_t* __restrict__ gpart) {
    constexpr int kSeg = Shape::seg;
    constexpr int kLds = Shape::lds_words;
    __shared__ uint32_t lmask_all[Shape::waves][kLds * 64];
    __shared__ uint32_t lwj0_all[Shape::waves][kLds];
    const uint32_t wave = uni(threadIdx.x >> 6);
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t* lmask = lmask_all[wave];
    uint32_t* lwj0 = lwj0_all[wave];
    const uint32_t item = xcd_unit(uni(nitems[0]), Shape::waves, wave);
    if (item == ~0u) return;
    Chunk ch;
    uint32_t s;
    bool active;
    float4 pi;
    if (!load_chunk(item, items, desc, nitems, skey, spm, c, scenes, lane, ch, s, active, pi)) return;
    const uint2 qi = active ? sq[s] : make_uint2(0u, 0u);
    MfmaFilter mf;
    mfma_filter_begin(mf, ch, qi, active, lane, c.qneg);
    WordTable wt;
    static_assert(kLds * 64 >= kTableWords, "the word table is built in the mask buffer");
    const bool tab = word_table_build(wt, ch, cs, -1, lane, lmask);
    init_sentinel<kLds>(lmask, lwj0, lane, c);
    uint32_t* const gm = gmask + (size_t)item * c.max_words * 64;
    uint32_t* const gj = gwj0 + (size_t)item * c.max_words;
    if (lane == 0) {
        gpart[item] = pack_parts(wt.ps1, wt.ps2);
        gnw[item] = (uint32_t)wt.total;
    }
    float total = 0.0f;
    if constexpr (Shape::pp) {
        Cursor cu;
        if (!tab) cursor_begin(cu, ch, cs, c);
        // per-part running sum `cur`, parts folded into `total` as (p0 + p1) + p2
        float cur = 0.0f;
        int cur_part = 0;
        int seg_base = wt.first;
        int ti = 0;  // next table entry
        // Segments are made in the newer buffer.  A segment of the part being walked joins
        // the walk at once; one of the next part waits there until every lane is through the
        // current part (the parts' sums are folded between them, in the same order as in
        // every other shape).
        uint32_t* const lm_new = lmask + kSeg * 64;
        uint32_t* const lj_new = lwj0 + kSeg;
        const float hh = 0.5f * c.inv_h;
        PingPong<kSeg> pp;
        pp.init(c.pad_slot);
        float4 q0, q1;  // rows of the next two pairs, requested (within a phase)
        bool more = true, pend = false;  // pend: the newer buffer holds the next part's segment
        int pend_part = 0, pend_nw = 0, walk_part = -1;
        for (;;) {
            if (pp.nw_new == 0 && !pend && more) {
                SegLane sl;
                int seg_part;
                const int nw =
                    tab ? phase1_table<kSeg, kFar>(wt, ti, sq, c, lm_new, lj_new, gm, gj, lane, sl,
                                                   seg_part, mf)
                        : phase1_segment<kSeg, true, kFar>(cu, ch, sq, cs, c, qi, active, lm_new,
                                                           lj_new, lane, sl, seg_part, &mf);
                if (nw == 0) {
                    more = false;
                } else {
                    wave_sync();
                    if (!tab) store_words(c.max_words, seg_base, nw, lm_new, lj_new, gm, gj, lane);
                    seg_base += nw;
                    if (tab ? ti >= wt.n : cu.done) more = false;
                    if (walk_part < 0 || seg_part == walk_part) {
                        if (walk_part < 0) {  // the walk's first segment
                            for (; cur_part < seg_part; ++cur_part) {
                                total = cur_part == 0 ? cur : total + cur;
                                cur = 0.0f;
                            }
                            walk_part = seg_part;
                        }
                        pp.add_newer(sl, nw, lmask, lwj0, lane, c.pad_slot);
                    } else {
                        pend = true;
                        pend_part = seg_part;
                        pend_nw = nw;
                    }
                }
            }
            // A phase: walk until every lane is through the older buffer (or, with nothing to
            // overlap, through all it holds).  Its read-ahead starts at the phase's start and its
            // last two rows are summed at its end, in walk order; nothing stays in flight while
            // the next segment is made.
            const bool overlap = pp.nw_new != 0;
            if (!overlap && walk_part < 0) break;  // no segment at all
            const uint32_t need = overlap ? pp.older_steps() : pp.all_steps();
            if (need != 0) {
                q0 = row_at(spm, pp.bw.template next<4>(lmask, lwj0, lane));
                q1 = row_at(spm, pp.bw.template next<4>(lmask, lwj0, lane));
                pp.walked(2);
                const uint32_t steps = need > 2u ? need - 2u : 0u;
                cur = density_run<kCut>(pp.bw, q0, q1, steps, lmask, lwj0, lane, spm, pi, c, cur);
                pp.walked(steps);
                cur = density_pair<kCut>(pi, q0, c, hh, cur);
                cur = density_pair<kCut>(pi, q1, c, hh, cur);
            }
            if (overlap) {
                pp.shift_down(lmask, lwj0, lane);
                continue;
            }
            if (!pend) break;
            for (; cur_part < pend_part; ++cur_part) {
                total = cur_part == 0 ? cur : total + cur;
                cur = 0.0f;
            }
            walk_part = pend_part;
            pend = false;
            pp.add_held(pend_nw, lmask, lwj0, lane, c.pad_slot);
        }
        for (; cur_part < kParts; ++cur_part) {
            total = cur_part == 0 ? cur : total + cur;
            cur = 0.0f;
        }
    } else {
        total = density_segments<Shape, kCut, kFar>(ch, wt, tab, mf, spm, sq, cs, c, qi, active,
                                                    pi, gm, gj, lmask, lwj0, lane);
    }
    if (active) density_epilogue(total, pi, s, c, svr, rows);
}

// ---------------------------------------------------------------------------
// Team walks (the "_split" shapes): one workgroup per chunk, for scenes whose chunks are fewer
// than the GPU's SIMDs hold (10,000 particles: 178 chunks for 1,024 SIMDs), where a step
// takes as long as its longest chunk.  A lone wavefront issues a dependent instruction every
// 6 to 8 cycles, so a chunk's time is its instruction count: kTeam wavefronts share the candidate
// words of the chunk (about 1,000 cycles each), then each part's pairs are walked by one
// wavefront (a part's sum runs in candidate order) and the first one finishes the
// particles from LDS.  Against three independent wavefronts per chunk and a finishing launch
// per walk: a step of 2,145 particles 108 -> 96 us, of 10,000 126 -> 110 us, ten steps of 33,000
// 1.36 -> 1.27 ms.  Pile-ups, whose chunks have too many words for the table, gain less (400 a
// cell: 3,000 particles 249 -> 220 us, 50,000 850 -> 824, 100,000 1483 -> 1210) and lose around
// 20,000 to 30,000, where the independent wavefronts filled every CU once (590 -> 604, 708 -> 752;
// at 1,500 a cell 1424 -> 1627).  Eight wavefronts a team are slower from 10,000 particles on (two
// workgroups a CU).
// ---------------------------------------------------------------------------
constexpr int kTeam = 4;

// In a pile-up (the reference formulas throw a block into its box's corners) a chunk has hundreds
// of words and one column holds nearly all of them: a team then has work for one wavefront and
// holds the LDS of four.  Where most chunks of the walk before were such, and enough to fill the
// GPU, every wavefront of the teams walks a chunk of its own.  Corner pile-ups, a step: 80,000
// particles 5.49 -> 5.38 ms, 100,000 7.37 -> 7.03, 120,000 9.69 -> 8.26, 160,000 16.06 -> 12.98;
// 66,000 are level, and piles over several columns are faster by teams (100,000 particles at 1,500
// a cell 4.7 ms against 6.9).
__device__ __forceinline__ bool lone_chunk(const WordTable& wt) {
    return wt.total > kMaxWords && 8 * max(wt.ps1, wt.ps2 - wt.ps1) > 7 * wt.total;
}

// LDS rows of the team's words: a part's words in groups of kSeg - 1, each group followed by
// the sentinel word of its walk.
__device__ __forceinline__ int team_rows(int words, int group) {
    return words + (words + group - 1) / group;
}

// The part's sum over the words of its cursor or its own table: chunks of more than kTableWords
// words, one wavefront per part.
template <class Shape, bool kCut, bool kFar>
__device__ __forceinline__ float density_part_alone(
    const Chunk& ch, MfmaFilter& mf, int part, const float4* __restrict__ spm,
    const uint2* __restrict__ sq, const uint32_t* __restrict__ cs, const StepConsts& c, uint2 qi,
    bool active, const float4& pi, uint32_t* __restrict__ gm, uint32_t* __restrict__ gj,
    uint32_t* __restrict__ lmask, uint32_t* __restrict__ lwj0, uint32_t* __restrict__ scratch,
    uint32_t lane) {
    constexpr int kSeg = Shape::seg;
    WordTable wt;
    const bool tab = word_table_build(wt, ch, cs, part, lane, scratch);
    init_sentinel<kSeg>(lmask, lwj0, lane, c);
    Cursor cu;
    if (!tab) cursor_begin(cu, ch, cs, c, 0, part);
    float cur = 0.0f;
    int seg_base = wt.first;
    int ti = 0;
    for (;;) {
        SegLane sl;
        int seg_part;
        const int nw = tab ? phase1_table<kSeg, kFar>(wt, ti, sq, c, lmask, lwj0, gm, gj, lane, sl,
                                                seg_part, mf)
                           : phase1_segment<kSeg, true, kFar>(cu, ch, sq, cs, c, qi, active, lmask,
                                                              lwj0, lane, sl, seg_part, &mf);
        if (nw == 0) break;
        wave_sync();
        if (!tab) store_words(c.max_words, seg_base, nw, lmask, lwj0, gm, gj, lane);
        BitWalk<kSeg> bw;
        bw.begin(sl.nonempty, lmask, lwj0, lane);
        cur = density_bits_deep<kCut, kSeg, kDeepAhead>(bw, wave_max(sl.count), lmask, lwj0, lane,
                                                        spm, pi, c, cur);
        seg_base += nw;
        wave_sync();
        if (tab ? ti >= wt.n : cu.done) break;
    }
    return cur;
}

template <class Shape, bool kCut, bool kFar>
__global__ __launch_bounds__(64 * kTeam) void k_density_team(
    const uint32_t* __restrict__ items, const uint4* __restrict__ desc,
    const uint32_t* __restrict__ nitems, const float4* __restrict__ spm,
    const uint2* __restrict__ sq, float4* __restrict__ svr, ForceRow* __restrict__ rows,
    const uint32_t* __restrict__ skey, const uint32_t* __restrict__ cs, StepConsts c,
    const SceneGrid* __restrict__ scenes, uint32_t* __restrict__ gmask,
    uint32_t* __restrict__ gwj0, uint32_t* __restrict__ gnw, uint32_t* __restrict__ gpart,
    uint32_t* __restrict__ lone_chunks) {
    constexpr int kSeg = Shape::seg;
    constexpr int kGroup = kSeg - 1;
    constexpr int kRows = kTableWords + kTableWords / kGroup + kParts;
    static_assert(kTeam >= kParts && kRows >= kTeam * kSeg, "a walk's words per wavefront");
    __shared__ uint32_t lmask[kRows * 64];
    __shared__ uint32_t lwj0[kRows];
    __shared__ uint32_t scratch[kTeam][kTableWords];
    __shared__ float lsum[kParts][64];
    const uint32_t wave = uni(threadIdx.x >> 6);
    const uint32_t lane = threadIdx.x & 63u;
    const bool lone = uni(nitems[2]) != 0u;
    const uint32_t item = xcd_unit(uni(nitems[0]), lone ? kTeam : 1u, lone ? wave : 0u);
    if (item == ~0u) return;
    Chunk ch;
    uint32_t s;
    bool active;
    float4 pi;
    if (!load_chunk(item, items, desc, nitems, skey, spm, c, scenes, lane, ch, s, active, pi)) return;
    const uint2 qi = active ? sq[s] : make_uint2(0u, 0u);
    MfmaFilter mf;
    mfma_filter_begin(mf, ch, qi, active, lane, c.qneg);
    WordTable wt;
    const bool tab = word_table_build(wt, ch, cs, -1, lane, scratch[wave]);
    uint32_t* const gm = gmask + (size_t)item * c.max_words * 64;
    uint32_t* const gj = gwj0 + (size_t)item * c.max_words;
    if ((lone || wave == 0) && lane == 0) {
        gpart[item] = pack_parts(wt.ps1, wt.ps2);
        gnw[item] = (uint32_t)wt.total;
        if (lone_chunk(wt)) atomicAdd(lone_chunks, 1u);
    }
    if (lone) {
        uint32_t* const lm = lmask + wave * kSeg * 64;
        uint32_t* const lj = lwj0 + wave * kSeg;
        init_sentinel<kSeg>(lm, lj, lane, c);
        const float total = density_segments<Shape, kCut, kFar>(
            ch, wt, tab, mf, spm, sq, cs, c, qi, active, pi, gm, gj, lm, lj, lane);
        if (active) density_epilogue(total, pi, s, c, svr, rows);
        return;
    }
    float cur = 0.0f;
    if (tab) {
        const int n0 = wt.ps1, n1 = wt.ps2 - wt.ps1, n2 = wt.total - wt.ps2;
        const int r1 = team_rows(n0, kGroup), r2 = r1 + team_rows(n1, kGroup);
        auto row_of = [&](int w) {
            const int l = w < wt.ps1 ? w : w < wt.ps2 ? w - wt.ps1 : w - wt.ps2;
            return (w < wt.ps1 ? 0 : w < wt.ps2 ? r1 : r2) + l + l / kGroup;
        };
        table_words<kTeam, true, kFar>(wt, mf, sq, (int)wave, wt.total, c.qneg, lane,
                                 [&](uint32_t word, int w, uint32_t j0) {
                                     const int r = row_of(w);
                                     lmask[r * 64 + lane] = word;
                                     if (lane == 0) lwj0[r] = j0;
                                     if (w < (int)c.max_words)
                                         __builtin_nontemporal_store(
                                             word, &gm[(size_t)w * 64 + lane]);
                                 });
        if (wave == kTeam - 1) {
            constexpr uint32_t kSlot = (1u << 27) - 1u;
            const int stored = min(wt.total, (int)c.max_words);
            if ((int)lane < stored) gj[lane] = wt.e0 & kSlot;
            if ((int)lane + 64 < stored) gj[lane + 64u] = wt.e1 & kSlot;
        }
        __syncthreads();
        if (wave < kParts) {
            const int n = wave == 0 ? n0 : wave == 1 ? n1 : n2;
            const int r0 = wave == 0 ? 0 : wave == 1 ? r1 : r2;
            for (int g = 0; g * kGroup < n; ++g) {
                const int m = min(kGroup, n - g * kGroup);
                uint32_t* const lm = lmask + (r0 + g * kSeg) * 64;
                uint32_t* const lj = lwj0 + r0 + g * kSeg;
                SegLane sl = {0u, 0u};
#pragma unroll 4
                for (int w = 0; w < m; ++w) {
                    const uint32_t word = lm[w * 64 + lane];
                    sl.nonempty |= min(word, 1u) << w;
                    sl.count += (uint32_t)__builtin_popcount(word);
                }
                lm[m * 64 + lane] = 0x80000000u;
                if (lane == 0) lj[m] = c.pad_slot;
                wave_sync();
                BitWalk<kSeg> bw;
                bw.begin(sl.nonempty, lm, lj, lane, 1u << m);
                cur = density_bits_deep<kCut, kSeg, kDeepAhead>(bw, wave_max(sl.count), lm, lj,
                                                                lane, spm, pi, c, cur);
            }
        }
    } else if (wave < kParts) {
        cur = density_part_alone<Shape, kCut, kFar>(ch, mf, (int)wave, spm, sq, cs, c, qi, active,
                                                    pi, gm, gj, lmask + wave * kSeg * 64,
                                                    lwj0 + wave * kSeg, scratch[wave], lane);
    }
    if (wave < kParts) lsum[wave][lane] = cur;
    __syncthreads();
    if (wave == 0 && active)
        density_epilogue((lsum[0][lane] + lsum[1][lane]) + lsum[2][lane], pi, s, c, svr, rows);
}

// ---------------------------------------------------------------------------
// forces + leapfrog + wall clamp
//   F_p = -sum_{j != i, |r| >= 1e-6} m_j (P_i + P_j) / (2 rho_j) gradW(r_ij)
//   F_v =  sum_{j != i} (m_j / rho_j) mu (v_j - v_i) laplacianW(r_ij)
//   a_i = (F_p + F_v + g m_i) / m_i        (rho_i instead of m_i: consistent formulation)
// (src/sph_engine.cpp:390-443), integrate_leapfrog (:290-310) and
// apply_boundary_conditions (src/particle.cpp:122-153).
// ---------------------------------------------------------------------------
// The wavefront runs its largest lane count; rows are requested two neighbours ahead, in
// three rotating register sets (a gather from L2 takes several hundred cycles, one step of
// pair arithmetic about a hundred).
template <int kSeg, bool kCut>
__device__ __forceinline__ void force_bits(BitWalk<kSeg>& bw, uint32_t steps,
                                           const uint32_t* __restrict__ lmask,
                                           const uint32_t* __restrict__ lwj0, uint32_t lane,
                                           const ForceRow* __restrict__ rows, const float4& pi,
                                           const float3& vi, float p_quarter, const StepConsts& c,
                                           ForceSums& f, uint32_t& cnt) {
    if (steps == 0) return;
    static_assert(sizeof(ForceRow) == 32, "rows are 32-byte blocks");
    uint32_t o = bw.template next<5>(lmask, lwj0, lane);
    float4 a0 = row_at(rows, o).a, b0 = row_at(rows, o).b;
    o = bw.template next<5>(lmask, lwj0, lane);
    float4 a1 = row_at(rows, o).a, b1 = row_at(rows, o).b;
    uint32_t t = 0;
    for (; t + 3 <= steps; t += 3) {
        o = bw.template next<5>(lmask, lwj0, lane);
        const float4 a2 = row_at(rows, o).a, b2 = row_at(rows, o).b;
        f.template add<kCut>(pi, vi, p_quarter, a0, b0, c, cnt);
        o = bw.template next<5>(lmask, lwj0, lane);
        a0 = row_at(rows, o).a;
        b0 = row_at(rows, o).b;
        f.template add<kCut>(pi, vi, p_quarter, a1, b1, c, cnt);
        o = bw.template next<5>(lmask, lwj0, lane);
        a1 = row_at(rows, o).a;
        b1 = row_at(rows, o).b;
        f.template add<kCut>(pi, vi, p_quarter, a2, b2, c, cnt);
    }
    if (t < steps) f.template add<kCut>(pi, vi, p_quarter, a0, b0, c, cnt);
    if (t + 1 < steps) f.template add<kCut>(pi, vi, p_quarter, a1, b1, c, cnt);
}

// force_bits with kAhead rows in flight (the split shapes; see density_bits_deep).
template <int kSeg, bool kCut, int kAhead>
__device__ __forceinline__ void force_bits_deep(BitWalk<kSeg>& bw, uint32_t steps,
                                                const uint32_t* __restrict__ lmask,
                                                const uint32_t* __restrict__ lwj0, uint32_t lane,
                                                const ForceRow* __restrict__ rows,
                                                const float4& pi, const float3& vi,
                                                float p_quarter, const StepConsts& c,
                                                ForceSums& f, uint32_t& cnt) {
    if (steps == 0) return;
    float4 a[kAhead + 1], b[kAhead + 1];
#pragma unroll
    for (int k = 0; k < kAhead; ++k) {
        const uint32_t o = bw.template next<5>(lmask, lwj0, lane);
        a[k] = row_at(rows, o).a;
        b[k] = row_at(rows, o).b;
    }
    uint32_t t = 0;
    for (; t + kAhead + 1 <= steps; t += kAhead + 1) {
#pragma unroll
        for (int k = 0; k <= kAhead; ++k) {
            const uint32_t o = bw.template next<5>(lmask, lwj0, lane);
            a[(k + kAhead) % (kAhead + 1)] = row_at(rows, o).a;
            b[(k + kAhead) % (kAhead + 1)] = row_at(rows, o).b;
            f.template add<kCut>(pi, vi, p_quarter, a[k], b[k], c, cnt);
            f.pin(cnt);
        }
    }
#pragma unroll
    for (int k = 0; k < kAhead; ++k)
        if (t + k < steps) f.template add<kCut>(pi, vi, p_quarter, a[k], b[k], c, cnt);
}

// force_bits for the ping-pong shapes: the walk goes on across calls with the rows of the
// lane's next kAhead pairs in flight (slots 0 .. kAhead - 1 on entry and on return, slot
// kAhead free); a call takes exactly `steps` bits and adds exactly `steps` pairs.  Each step
// requests into the free slot and sums the oldest, so over a block of kAhead + 1 steps the
// slots come back to their order and no row set is copied between blocks.
template <int kW, bool kCut, int kAhead>
__device__ __forceinline__ void force_run_n(BitWalk<kW>& bw, float4 (&a)[kAhead + 1],
                                            float4 (&b)[kAhead + 1], uint32_t steps,
                                            const uint32_t* __restrict__ lmask,
                                            const uint32_t* __restrict__ lwj0, uint32_t lane,
                                            const ForceRow* __restrict__ rows, const float4& pi,
                                            const float3& vi, float p_quarter,
                                            const StepConsts& c, ForceSums& f, uint32_t& cnt) {
    uint32_t t = 0;
    for (; t + kAhead + 1 <= steps; t += kAhead + 1) {
#pragma unroll
        for (int k = 0; k <= kAhead; ++k) {
            const uint32_t o = bw.template next<5>(lmask, lwj0, lane);
            a[(k + kAhead) % (kAhead + 1)] = row_at(rows, o).a;
            b[(k + kAhead) % (kAhead + 1)] = row_at(rows, o).b;
            f.template add<kCut>(pi, vi, p_quarter, a[k], b[k], c, cnt);
        }
    }
    for (; t < steps; ++t) {
        const uint32_t o = bw.template next<5>(lmask, lwj0, lane);
        a[kAhead] = row_at(rows, o).a;
        b[kAhead] = row_at(rows, o).b;
        f.template add<kCut>(pi, vi, p_quarter, a[0], b[0], c, cnt);
#pragma unroll
        for (int k = 0; k < kAhead; ++k) {
            a[k] = a[k + 1];
            b[k] = b[k + 1];
        }
    }
}

// Folds the sums of finished parts into the running total, which starts at +0:
// ((0 + part 0) + part 1) + part 2.  Closing `n` parts at once adds `f` for the first and
// +0 for each further (empty) one, as the team walk does.  The single-wavefront
// walk keeps the total in LDS (`t`, six rows of 64 lanes): six more live registers would cost
// it a wavefront per SIMD.
__device__ __forceinline__ void fold_parts(float* __restrict__ t, uint32_t lane, ForceSums& f,
                                           int n) {
    if (n <= 0) return;
    const float v[6] = {f.fp.x, f.fp.y, f.fp.z, f.fv.x, f.fv.y, f.fv.z};
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        float x = t[k * 64 + lane] + v[k];
        if (n >= 2) x = x + 0.0f;
        t[k * 64 + lane] = x;
    }
    f = ForceSums();
}

// The same fold with the running total in registers (shapes whose occupancy LDS limits).
__device__ __forceinline__ void fold_parts_reg(float (&t)[6], ForceSums& f, int n) {
    if (n <= 0) return;
    const float v[6] = {f.fp.x, f.fp.y, f.fp.z, f.fv.x, f.fv.y, f.fv.z};
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        float x = t[k] + v[k];
        if (n >= 2) x = x + 0.0f;
        t[k] = x;
    }
    f = ForceSums();
}

// The running total as it is kept in LDS or in registers.
__device__ __forceinline__ void clear_parts(float* __restrict__ t, uint32_t lane) {
#pragma unroll
    for (int k = 0; k < 6; ++k) t[k * 64 + lane] = 0.0f;
}
__device__ __forceinline__ ForceSums total_sums(const float* __restrict__ t, uint32_t lane) {
    ForceSums f;
    f.fp = make_float3(t[0 * 64 + lane], t[1 * 64 + lane], t[2 * 64 + lane]);
    f.fv = make_float3(t[3 * 64 + lane], t[4 * 64 + lane], t[5 * 64 + lane]);
    return f;
}
__device__ __forceinline__ ForceSums total_sums(const float (&t)[6]) {
    ForceSums f;
    f.fp = make_float3(t[0], t[1], t[2]);
    f.fv = make_float3(t[3], t[4], t[5]);
    return f;
}

// Loads a segment of `nw` stored words (from stored word `base` on) into LDS, with the lane's
// summary.  All loads are issued before the first is used (a loop over nw would wait for each
// load of its remainder in turn); slots past nw re-read word nw - 1 and are dropped.  The words
// are read once: nontemporal loads keep them from evicting the neighbour rows from L2.
template <int kSeg>
__device__ __forceinline__ void load_words(const uint32_t* __restrict__ gmask,
                                           const uint32_t* __restrict__ gwj0, size_t base, int nw,
                                           uint32_t* __restrict__ lmask,
                                           uint32_t* __restrict__ lwj0, uint32_t lane,
                                           SegLane& sl) {
    uint32_t wv[kSeg - 1];
    sl.nonempty = 0;
    sl.count = 0;
#pragma unroll
    for (int w = 0; w < kSeg - 1; ++w)
        wv[w] = __builtin_nontemporal_load(&gmask[(base + (size_t)min(w, nw - 1)) * 64 + lane]);
#pragma unroll
    for (int w = 0; w < kSeg - 1; ++w) {
        if (w < nw) {
            lmask[w * 64 + lane] = wv[w];
            sl.nonempty |= (wv[w] != 0u ? 1u : 0u) << w;
            sl.count += (uint32_t)__builtin_popcount(wv[w]);
        }
    }
    if ((int)lane < nw) lwj0[lane] = gwj0[base + lane];
}

// The sums over a chunk's words by one wavefront, a segment at a time: stored words, or the words
// formed again.  The parts' running total is in registers (kRegTot) or in `ltot`, six rows of 64
// lanes in LDS.
template <class Shape, bool kCut, bool kFar, bool kRegTot>
__device__ __forceinline__ ForceSums force_segments(
    const Chunk& ch, bool stored, int total_words, uint32_t pstarts, size_t first_word,
    const uint2* __restrict__ sq, const ForceRow* __restrict__ rows,
    const uint32_t* __restrict__ cs, const StepConsts& c, uint2 qi, bool active, const float4& pi,
    const float3& vi, float p_quarter, const uint32_t* __restrict__ gmask,
    const uint32_t* __restrict__ gwj0, uint32_t* __restrict__ lmask, uint32_t* __restrict__ lwj0,
    float* __restrict__ ltot, uint32_t lane, uint32_t& cnt) {
    constexpr int kSeg = Shape::seg;
    float rtot[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (!kRegTot) clear_parts(ltot, lane);
    ForceSums f;
    int cur_part = 0;
    Cursor cu;
    if (!stored) cursor_begin(cu, ch, cs, c);
    int seg_base = 0;
    for (;;) {
        int nw, seg_part;
        SegLane sl;
        if (stored) {
            if (seg_base >= total_words) break;
            seg_part = part_of_word(seg_base, pstarts);
            const int pend = part_word_end(pstarts, seg_part, total_words);
            nw = min(kSeg - 1, pend - seg_base);
            load_words<kSeg>(gmask, gwj0, first_word + seg_base, nw, lmask, lwj0, lane, sl);
        } else {
            nw = phase1_segment<kSeg, false, kFar>(cu, ch, sq, cs, c, qi, active, lmask, lwj0, lane,
                                                   sl, seg_part);
            if (nw == 0) break;
        }
        if (kRegTot)
            fold_parts_reg(rtot, f, seg_part - cur_part);
        else
            fold_parts(ltot, lane, f, seg_part - cur_part);
        cur_part = seg_part;
        wave_sync();
        BitWalk<kSeg> bw;
        bw.begin(sl.nonempty, lmask, lwj0, lane);
        force_bits<kSeg, kCut>(bw, wave_max(sl.count), lmask, lwj0, lane, rows, pi, vi, p_quarter,
                               c, f, cnt);
        seg_base += nw;
        wave_sync();
        if (!stored && cu.done) break;
    }
    if (kRegTot)
        fold_parts_reg(rtot, f, kParts - cur_part);
    else
        fold_parts(ltot, lane, f, kParts - cur_part);
    return kRegTot ? total_sums(rtot) : total_sums(ltot, lane);
}

// Force pass over one chunk by one wavefront.  Shapes of 24 words and more keep
// the parts' running total in registers: their LDS, not their registers, limits occupancy,
// and the 1.5 KB per wavefront it frees lets the 28-word shape run 5 wavefronts per SIMD.
template <class Shape, bool kCut, bool kFar>
__global__ __launch_bounds__(Shape::threads) __attribute__((amdgpu_waves_per_eu(Shape::force_waves)))
void k_force_walk(
    const uint32_t* __restrict__ items, const uint4* __restrict__ desc,
    const uint32_t* __restrict__ nitems,
    const float4* __restrict__ spm, const uint2* __restrict__ sq,
    const float4* __restrict__ svr, const ForceRow* __restrict__ rows,
    const uint32_t* __restrict__ skey, const uint32_t* __restrict__ sid,
    const uint32_t* __restrict__ cs, StepConsts c, const SceneGrid* __restrict__ scenes,
    const uint32_t* __restrict__ gmask, const uint32_t* __restrict__ gwj0,
    const uint32_t* __restrict__ gnw, const uint32_t* __restrict__ gpart,
    const float* __restrict__ dt_dev, float dt_arg,
    float4* __restrict__ pm,
    float4* __restrict__ vel, float4* __restrict__ acc_out, float* __restrict__ rho_out,
    float* __restrict__ prs_out, unsigned long long* __restrict__ stats) {
    constexpr int kSeg = Shape::seg;
    constexpr int kLds = Shape::lds_words;
    __shared__ uint32_t lmask_all[Shape::waves][kLds * 64];
    __shared__ uint32_t lwj0_all[Shape::waves][kLds];
    const uint32_t wave = uni(threadIdx.x >> 6);
    const uint32_t lane = threadIdx.x & 63u;
    constexpr bool kRegTot = !Shape::pp && kSeg >= 24;
    constexpr bool kLdsTot = !kRegTot;
    __shared__ float ltot_all[kLdsTot ? Shape::waves : 1][kLdsTot ? 6 * 64 : 1];
    uint32_t* lmask = lmask_all[wave];
    uint32_t* lwj0 = lwj0_all[wave];
    float* ltot = ltot_all[kLdsTot ? wave : 0];
    const uint32_t item = xcd_unit(uni(nitems[0]), Shape::waves, wave);
    if (item == ~0u) return;
    Chunk ch;
    uint32_t s;
    bool active;
    float4 pi;
    const int total_words = (int)uni(gnw[item]);
    const bool stored = total_words <= (int)c.max_words;
    const uint32_t pstarts = uni(gpart[item]);
    // (the whole chunk description serves the re-test alone)
    uint2 qi = make_uint2(0u, 0u);
    if (stored) {
        load_targets(item, items, desc, spm, c, lane, ch, s, active, pi);
    } else {
        if (!load_chunk(item, items, desc, nitems, skey, spm, c, scenes, lane, ch, s, active, pi))
            return;
        if (active) qi = sq[s];
    }
    init_sentinel<kLds>(lmask, lwj0, lane, c);
    const float4 vr = active ? svr[s] : make_float4(0.f, 0.f, 0.f, 1.f);
    const float3 vi = make_float3(vr.x, vr.y, vr.z);
    const float rho_i = vr.w;
    const float P_i = c.k_gas * (rho_i - c.rho0);
    const float p_quarter = 0.25f * P_i;
    ForceSums tot;
    uint32_t cnt = 0;  // neighbours
    if constexpr (Shape::pp) {
        clear_parts(ltot, lane);
        ForceSums f;
        int cur_part = 0;
        Cursor cu;
        if (!stored) cursor_begin(cu, ch, cs, c);
        int seg_base = 0;
        const int words_end = total_words;
        // As in the density walk: segments are loaded into the newer buffer; one of the part
        // being walked joins the walk at once, one of the next part waits until every lane
        // is through the current part.
        uint32_t* const lm_new = lmask + kSeg * 64;
        uint32_t* const lj_new = lwj0 + kSeg;
        PingPong<kSeg> pp;
        pp.init(c.pad_slot);
        float4 a[kPPAhead + 1], b[kPPAhead + 1];  // rows requested ahead (within a phase)
        bool more = true, pend = false;  // pend: the newer buffer holds the next part's segment
        int pend_part = 0, pend_nw = 0, walk_part = -1;
        auto request_ahead = [&]() {
#pragma unroll
            for (int k = 0; k < kPPAhead; ++k) {
                const uint32_t o = pp.bw.template next<5>(lmask, lwj0, lane);
                a[k] = row_at(rows, o).a;
                b[k] = row_at(rows, o).b;
            }
            pp.walked(kPPAhead);
        };
        for (;;) {
            if (pp.nw_new == 0 && !pend && more) {
                int nw = 0, seg_part = 0;
                SegLane sl = {0u, 0u};
                if (stored) {
                    if (seg_base < words_end) {
                        seg_part = part_of_word(seg_base, pstarts);
                        const int pend_end = part_word_end(pstarts, seg_part, total_words);
                        nw = min(kSeg - 1, pend_end - seg_base);
                        load_words<kSeg>(gmask, gwj0, (size_t)item * c.max_words + seg_base, nw,
                                         lm_new, lj_new, lane, sl);
                        seg_base += nw;
                    }
                    if (seg_base >= words_end) more = false;
                } else {
                    nw = phase1_segment<kSeg, false, kFar>(cu, ch, sq, cs, c, qi, active, lm_new,
                                                           lj_new, lane, sl, seg_part);
                    if (cu.done) more = false;
                }
                if (nw == 0) {
                    more = false;
                } else {
                    wave_sync();
                    if (walk_part < 0 || seg_part == walk_part) {
                        if (walk_part < 0) {  // the walk's first segment
                            fold_parts(ltot, lane, f, seg_part - cur_part);
                            cur_part = seg_part;
                            walk_part = seg_part;
                        }
                        pp.add_newer(sl, nw, lmask, lwj0, lane, c.pad_slot);
                    } else {
                        pend = true;
                        pend_part = seg_part;
                        pend_nw = nw;
                    }
                }
            }
            // A phase, as in the density walk: nothing stays in flight between phases.
            const bool overlap = pp.nw_new != 0;
            if (!overlap && walk_part < 0) break;  // no segment at all
            const uint32_t need = overlap ? pp.older_steps() : pp.all_steps();
            if (need != 0) {
                request_ahead();
                const uint32_t steps = need > kPPAhead ? need - kPPAhead : 0u;
                force_run_n<kLds, kCut, kPPAhead>(pp.bw, a, b, steps, lmask, lwj0, lane, rows,
                                                  pi, vi, p_quarter, c, f, cnt);
                pp.walked(steps);
#pragma unroll
                for (int k = 0; k < kPPAhead; ++k)
                    f.template add<kCut>(pi, vi, p_quarter, a[k], b[k], c, cnt);
            }
            if (overlap) {
                pp.shift_down(lmask, lwj0, lane);
                continue;
            }
            if (!pend) break;
            fold_parts(ltot, lane, f, pend_part - cur_part);
            cur_part = pend_part;
            walk_part = pend_part;
            pend = false;
            pp.add_held(pend_nw, lmask, lwj0, lane, c.pad_slot);
        }
        fold_parts(ltot, lane, f, kParts - cur_part);
        tot = total_sums(ltot, lane);
    } else {
        tot = force_segments<Shape, kCut, kFar, kRegTot>(
            ch, stored, total_words, pstarts, (size_t)item * c.max_words, sq, rows, cs, c, qi,
            active, pi, vi, p_quarter, gmask, gwj0, lmask, lwj0, ltot, lane, cnt);
    }
    if (stats) add_nbr_stats(cnt, stats, lane);
    if (!active) return;
    force_epilogue(tot, pi, vi, rho_i, P_i, s, scenes[ch.scene], c, sid, dt_dev, dt_arg, pm, vel,
                   acc_out, rho_out, prs_out);
}

// Force pass over one chunk by a team of two wavefronts (see k_density_team): the first walks
// part 0, the second parts 1 and 2 (the ring two columns out is nearly always empty); the first
// folds the parts' sums from LDS and finishes the particles.  Two teams in one workgroup of four
// wavefronts were slower (33,000 particles: 41 -> 46 us a walk: coarser workgroups spread the
// chunks less evenly over the CUs), a wavefront per part no faster.
constexpr int kForceTeam = 2;

template <class Shape, bool kCut, bool kFar>
__global__ __launch_bounds__(64 * kForceTeam) void k_force_team(
    const uint32_t* __restrict__ items, const uint4* __restrict__ desc,
    const uint32_t* __restrict__ nitems, const float4* __restrict__ spm,
    const uint2* __restrict__ sq, const float4* __restrict__ svr,
    const ForceRow* __restrict__ rows, const uint32_t* __restrict__ skey,
    const uint32_t* __restrict__ sid, const uint32_t* __restrict__ cs, StepConsts c,
    const SceneGrid* __restrict__ scenes, const uint32_t* __restrict__ gmask,
    const uint32_t* __restrict__ gwj0, const uint32_t* __restrict__ gnw,
    const uint32_t* __restrict__ gpart, const float* __restrict__ dt_dev, float dt_arg,
    float4* __restrict__ pm, float4* __restrict__ vel, float4* __restrict__ acc_out,
    float* __restrict__ rho_out, float* __restrict__ prs_out,
    unsigned long long* __restrict__ stats) {
    constexpr int kSeg = Shape::seg;
    __shared__ uint32_t lmask_all[kForceTeam][kSeg * 64];
    __shared__ uint32_t lwj0_all[kForceTeam][kSeg];
    __shared__ float lsum[kParts][6][64];
    __shared__ uint32_t lcnt[64];
    const uint32_t wave = uni(threadIdx.x >> 6);
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t* lmask = lmask_all[wave];
    uint32_t* lwj0 = lwj0_all[wave];
    const bool lone = uni(nitems[2]) != 0u;
    const uint32_t item = xcd_unit(uni(nitems[0]), lone ? kForceTeam : 1u, lone ? wave : 0u);
    if (item == ~0u) return;
    Chunk ch;
    uint32_t s;
    bool active;
    float4 pi;
    const int total_words = (int)uni(gnw[item]);
    const bool stored = total_words <= (int)c.max_words;
    const uint32_t pstarts = uni(gpart[item]);
    // (the whole chunk description serves the re-test alone)
    uint2 qi = make_uint2(0u, 0u);
    if (stored) {
        load_targets(item, items, desc, spm, c, lane, ch, s, active, pi);
    } else {
        if (!load_chunk(item, items, desc, nitems, skey, spm, c, scenes, lane, ch, s, active, pi))
            return;
        if (active) qi = sq[s];
    }
    init_sentinel<kSeg>(lmask, lwj0, lane, c);
    const float4 vr = active ? svr[s] : make_float4(0.f, 0.f, 0.f, 1.f);
    const float3 vi = make_float3(vr.x, vr.y, vr.z);
    const float rho_i = vr.w;
    const float P_i = c.k_gas * (rho_i - c.rho0);
    const float p_quarter = 0.25f * P_i;
    uint32_t cnt = 0;
    if (lone) {
        const ForceSums tot = force_segments<Shape, kCut, kFar, true>(
            ch, stored, total_words, pstarts, (size_t)item * c.max_words, sq, rows, cs, c, qi,
            active, pi, vi, p_quarter, gmask, gwj0, lmask, lwj0, nullptr, lane, cnt);
        if (stats) add_nbr_stats(cnt, stats, lane);
        if (active)
            force_epilogue(tot, pi, vi, rho_i, P_i, s, scenes[ch.scene], c, sid, dt_dev, dt_arg, pm,
                           vel, acc_out, rho_out, prs_out);
        return;
    }
    for (int part = (int)wave; part < (wave == 0 ? 1 : kParts); ++part) {
        ForceSums f;
        Cursor cu;
        int w = 0, end = 0;
        if (stored) {
            w = part_word_start(pstarts, part);
            end = part_word_end(pstarts, part, total_words);
        } else {
            cursor_begin(cu, ch, cs, c, 0, part);
        }
        for (;;) {
            int nw, seg_part;
            SegLane sl;
            if (stored) {
                if (w >= end) break;
                nw = min(kSeg - 1, end - w);
                load_words<kSeg>(gmask, gwj0, (size_t)item * c.max_words + w, nw, lmask, lwj0,
                                 lane, sl);
                w += nw;
            } else {
                nw = phase1_segment<kSeg, false, kFar>(cu, ch, sq, cs, c, qi, active, lmask, lwj0,
                                                       lane, sl, seg_part);
                if (nw == 0) break;
            }
            wave_sync();
            BitWalk<kSeg> bw;
            bw.begin(sl.nonempty, lmask, lwj0, lane);
            force_bits_deep<kSeg, kCut, kDeepAhead>(bw, wave_max(sl.count), lmask, lwj0, lane,
                                                    rows, pi, vi, p_quarter, c, f, cnt);
            wave_sync();
        }
        const float v[6] = {f.fp.x, f.fp.y, f.fp.z, f.fv.x, f.fv.y, f.fv.z};
#pragma unroll
        for (int k = 0; k < 6; ++k) lsum[part][k][lane] = v[k];
    }
    if (wave == 1) lcnt[lane] = cnt;
    __syncthreads();
    if (wave != 0) return;
    if (stats) add_nbr_stats(cnt + lcnt[lane], stats, lane);
    if (!active) return;
    // ((0 + part 0) + part 1) + part 2, as the single-wavefront walk folds them
    float t[6];
#pragma unroll
    for (int k = 0; k < 6; ++k)
        t[k] = ((0.0f + lsum[0][k][lane]) + lsum[1][k][lane]) + lsum[2][k][lane];
    ForceSums tot;
    tot.fp = make_float3(t[0], t[1], t[2]);
    tot.fv = make_float3(t[3], t[4], t[5]);
    force_epilogue(tot, pi, vi, rho_i, P_i, s, scenes[ch.scene], c, sid, dt_dev, dt_arg, pm, vel,
                   acc_out, rho_out, prs_out);
}

// Particles with a non-finite coordinate (dense index G) have no neighbour, not even
// themselves: rho = m W(0), a = (0, g, 0); they are integrated and clamped like the rest.
__device__ __forceinline__ void nonfinite_particle(const StepTail& t, const float4& pi,
                                                   const float4& vi, uint32_t id, float dt,
                                                   const StepConsts& c,
                                                   const SceneGrid* __restrict__ scenes) {
    const float rho_i = pi.w * c.w0;
    const float P_i = c.k_gas * (rho_i - c.rho0);
    const float3 a = final_accel(make_float3(0.f, 0.f, 0.f), make_float3(0.f, 0.f, 0.f), pi.w,
                                 rho_i, c);
    float3 v = make_float3(vi.x, vi.y, vi.z);
    float4 p = pi;
    const SceneGrid& g = scenes[scene_of_particle(scenes, c.nscenes, id)];
    integrate_clamp(p, v, a, dt, c, g.lo, g.hi);
    t.pm[id] = p;
    t.vel[id] = make_float4(v.x, v.y, v.z, 0.0f);
    t.acc[id] = make_float4(a.x, a.y, a.z, 0.0f);
    t.rho[id] = rho_i;
    t.prs[id] = P_i;
}

// The non-finite bin's step: it holds the sorted slots [cs[G], n); workgroup `b` of `nb` takes
// every nb-th run of 256.  Workgroup 0 also advances the simulation time (time_dev, if given) by dt.
__device__ __forceinline__ void nonfinite_particles(const StepTail& t,
                                                    const uint32_t* __restrict__ cs,
                                                    const StepConsts& c,
                                                    const SceneGrid* __restrict__ scenes,
                                                    uint32_t b, uint32_t nb) {
    const float dt = t.dt_dev ? *t.dt_dev : t.dt;
    if (t.time_dev && b == 0 && threadIdx.x == 0) *t.time_dev = *t.time_dev + dt;
    for (uint32_t s = cs[c.G] + b * blockDim.x + threadIdx.x; s < t.n; s += nb * blockDim.x)
        nonfinite_particle(t, t.spm[s], t.svr[s], t.sid[s], dt, c, scenes);
}

__global__ __launch_bounds__(256) void k_nonfinite_step(StepTail t, const uint32_t* __restrict__ cs,
                                                        StepConsts c,
                                                        const SceneGrid* __restrict__ scenes) {
    nonfinite_particles(t, cs, c, scenes, blockIdx.x, gridDim.x);
}

// Grids of at most this many (x, y) columns get their chunk list from one launch: every
// workgroup counts the chunks of all columns and scans the counts in LDS, then writes the
// items of its own 256 columns.  Workgroups from `fill_blocks` on do the non-finite bin's step
// (kTail).
constexpr uint32_t kChunkListLocal = 8192;

// Sorted slots [x, y) of column `col` (its cells are consecutive, z fastest).  kOne: a
// one-scene grid, whose geometry g0 is loaded once instead of looked up per column.
template <bool kOne>
__device__ __forceinline__ uint2 column_slots(const uint32_t* __restrict__ cs,
                                              const SceneGrid* __restrict__ scenes,
                                              const StepConsts& c, const SceneGrid& g0,
                                              uint32_t col) {
    const SceneGrid& g = kOne ? g0 : scenes[scene_of_col(scenes, c.nscenes, col)];
    const uint32_t nz = (uint32_t)g.nz;
    const uint32_t first = g.cell_base + (col - g.col_base) * nz;
    return make_uint2(cs[first], cs[first + nz]);
}

template <bool kTail>
__global__ __launch_bounds__(256) void k_chunk_list(const uint32_t* __restrict__ cs, StepConsts c,
                                                    const SceneGrid* __restrict__ scenes,
                                                    uint32_t* __restrict__ items,
                                                    uint4* __restrict__ desc,
                                                    uint32_t* __restrict__ nitems,
                                                    uint32_t fill_blocks, StepTail t) {
    if (blockIdx.x >= fill_blocks) {
        if constexpr (kTail)
            nonfinite_particles(t, cs, c, scenes, blockIdx.x - fill_blocks,
                                gridDim.x - fill_blocks);
        return;
    }
    constexpr int kPer = (int)(kChunkListLocal / 256u);
    __shared__ uint32_t off[kChunkListLocal];
    __shared__ uint32_t lw[4];
    const uint32_t ncols = c.ncols;
    // thread k counts the columns [k*per, (k+1)*per), all its loads in flight at once
    const uint32_t per = (ncols + 255u) / 256u;
    const uint32_t beg = threadIdx.x * per;
    const SceneGrid g0 = scenes[0];
    const bool one = c.nscenes == 1;
    uint32_t cnt[kPer];
    uint32_t sum = 0;
    if (one) {
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            const uint32_t col = beg + (uint32_t)j;
            const uint2 r = (uint32_t)j < per && col < ncols
                                ? column_slots<true>(cs, scenes, c, g0, col)
                                : make_uint2(0u, 0u);
            cnt[j] = (r.y - r.x + 63u) / 64u;
            sum += cnt[j];
        }
    } else {
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            const uint32_t col = beg + (uint32_t)j;
            const uint2 r = (uint32_t)j < per && col < ncols
                                ? column_slots<false>(cs, scenes, c, g0, col)
                                : make_uint2(0u, 0u);
            cnt[j] = (r.y - r.x + 63u) / 64u;
            sum += cnt[j];
        }
    }
    uint32_t total;
    uint32_t run = block_exclusive_scan_256(sum, lw, &total);
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const uint32_t col = beg + (uint32_t)j;
        if ((uint32_t)j < per && col < ncols) off[col] = run;
        run += cnt[j];
    }
    __syncthreads();
    if (blockIdx.x == 0 && threadIdx.x == 0) publish_chunks(nitems, total);
    const uint32_t col = blockIdx.x * 256u + threadIdx.x;
    if (col >= ncols) return;
    const uint32_t scene = one ? 0u : scene_of_col(scenes, c.nscenes, col);
    const SceneGrid g = one ? g0 : scenes[scene];
    column_items(column_slots<true>(cs, scenes, c, g, col), scene, g, col, off[col], items, desc);
}

// Small scenes: rows in sorted order (see k_gather_cells); with kTail, the thread that gathers
// a particle of the non-finite bin also steps it (nobody else reads its home rows).
template <bool kTail>
__global__ __launch_bounds__(256) void k_gather_rows(const float4* pm, const float4* vel,
                                                     const uint32_t* __restrict__ sid, uint32_t n,
                                                     double qscale, uint2* __restrict__ sq,
                                                     float4* __restrict__ spm,
                                                     float4* __restrict__ svr,
                                                     const uint32_t* __restrict__ cs, StepConsts c,
                                                     const SceneGrid* __restrict__ scenes,
                                                     StepTail t) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t id = s < n ? sid[s] : 0u;
    float4 p = pm[id], v = vel[id];
    if constexpr (kTail) {
        if (s == 0u && t.time_dev) *t.time_dev = *t.time_dev + (t.dt_dev ? *t.dt_dev : t.dt);
    }
    if (s >= n) return;
    v.w = 0.0f;
    spm[s] = p;
    svr[s] = v;
    const uint32_t qx = quantize(p.x, qscale), qy = quantize(p.y, qscale);
    sq[s] = make_uint2((qx & 0xffffu) | (qy << 16), quantize(p.z, qscale));
    if constexpr (kTail) {
        if (s >= cs[c.G]) nonfinite_particle(t, p, v, id, t.dt_dev ? *t.dt_dev : t.dt, c, scenes);
    }
}

hipError_t launch_gather_rows(const float4* pm, const float4* vel, const uint32_t* sid, uint32_t n,
                              double qscale, uint2* sq, float4* spm, float4* svr,
                              const uint32_t* cell_start, const StepConsts& c,
                              const SceneGrid* scenes, const StepTail* tail, hipStream_t st) {
    const dim3 grid((n + 255) / 256);
    if (tail)
        hipLaunchKernelGGL(k_gather_rows<true>, grid, dim3(256), 0, st, pm, vel, sid, n, qscale,
                           sq, spm, svr, cell_start, c, scenes, *tail);
    else
        hipLaunchKernelGGL(k_gather_rows<false>, grid, dim3(256), 0, st, pm, vel, sid, n, qscale,
                           sq, spm, svr, cell_start, c, scenes, StepTail{});
    return hipGetLastError();
}

hipError_t launch_chunks(const uint32_t* cell_start, const StepConsts& c, const SceneGrid* scenes,
                         uint32_t* cnt_scratch, uint32_t* scan_scratch, uint32_t* items,
                         uint4* desc, uint32_t* nitems, const StepTail* tail, hipStream_t st) {
    // the non-finite bin holds at most n particles; its start is read on the device
    const uint32_t tail_blocks =
        tail ? std::max<uint32_t>(1u, std::min<uint32_t>((tail->n + 255u) / 256u, 64u)) : 0u;
    if (c.ncols <= kChunkListLocal) {
        const uint32_t fill_blocks = std::max<uint32_t>(1u, (c.ncols + 255u) / 256u);
        if (tail)
            hipLaunchKernelGGL(k_chunk_list<true>, dim3(fill_blocks + tail_blocks), dim3(256), 0,
                               st, cell_start, c, scenes, items, desc, nitems, fill_blocks, *tail);
        else
            hipLaunchKernelGGL(k_chunk_list<false>, dim3(fill_blocks), dim3(256), 0, st,
                               cell_start, c, scenes, items, desc, nitems, fill_blocks, StepTail{});
        return hipGetLastError();
    }
    hipLaunchKernelGGL(k_chunk_count, dim3((c.ncols + 1 + 255) / 256), dim3(256), 0, st,
                       cell_start, c, scenes, cnt_scratch);
    hipError_t e = scan_exclusive(cnt_scratch, c.ncols + 1, scan_scratch, st);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_chunk_fill, dim3((c.ncols + 255) / 256 + 1), dim3(256), 0, st, cell_start,
                       c, scenes, cnt_scratch, items, desc, nitems);
    if (tail)
        hipLaunchKernelGGL(k_nonfinite_step, dim3(tail_blocks), dim3(256), 0, st, *tail,
                           cell_start, c, scenes);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// neighbour lists for parity checks: the production phase-1 test, expanded to CSR over
// caller ids in reference order.  pass 0 counts, pass 1 writes.
// ---------------------------------------------------------------------------
template <class Shape>
__global__ __launch_bounds__(Shape::threads) void k_nbr_lists(
    const uint32_t* __restrict__ items, const uint4* __restrict__ desc,
    const uint32_t* __restrict__ nitems,
    const float4* __restrict__ spm, const uint2* __restrict__ sq,
    const uint32_t* __restrict__ skey, const uint32_t* __restrict__ sid,
    const uint32_t* __restrict__ cs, StepConsts c, const SceneGrid* __restrict__ scenes,
    int pass,
    uint32_t* __restrict__ cnt_by_id, const int64_t* __restrict__ offs_by_id,
    int64_t* __restrict__ idx) {
    constexpr int kSeg = Shape::seg;
    __shared__ uint32_t lmask_all[Shape::waves][kSeg * 64];
    __shared__ uint32_t lwj0_all[Shape::waves][kSeg];
    const uint32_t wave = uni(threadIdx.x >> 6);
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t* lmask = lmask_all[wave];
    uint32_t* lwj0 = lwj0_all[wave];
    Chunk ch;
    uint32_t s;
    bool active;
    float4 pi;
    const uint32_t wid = xcd_unit(uni(nitems[0]), Shape::waves, wave);
    if (wid == ~0u) return;
    if (!load_chunk(wid, items, desc, nitems, skey, spm, c, scenes,
                    lane, ch, s, active, pi))
        return;
    const uint2 qi = active ? sq[s] : make_uint2(0u, 0u);
    Cursor cu;
    cursor_begin(cu, ch, cs, c, 1);
    uint32_t cnt = 0;
    int64_t o = (pass == 1 && active) ? offs_by_id[sid[s]] : 0;
    for (;;) {
        SegLane sl;
        int part;  // always 0 in the reference order
        const int nw =
            phase1_segment<kSeg, false, false>(cu, ch, sq, cs, c, qi, active, lmask, lwj0, lane, sl,
                                               part);
        if (nw == 0) break;
        wave_sync();
        BitWalk<kSeg> bw;
        bw.begin(sl.nonempty, lmask, lwj0, lane);
        for (uint32_t t = 0; t < sl.count; ++t) {
            const uint32_t j = bw.next(lmask, lwj0, lane);
            const float4 q = spm[j];
            if (dist2_exact(pi.x, pi.y, pi.z, q.x, q.y, q.z) <= c.r2) {
                if (pass == 1) idx[o++] = sid[j];
                ++cnt;
            }
        }
        wave_sync();
        if (cu.done) break;
    }
    if (pass == 0 && active) cnt_by_id[sid[s]] = cnt;
}

// ---------------------------------------------------------------------------
// launch shape table (index = WalkTuning value)
// ---------------------------------------------------------------------------
using Shape0 = WalkShape<16, 4>;
using Shape1 = WalkShape<32, 4>;
using Shape2 = WalkShape<28, 4>;
using Shape3 = WalkShape<32, 1>;
using Shape4 = WalkShape<24, 4>;
using Shape5 = WalkShape<12, 4, true>;
using Shape6 = WalkShape<16, 4, true>;

const char* walk_shape_name(int v) {
    switch (v) {
        case 0: return "seg16_waves4";
        case 1: return "seg32_waves4";
        case 2: return "seg28_waves4";
        case 3: return "seg32_waves1";
        case 4: return "seg24_waves4";
        case 5: return "seg16_waves4_split";
        case 6: return "seg32_waves4_split";
        case 7: return "pp12_waves4";
        case 8: return "pp16_waves4";
        default: return "?";
    }
}

// Workgroups are dispatched round-robin over the 8 XCDs, each with its own L2.  The grid is
// padded to a multiple of 8 and sized for the most chunks a step can have (the host does not
// know the count, which the chunk list leaves on the device); each XCD walks one contiguous
// eighth of the chunks that exist (xcd_unit), whose candidate columns overlap.  A team (split)
// shape runs one workgroup per chunk.
static uint32_t grid_for(uint32_t chunks, uint32_t per_block) {
    const uint32_t blocks = (chunks + per_block - 1) / per_block;
    return (blocks + kXcds - 1) / kXcds * kXcds;
}

// CALL sees the shape as type S; TEAM, for the split shapes, likewise.
#define SPHK_DISPATCH_SHAPE(v, CALL, TEAM)  \
    switch (v) {                            \
        case 0: { using S = Shape0; CALL; break; } \
        case 1: { using S = Shape1; CALL; break; } \
        case 2: { using S = Shape2; CALL; break; } \
        case 3: { using S = Shape3; CALL; break; } \
        case 5: { using S = Shape0; TEAM; break; } \
        case 6: { using S = Shape1; TEAM; break; } \
        case 7: { using S = Shape5; CALL; break; } \
        case 8: { using S = Shape6; CALL; break; } \
        default: { using S = Shape4; CALL; break; } \
    }

hipError_t launch_density_walk(const WalkBuffers& wb, const float4* spm, const uint2* sq,
                               float4* svr,
                               ForceRow* rows, const uint32_t* skey,
                               const uint32_t* cell_start, uint32_t n,
                               const StepConsts& c, const SceneGrid* scenes, int shape,
                               hipStream_t st) {
    if (n == 0) return hipSuccess;
    const uint32_t chunks = max_chunks(n, c);
#define SPHK_DENSITY_KERNEL(KERNEL, CUT, FAR, PER_BLOCK, THREADS, ...)                         \
    hipLaunchKernelGGL((KERNEL<S, CUT, FAR>), dim3(grid_for(chunks, PER_BLOCK)), dim3(THREADS), \
                       0, st, wb.items, wb.desc, wb.nitems, spm, sq, svr, rows, skey, cell_start, \
                       c, scenes, wb.mask, wb.wj0, wb.nwords, wb.pstarts, ##__VA_ARGS__)
#define SPHK_DENSITY_LAUNCH(CUT, FAR)                                                         \
    SPHK_DISPATCH_SHAPE(                                                                      \
        shape, SPHK_DENSITY_KERNEL(k_density_walk, CUT, FAR, S::waves, S::threads),           \
        SPHK_DENSITY_KERNEL(k_density_team, CUT, FAR, 1, 64 * kTeam, wb.nitems + 1))
    if (c.cut) {
        if (c.far) {
            SPHK_DENSITY_LAUNCH(true, true);
        } else {
            SPHK_DENSITY_LAUNCH(true, false);
        }
    } else {
        if (c.far) {
            SPHK_DENSITY_LAUNCH(false, true);
        } else {
            SPHK_DENSITY_LAUNCH(false, false);
        }
    }
#undef SPHK_DENSITY_LAUNCH
#undef SPHK_DENSITY_KERNEL
    return hipGetLastError();
}

hipError_t launch_force_walk(const WalkBuffers& wb, const float4* spm, const uint2* sq,
                             const float4* svr,
                             const ForceRow* rows, const uint32_t* skey,
                             const uint32_t* sid,
                             const uint32_t* cell_start, uint32_t n, const StepConsts& c,
                             const SceneGrid* scenes, const float* dt_dev, float dt, float4* pm,
                             float4* vel, float4* acc, float* rho, float* prs, int shape,
                             unsigned long long* nbr_stats, hipStream_t st) {
    if (n == 0) return hipSuccess;
    const uint32_t chunks = max_chunks(n, c);
#define SPHK_FORCE_KERNEL(KERNEL, CUT, FAR, PER_BLOCK, THREADS)                               \
    hipLaunchKernelGGL((KERNEL<S, CUT, FAR>), dim3(grid_for(chunks, PER_BLOCK)), dim3(THREADS), \
                       0, st, wb.items, wb.desc, wb.nitems, spm, sq, svr, rows, skey, sid,     \
                       cell_start, c, scenes, wb.mask, wb.wj0, wb.nwords, wb.pstarts, dt_dev,  \
                       dt, pm, vel, acc, rho, prs, nbr_stats)
#define SPHK_FORCE_LAUNCH(CUT, FAR)                                                           \
    SPHK_DISPATCH_SHAPE(shape,                                                                \
                        SPHK_FORCE_KERNEL(k_force_walk, CUT, FAR, S::waves, S::threads),      \
                        SPHK_FORCE_KERNEL(k_force_team, CUT, FAR, 1, 64 * kForceTeam))
    if (c.cut) {
        if (c.far) {
            SPHK_FORCE_LAUNCH(true, true);
        } else {
            SPHK_FORCE_LAUNCH(true, false);
        }
    } else {
        if (c.far) {
            SPHK_FORCE_LAUNCH(false, true);
        } else {
            SPHK_FORCE_LAUNCH(false, false);
        }
    }
#undef SPHK_FORCE_LAUNCH
#undef SPHK_FORCE_KERNEL
    return hipGetLastError();
}

hipError_t launch_nbr_lists(const WalkBuffers& wb, const float4* spm, const uint2* sq,
                            const uint32_t* skey,
                            const uint32_t* sid, const uint32_t* cell_start, uint32_t n,
                            const StepConsts& c, const SceneGrid* scenes, int pass,
                            uint32_t* count_by_id, const int64_t* offsets_by_id, int64_t* idx,
                            int shape, hipStream_t st) {
    if (n == 0) return hipSuccess;
    const uint32_t chunks = max_chunks(n, c);
    // one wavefront per chunk in every shape (a split shape lists with its unsplit twin, a
    // ping-pong shape with the single-buffer shape of the same LDS size)
    const int base = shape == 5 ? 0 : shape == 6 ? 1 : shape == 7 ? 4 : shape == 8 ? 1 : shape;
#define SPHK_LISTS_LAUNCH                                                                     \
    hipLaunchKernelGGL(k_nbr_lists<S>, dim3(grid_for(chunks, S::waves)), dim3(S::threads), 0, \
                       st, wb.items, wb.desc, wb.nitems, spm, sq, skey, sid, cell_start, c,   \
                       scenes, pass, count_by_id, offsets_by_id, idx)
    SPHK_DISPATCH_SHAPE(base, SPHK_LISTS_LAUNCH, SPHK_LISTS_LAUNCH);
#undef SPHK_LISTS_LAUNCH
    return hipGetLastError();
}

}  // namespace sphk
