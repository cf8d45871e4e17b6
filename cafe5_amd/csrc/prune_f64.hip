// prune_f64.hip -- FP64 pruning on the matrix cores, in the reference's
// summation order (inference_prune / compute_node_probability,
// src/core.cpp:134-145, src/probability.cpp:175-330): the PLAIN64 and BATCHED64
// paths and the FP64 recompute of the reduced paths.
//
// v_mfma_f64_16x16x4f64 adds its four products to the accumulator one after
// another, each as a fused multiply-add, in ascending k (checked bit for bit
// against a chain of fma() on the device, subnormal values included).  MFMA j
// of k-tile kt contracts the sizes x = 16 kt + 4 j + g of lane group g, so
// every sum runs over x = 0, 1, 2, ... as matrix::multiply's does
// (matrix_cache.cpp:50-56), and a node's factors multiply in the children's
// order (probability.cpp:208-217, 222-231).
//
// Lane l = 16 g + f of a wave holds, for 16-row tile t of a vector, the sizes
// 16 t + 4 r + g (r = 0..3) of family f: the D layout of the instruction, and
// the B layout of the next contraction, so a node's output is its parent's
// input as stored.  A workgroup of W waves carries FB blocks of 16 families of
// one bucket at one parameter point through the tree; a wave takes chunks of
// NTW row tiles (chunk = wave, wave + W, ...), and each matrix fragment it loads
// feeds the MFMAs of all FB blocks.
//
// What bounds it: an FP64 MFMA takes a SIMD's FP64 unit for 64 cycles, so the
// steps' address arithmetic is kept on the scalar side; at 201 rows a step is
// 13,300 cycles of MFMAs on the SIMD with four of the thirteen waves and about
// 7,000 of barrier and step start.  10,000 families of 34 taxa at bound 200
// take 0.96 ms (27 TF/s of 71 the library's products reach), against 37.2 ms
// one family per wave with the lanes over rows; 250 families of 12 taxa 0.06
// against 2.2 ms.  Over shared subtrees the 10,000 take 0.37 ms in four launches,
// the last 0.20 at 33% of the matrix cores' cycles (26 TF/s), the small first ones
// at 9 to 25%; at 501 rows, 1.6 M family-likelihoods of 100 taxa keep them busy 73%.
#include "prune_common.h"

namespace cafe {

typedef double d4 __attribute__((ext_vector_type(4)));

// A key this far (relatively) below the best product cannot be the best key:
// the logarithms' rounding is 1e-13 at most over FP64's range.
constexpr double kNearBest = 1.0 - 1e-9;

// Most waves of a workgroup: sixteen leave 128 VGPRs per wave, eight 256.
template <int NTW, int FB> struct F64Waves { static constexpr int v = NTW * FB > 2 || FB > 1 ? 8 : 16; };

// q, kept as a scalar base: the compiler would otherwise fold the lane offset
// into per-lane 64-bit addresses, and an FP64 matrix instruction holds the
// SIMD's vector unit for its 64 cycles, so every vector instruction beside
// the matrix ones waits for one of another wave.
typedef const __attribute__((address_space(1))) double* Gptr;
__device__ __forceinline__ Gptr uniform(const double* q)
{
    Gptr r = (Gptr)q;
    asm("" : "+s"(r));
    return r;
}

// *(q + byte offset): one 32-bit lane offset serves all loads (hidden here, or
// its 64-bit form would be kept across the loop).
__device__ __forceinline__ double at(Gptr q, unsigned off)
{
    asm volatile("" : "+v"(off));
    return *(Gptr)((const __attribute__((address_space(1))) char*)q + off);
}

// Partial vectors in LDS or in global scratch (typed by address space: a
// generic pointer would make their accesses flat ones).
template <bool LDSP> struct Partials { typedef __attribute__((address_space(1))) d4* ptr; };
template <> struct Partials<true> { typedef __attribute__((address_space(3))) d4* ptr; };

template <int NTW, int FB, bool LDSP, bool STAGED>
__global__ __launch_bounds__((64 * F64Waves<NTW, FB>::v)) void k_prune_f64(PruneParams p)
{
    constexpr int FW = 16 * FB;   // families per tile
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int W = __builtin_amdgcn_readfirstlane((int)(blockDim.x >> 6));
    const int fl = lane & 15;
    const int g = lane >> 4;
    const int Np = p.Np;
    const int slot_tiles = p.slot_tiles;
    extern __shared__ __align__(32) unsigned char s_dyn[];
    typedef __attribute__((address_space(3))) unsigned char* Lds;
    const Lds lds = (Lds)s_dyn;
    __attribute__((address_space(3))) double* s_a = (__attribute__((address_space(3))) double*)lds;   // [W][FW] per-wave maxima
    __attribute__((address_space(3))) double* s_b = s_a + W * FW;                                     // [W][FW]
    // [leaf][FW] byte offsets of the tile's leaf columns (where they fit)
    __attribute__((address_space(3))) unsigned* s_cnt = (__attribute__((address_space(3))) unsigned*)(s_b + W * FW);
    typedef typename Partials<LDSP>::ptr Frag;
    Frag frag;
    if constexpr (LDSP) frag = (Frag)(lds + f64_meta_bytes(W, FB, p.n_leaves, STAGED));
    else frag = (Frag)p.scratch + (long long)blockIdx.x * p.n_slots * slot_tiles * FB * 64;
    unsigned a_lane[4];   // byte offsets of the lane's entries (fl, 4 j + g) of a 16 x 16 block
#pragma unroll
    for (int j = 0; j < 4; ++j) a_lane[j] = 8u * ((4 * j + g) * Np + fl);
    // a block past the matrix's last column: zeros (Np >= N + 16)
    const int zero_col = Np - kTile;

    // each XCD (workgroup b runs on b % 8) takes one contiguous range of the
    // list, whose neighbours share their matrices in its L2
    const int n_tiles = *as_const(p.n_tiles_dev);
    if (n_tiles <= p.skip_tiles) return;   // launch_f64_levels'
    const int groups = (gridDim.x % 8 == 0) ? 8 : 1;
    const int per_group = gridDim.x / groups;
    const int grp = blockIdx.x % groups;
    const int t_lo = (int)((long long)n_tiles * grp / groups);
    const int t_hi = (int)((long long)n_tiles * (grp + 1) / groups);
    for (int tile = t_lo + (int)blockIdx.x / groups; tile < t_hi; tile += per_group) {
        const TileDesc td = ld_const(p.tiles, tile);
        const BucketDev bk = ld_const(p.buckets, td.bucket);
        const int nf = td.nf < 0 ? -td.nf : td.nf;
        const bool units = STAGED && p.units;
        const StepDev* __restrict__ steps = p.steps + (units ? bk.step0 : 0);
        const int n_steps = units ? bk.n_steps : p.n_steps;
        const int n_cols = units ? bk.n_cols : p.n_leaves;
        for (int i = threadIdx.x; STAGED && i < n_cols * FW; i += 64 * W) {
            const int f = i & (FW - 1), c = i / FW;
            const int ff = td.fam0 + (f < nf ? f : 0);
            const int fam = td.nf < 0 ? p.fam_list[ff] : bk.fam_begin + ff;
            const ColDev cd = units ? p.cols[bk.col0 + c] : ColDev{c, 0};
            s_cnt[i] = 8u * (cd.stride ? cd.stride : Np) * p.counts_T[(long long)cd.row * p.F + fam];
        }
        int fam[FB], dst[FB];   // this lane's families, and their places in the caller's order
#pragma unroll
        for (int f = 0; f < FB; ++f) {
            const int ff = td.fam0 + (16 * f + fl < nf ? 16 * f + fl : 0);
            fam[f] = td.nf < 0 ? p.fam_list[ff] : bk.fam_begin + ff;
            dst[f] = p.perm[fam[f]];
        }
        const __attribute__((address_space(4))) int* nslot = as_const(p.node_slot + (long long)td.point * p.n_nodes);
        const int nkt = bk.Lp / kTile;   // k-tiles of a child vector
        __syncthreads();

        // The wave's work is a list of steps: for every op and each of the wave's
        // chunks of it, the op's children.  While a step is computed, the next
        // one's first loads -- its leaf columns, or the first FB k-tiles of its
        // A operand (the same loads from a selected base, stride and lane
        // offset) -- are in flight, also across the barrier between ops: they
        // read nothing the kernel writes.
        struct Step {
            StepDev sd;
            int st;      // its index in the program
            int first;   // the op's first step
            int c;       // chunk
        };
        auto root_of = [&](const Step& s) { return (s.sd.ctl & kStepRoot) != 0; };
        auto tiles_of = [&](bool root) { return ((root ? bk.R : bk.L) + kTile - 1) / kTile; };
        auto base_of = [&](const Step& s) {   // root rows are sizes 1..R
            return (long long)nslot[s.sd.node] * p.slot_elems + (root_of(s) ? 1 : 0);
        };
        auto row_tile = [&](const Step& s, int i) {   // clamped: a chunk's tiles past the end are dropped
            const int n = tiles_of(root_of(s));
            return s.c * NTW + i < n ? s.c * NTW + i : n - 1;
        };
        auto issue = [&](d4 (&pf)[FB][NTW], const Step& s) {
            const bool leaf = s.sd.leaf_col >= 0;
            const double* M = (leaf ? p.leaf64 : p.mt64) + base_of(s);
            if (STAGED && (s.sd.ctl & kStepPattern)) {   // columns of the rows themselves
                const UnitDev u = ld_const(p.units, s.sd.in_slot);
                M = p.x64 + u.x0 + (long long)td.point * u.n * u.xs;
            }
#pragma unroll
            for (int f = 0; f < FB; ++f) {
                const int col = leaf ? s.sd.leaf_col : 0;
                const unsigned cnt = STAGED ? s_cnt[col * FW + 16 * f + fl] : 8u * Np * p.counts_T[(long long)col * p.F + fam[f]];
                const unsigned cn = cnt + 8u * g;
                const int kt = leaf ? 0 : Np * (f < nkt ? kTile * f : zero_col);
                const unsigned off = leaf ? cn : a_lane[0];
                const int step = leaf ? 4 : 4 * Np;
#pragma unroll
                for (int i = 0; i < NTW; ++i) {
                    const double* C = M + (kt + kTile * row_tile(s, i));
#pragma unroll
                    for (int r = 0; r < 4; ++r) pf[f][i][r] = at(uniform(C + r * step), off);
                }
            }
        };
        d4 acc[FB][NTW];
        auto compute = [&](const d4 (&pf)[FB][NTW], const Step& s) {
            const bool root = root_of(s);
            d4 x[FB][NTW];
            if (s.sd.leaf_col >= 0) {   // column `count` (the error model is folded into it)
#pragma unroll
                for (int f = 0; f < FB; ++f)
#pragma unroll
                    for (int i = 0; i < NTW; ++i) x[f][i] = pf[f][i];
            } else {
                const Frag V = frag + s.sd.in_slot * slot_tiles * FB * 64 + lane;
                const double* M = p.mt64 + base_of(s);
                auto mma = [&](const d4 (&a)[NTW], const d4 (&b)[FB]) {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
#pragma unroll
                        for (int f = 0; f < FB; ++f)
#pragma unroll
                            for (int i = 0; i < NTW; ++i)
                                x[f][i] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i][j], b[f][j], x[f][i], 0, 0, 0);
                };
                // k-tiles FB .. nkt - 1: D in flight while one is multiplied.  The
                // loop has no other branch, so that every wait covers only the
                // oldest k-tile: past the end it multiplies the zero block,
                // which adds exactly 0.
                constexpr int D = 2;
                d4 a[D][NTW], b[D][FB];
                auto load = [&](d4 (&a)[NTW], d4 (&b)[FB], int kt) {
                    const int kb = kt < nkt ? kt : nkt - 1;
                    const int c = Np * (kt < nkt ? kTile * kt : zero_col);
#pragma unroll
                    for (int i = 0; i < NTW; ++i) {
                        const Gptr C = uniform(M + (c + kTile * row_tile(s, i)));
#pragma unroll
                        for (int j = 0; j < 4; ++j) a[i][j] = at(C, a_lane[j]);
                    }
#pragma unroll
                    for (int f = 0; f < FB; ++f) b[f] = V[(kb * FB + f) * 64];
                };
#pragma unroll
                for (int f = 0; f < FB; ++f)
#pragma unroll
                    for (int i = 0; i < NTW; ++i) x[f][i] = d4{0, 0, 0, 0};
                d4 b0[FB][FB];
#pragma unroll
                for (int k = 0; k < FB; ++k)
#pragma unroll
                    for (int f = 0; f < FB; ++f) b0[k][f] = V[((k < nkt ? k : 0) * FB + f) * 64];
                if (nkt > FB) {
#pragma unroll
                    for (int d = 0; d < D; ++d) load(a[d], b[d], FB + d);
#pragma unroll
                    for (int k = 0; k < FB; ++k) mma(pf[k], b0[k]);
                    for (int kt = FB; kt < nkt; kt += D)
#pragma unroll
                        for (int d = 0; d < D; ++d) {
                            mma(a[d], b[d]);
                            load(a[d], b[d], kt + d + D);
                            __builtin_amdgcn_sched_barrier(0);
                        }
                } else {
#pragma unroll
                    for (int k = 0; k < FB; ++k) mma(pf[k], b0[k]);
                }
            }
            if (s.sd.ctl & kStepFirst) {
#pragma unroll
                for (int f = 0; f < FB; ++f)
#pragma unroll
                    for (int i = 0; i < NTW; ++i) acc[f][i] = x[f][i];
                asm volatile("");   // (a branch: the vector unit is the scarce one)
            } else {
#pragma unroll
                for (int f = 0; f < FB; ++f)
#pragma unroll
                    for (int i = 0; i < NTW; ++i) acc[f][i] *= x[f][i];
            }
            if (!(s.sd.ctl & kStepLast)) return;
            const int len = root ? bk.R : bk.L, nrt = tiles_of(root);
            if (STAGED && (s.sd.ctl & kStepOut)) {   // the branch's factor (its one step's) as columns
                const UnitDev u = ld_const(p.units, bk.out);
                const long long c = (long long)td.point * u.n + td.fam0 - bk.list0;
#pragma unroll
                for (int f = 0; f < FB; ++f) {
                    if (16 * f + fl >= nf) continue;
                    double* X = p.x64 + u.x0 + (c + 16 * f + fl) * u.xs + g;
#pragma unroll
                    for (int i = 0; i < NTW; ++i) {
                        const int t = s.c * NTW + i;
                        if (t >= nrt) break;
#pragma unroll
                        for (int r = 0; r < 4; ++r) X[kTile * t + 4 * r] = acc[f][i][r];
                    }
                }
                return;
            }
            const Frag out = frag + (s.sd.ctl & kStepSlotMask) * slot_tiles * FB * 64 + lane;
#pragma unroll
            for (int i = 0; i < NTW; ++i) {
                const int t = s.c * NTW + i;
                if (t >= nrt) break;
#pragma unroll
                for (int f = 0; f < FB; ++f) {
                    d4 v = acc[f][i];
                    if (kTile * t + kTile > len) {   // rows past the bound
                        asm volatile("");
#pragma unroll
                        for (int r = 0; r < 4; ++r) v[r] = kTile * t + 4 * r + g < len ? v[r] : 0.0;
                    }
                    out[(t * FB + f) * 64] = v;
                    if (root && p.root_out && 16 * f + fl < nf)
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const int j = kTile * t + 4 * r + g;
                            if (j < len) p.root_out[(long long)dst[f] * p.root_stride + j] = v[r];
                        }
                }
            }
        };
        // the step after s: the next child, the op's next chunk, or the next op
        auto advance = [&](Step& s) {
            if (!(s.sd.ctl & kStepLast)) {
                ++s.st;
            } else if ((s.c + W) * NTW < tiles_of(root_of(s))) {
                s.c += W;
                s.st = s.first;
            } else {
                s.c = wv;
                s.first = ++s.st;
            }
            s.sd = ld_const(steps, s.st < n_steps ? s.st : n_steps - 1);
        };
        d4 pfa[FB][NTW], pfb[FB][NTW];
        Step sa{ld_const(steps, 0), 0, 0, wv}, sb;
        issue(pfa, sa);
        // an op ends where the following step is another op's
        for (;;) {
            sb = sa;
            advance(sb);
            issue(pfb, sb);
            compute(pfa, sa);
            if (sb.first != sa.first) __syncthreads();
            if (sb.st >= n_steps) break;
            sa = sb;
            advance(sa);
            issue(pfa, sa);
            compute(pfb, sb);
            if (sa.first != sb.first) __syncthreads();
            if (sa.st >= n_steps) break;
        }
        if (units && bk.out >= 0) {   // (the last step has ended behind a barrier)
            continue;
        }
        const int root_slot = ld_const(steps, n_steps - 1).ctl & kStepSlotMask;

        // max_j log x_j + log prior_j (base_model.cpp:84-90) or x_j prior_j
        // (gamma_core.cpp:156-161): the largest product first, then the
        // logarithms of the rows near it only (of all rows where the product
        // leaves FP64's normal range), so the maximum is over the same values
        const Frag x = frag + root_slot * slot_tiles * FB * 64 + lane;
        const double* __restrict__ pr = p.prior64 + bk.prior_off;
        const double inf = __builtin_huge_val();
        const int nrt = (bk.R + kTile - 1) / kTile;
        double best[FB], xmax[FB];
#pragma unroll
        for (int f = 0; f < FB; ++f) {
            best[f] = -inf;
            xmax[f] = 0.0;
        }
        for (int t = wv; t < nrt; t += W)
#pragma unroll
            for (int f = 0; f < FB; ++f) {
                const d4 v = x[(t * FB + f) * 64];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int j = kTile * t + 4 * r + g;
                    if (j >= bk.R) continue;
                    const double q = v[r] * pr[j];
                    best[f] = q > best[f] ? q : best[f];
                    xmax[f] = v[r] > xmax[f] ? v[r] : xmax[f];
                }
            }
        // a family's maxima over its lanes, then over the waves
        auto over_lanes = [&](double v) {
            for (int d = 16; d <= 32; d <<= 1) {
                const double o = __shfl_xor(v, d);
                v = o > v ? o : v;
            }
            return v;
        };
#pragma unroll
        for (int f = 0; f < FB; ++f) {
            best[f] = over_lanes(best[f]);
            xmax[f] = over_lanes(xmax[f]);
            if (g == 0) {
                s_a[wv * FW + 16 * f + fl] = best[f];
                s_b[wv * FW + 16 * f + fl] = xmax[f];
            }
        }
        __syncthreads();
#pragma unroll
        for (int f = 0; f < FB; ++f)
            for (int w = 0; w < W; ++w) {
                const double b = s_a[w * FW + 16 * f + fl], m = s_b[w * FW + 16 * f + fl];
                best[f] = b > best[f] ? b : best[f];
                xmax[f] = m > xmax[f] ? m : xmax[f];
            }
        double val[FB];
#pragma unroll
        for (int f = 0; f < FB; ++f) val[f] = best[f];
        if (p.model == 0) {
#pragma unroll
            for (int f = 0; f < FB; ++f) val[f] = -inf;
            for (int t = wv; t < nrt; t += W)
#pragma unroll
                for (int f = 0; f < FB; ++f) {
                    const d4 v = x[(t * FB + f) * 64];
                    const bool every = !(best[f] >= kFp64Floor && best[f] < inf);
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int j = kTile * t + 4 * r + g;
                        if (j < bk.R && (every || v[r] * pr[j] >= best[f] * kNearBest)) {
                            const double k = log(v[r]) + log(pr[j]);
                            val[f] = k > val[f] ? k : val[f];
                        }
                    }
                }
            __syncthreads();   // the waves have read the first maxima
#pragma unroll
            for (int f = 0; f < FB; ++f) {
                val[f] = over_lanes(val[f]);
                if (g == 0) s_a[wv * FW + 16 * f + fl] = val[f];
            }
            __syncthreads();
#pragma unroll
            for (int f = 0; f < FB; ++f)
                for (int w = 0; w < W; ++w) {
                    const double b = s_a[w * FW + 16 * f + fl];
                    val[f] = b > val[f] ? b : val[f];
                }
        }
        if (wv == 0 && g == 0) {
#pragma unroll
            for (int f = 0; f < FB; ++f) {
                if (16 * f + fl >= nf) continue;
                // a first key that is not a number stays (std::max_element
                // keeps it): row 0 of the vector is this lane's
                const double x0 = x[f * 64][0];
                const double k0 = p.model == 0 ? log(x0) + log(pr[0]) : x0 * pr[0];
                p.out_val[(long long)td.point * p.F + dst[f]] = k0 != k0 ? k0 : val[f];
                p.out_flag[(long long)td.point * p.F + dst[f]] = xmax[f] == 0.0 ? kFlagZeroSum : 0;
                // values near the subnormal range are counted
                if (p.near_floor && (xmax[f] < kFp64Floor || best[f] < kFp64Floor)) atomicAdd(p.near_floor, 1);
            }
        }
        __syncthreads();   // every wave is done with this tile's LDS and vectors
    }
}

// ---------------------------------------------------------------------------
// Short recompute lists of long vectors, level by level: a launch takes the ops
// of one level of the tree (their children's vectors are complete), a wave 64
// rows of one op for one family.  A contraction is its row's chain of fused
// multiply-adds in ascending order -- the matrix instruction's sums, bit for
// bit -- over the child's vector in LDS; vectors are in global memory.
//
// A few families are a chain of steps, and one CU's share of the memory system
// bounds it: at 501 rows a step's matrix is 2 MB that no cache holds, 45 us at
// what one CU can have in flight (59 on the matrix cores, sixteen families at
// once whether they are there or not).  Spread over rows and branches, four
// families of 100 taxa at B = 500 take 0.43 ms, against 4.4 one per workgroup
// and 5.7 on the matrix cores.
// ---------------------------------------------------------------------------
constexpr int kLevelK = 32;   // columns per load group, two groups in flight

__global__ __launch_bounds__(64) void k_f64_level(PruneParams p, const int* __restrict__ op_steps, int op0, int n_level,
                                                  int n_ops, int max_tiles, int stride)
{
    const int n_tiles = *as_const(p.n_tiles_dev);
    if (n_tiles > max_tiles) return;   // k_prune_f64's
    extern __shared__ double s_vec[];   // [stride] a child's vector
    const int lane = threadIdx.x, Np = p.Np;
    const int chunks = (stride + 63) / 64;
    double* V = (double*)p.scratch;     // [family of the list][op][stride]
    const int n_items = n_tiles * kTile * n_level * chunks;
    for (int item = blockIdx.x; item < n_items; item += gridDim.x) {
        const int op = op0 + item / chunks % n_level, fi = item / chunks / n_level;
        const TileDesc td = ld_const(p.tiles, fi / kTile);
        const int nf = td.nf < 0 ? -td.nf : td.nf;
        if (fi % kTile >= nf) continue;
        const BucketDev bk = ld_const(p.buckets, td.bucket);
        const int ff = td.fam0 + fi % kTile;
        const int fam = td.nf < 0 ? p.fam_list[ff] : bk.fam_begin + ff;
        const int* nslot = p.node_slot + (long long)td.point * p.n_nodes;
        double* Vf = V + (long long)fi * n_ops * stride;
        const int row = item % chunks * 64 + lane;
        double acc = 1.0;
        bool root = false;
        for (int st = op_steps[op];;) {
            const StepDev sd = ld_const(p.steps, __builtin_amdgcn_readfirstlane(st++));
            root = (sd.ctl & kStepRoot) != 0;
            const int len = root ? bk.R : bk.L;   // (root rows are sizes 1..R)
            const int r = row < len ? row : len - 1;
            const long long base = (long long)nslot[sd.node] * p.slot_elems + (root ? 1 : 0) + r;
            double x = 0.0;
            if (sd.leaf_col >= 0) {
                x = p.leaf64[base + (long long)p.counts_T[(long long)sd.leaf_col * p.F + fam] * Np];
            } else {
                const double* M = p.mt64 + base;
                const int groups = (bk.L + kLevelK - 1) / kLevelK;   // (the vector's entries past the bound are 0)
                double a[2][kLevelK];
                auto load = [&](double (&m)[kLevelK], int gr) {
                    const double* C = M + (long long)kLevelK * (gr < groups ? gr : groups - 1) * Np;
#pragma unroll
                    for (int k = 0; k < kLevelK; ++k) m[k] = C[(long long)k * Np];
                };
                auto sum = [&](const double (&m)[kLevelK], int gr) {
                    const double* v = s_vec + kLevelK * gr;
#pragma unroll
                    for (int k = 0; k < kLevelK; ++k) x = fma(m[k], v[k], x);
                };
                load(a[0], 0);
                const double* v = Vf + (long long)sd.in_slot * stride;
                __syncthreads();
                for (int k = lane; k < stride; k += 64) s_vec[k] = v[k];
                __syncthreads();
                for (int gr = 0; gr < groups; gr += 2) {
                    load(a[1], gr + 1);
                    sum(a[0], gr);
                    if (gr + 1 >= groups) break;
                    load(a[0], gr + 2);
                    sum(a[1], gr + 1);
                }
            }
            acc = sd.ctl & kStepFirst ? x : acc * x;
            if (sd.ctl & kStepLast) break;
        }
        if (row < stride) Vf[(long long)op * stride + row] = row < (root ? bk.R : bk.L) ? acc : 0.0;
    }
}

// The root's maximum of each family of the list, as k_prune_f64 takes it.
__global__ __launch_bounds__(64) void k_f64_root(PruneParams p, int n_ops, int max_tiles, int stride)
{
    const int n_tiles = *as_const(p.n_tiles_dev);
    if (n_tiles > max_tiles) return;
    const int lane = threadIdx.x;
    auto over_wave = [&](double v) {
        for (int d = 1; d < 64; d <<= 1) {
            const double o = __shfl_xor(v, d);
            v = o > v ? o : v;
        }
        return v;
    };
    for (int fi = blockIdx.x; fi < n_tiles * kTile; fi += gridDim.x) {
        const TileDesc td = ld_const(p.tiles, fi / kTile);
        const int nf = td.nf < 0 ? -td.nf : td.nf;
        if (fi % kTile >= nf) continue;
        const BucketDev bk = ld_const(p.buckets, td.bucket);
        const int ff = td.fam0 + fi % kTile;
        const int dst = p.perm[td.nf < 0 ? p.fam_list[ff] : bk.fam_begin + ff];
        const double* x = (const double*)p.scratch + ((long long)fi * n_ops + n_ops - 1) * stride;
        const double* pr = p.prior64 + bk.prior_off;
        const double inf = __builtin_huge_val();
        double best = -inf, xmax = 0.0, val = -inf;
        for (int j = lane; j < bk.R; j += 64) {
            const double q = x[j] * pr[j];
            best = q > best ? q : best;
            xmax = x[j] > xmax ? x[j] : xmax;
        }
        best = over_wave(best);
        xmax = over_wave(xmax);
        if (p.model == 0) {
            const bool every = !(best >= kFp64Floor && best < inf);
            for (int j = lane; j < bk.R; j += 64)
                if (every || x[j] * pr[j] >= best * kNearBest) {
                    const double k = log(x[j]) + log(pr[j]);
                    val = k > val ? k : val;
                }
            val = over_wave(val);
        } else {
            val = best;
        }
        if (lane == 0) {
            const double k0 = p.model == 0 ? log(x[0]) + log(pr[0]) : x[0] * pr[0];
            p.out_val[(long long)td.point * p.F + dst] = k0 != k0 ? k0 : val;
            p.out_flag[(long long)td.point * p.F + dst] = xmax == 0.0 ? kFlagZeroSum : 0;
            if (p.near_floor && (xmax < kFp64Floor || best < kFp64Floor)) atomicAdd(p.near_floor, 1);
        }
    }
}

// Entries of a vector of nt tiles, in whole load groups.
int f64_level_stride(int nt) { return (nt * kTile + kLevelK - 1) / kLevelK * kLevelK; }

// A list of at most max_tiles tiles (p.n_tiles_dev; a longer one is left to
// k_prune_f64) over the program p.steps, whose interior steps name their
// child's op in in_slot: op_steps[op] is an op's first step, level l's ops are
// [level_ops[l], level_ops[l + 1]), the root's op the last.  p.scratch holds
// kTile max_tiles n_ops vectors.
hipError_t launch_f64_levels(int nt, int max_tiles, const int* op_steps, const int* level_ops, int n_levels,
                             const PruneParams& p, hipStream_t st)
{
    const int stride = f64_level_stride(nt), n_ops = level_ops[n_levels];
    for (int l = 0; l < n_levels; ++l)
        hipLaunchKernelGGL(k_f64_level, dim3(2048), dim3(64), sizeof(double) * stride, st, p, op_steps, level_ops[l],
                           level_ops[l + 1] - level_ops[l], n_ops, max_tiles, stride);
    hipLaunchKernelGGL(k_f64_root, dim3(kTile * max_tiles), dim3(64), 0, st, p, n_ops, max_tiles, stride);
    return hipGetLastError();
}

// One instance per shape; with per_cu set, reports how many workgroups of it
// fit on one CU (0: no such shape or it does not fit) instead of launching.
hipError_t f64_dispatch(const MfmaShape& s, int grid, const PruneParams& p, hipStream_t st, int* per_cu)
{
    if (per_cu) *per_cu = 0;
#define CAFE_F64_CASE(NTW, FB, LDSP, STAGED)                                                                      \
    if (s.ntw == NTW && s.fb == FB && s.lds == LDSP && s.staged == STAGED && s.w >= 1 && s.w <= F64Waves<NTW, FB>::v) { \
        if (per_cu)                                                                                               \
            return hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, k_prune_f64<NTW, FB, LDSP, STAGED>, 64 * s.w, \
                                                                s.shm);                                           \
        hipLaunchKernelGGL((k_prune_f64<NTW, FB, LDSP, STAGED>), dim3(grid < 1 ? 1 : grid), dim3(64 * s.w), s.shm, st, \
                           p);                                                                                    \
        return hipGetLastError();                                                                                 \
    }
    CAFE_F64_CASE(1, 1, true, true) CAFE_F64_CASE(1, 1, false, true) CAFE_F64_CASE(1, 1, false, false)
    CAFE_F64_CASE(2, 1, false, true) CAFE_F64_CASE(1, 2, true, true) CAFE_F64_CASE(2, 2, false, true)
#undef CAFE_F64_CASE
    return hipErrorInvalidValue;
}

}  // namespace cafe
