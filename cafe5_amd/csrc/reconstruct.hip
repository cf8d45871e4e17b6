// reconstruct.hip -- Pupko's joint ancestral reconstruction on the GPU
// (replaces pupko_reconstructor::reconstruct_gene_family and its node steps,
// src/gene_family_reconstructor.cpp:30-189).
//
// Up the tree (children first) a node's row over parent sizes i is
//     L[i] = max_j  (prod_children L_child[j]) * M[i][j],
// with the product formed in the reference's order (1.0 times each child's
// entry in descendant order; a leaf's row is column `count` of its matrix).
// The reference also keeps the first j that reaches each maximum; of those a
// family needs one per node, the one at its parent's state, so it is looked up
// on the way down: the first j whose value equals L[i].  Values and
// comparisons are the reference's, bit for bit, so the states are.  The root
// takes the first best j = 1..Rr-1 of the product times the prior
// (root_equilibrium_distribution::compute(j)).
//
// The contraction is a max of products, so it runs on the vector units: two
// neighbouring parent sizes per lane (one 16-byte load per child size), FT
// families per wave, a matrix block of kRecJB child sizes by 128 parent sizes
// in registers for all of them, the products broadcast from LDS.  A block is
// skipped where (its largest product) x (the largest matrix entry of the two
// rows in it) exceeds no row's maximum so far: rounding is monotonic, so no
// value of it could.  The products fall off past the family's own sizes;
// 20,000 families of 34 taxa at B = 200 keep a quarter of their blocks.
//
// Bound by: the vector units half of the time (670 M instructions), the rest
// latency of the matrix blocks (16 loads each) with three waves per SIMD, and
// 1 GB of rows written and read again.  20,000 families of 34 taxa at B = 200:
// 2.4 ms, against 17.4 ms for one family per wave with every block taken, the
// argmax kept along and the matrix through LDS.  Blocks of 8 halve the
// registers but double the tests (3.0 ms), loading a block ahead costs a wave
// per SIMD (3.4 ms), one row per lane doubles the loads (3.5 ms).
#include <algorithm>

#include "engine.h"
#include "prune_common.h"

namespace cafe {

constexpr int kRecJB = 16;   // child sizes per block
typedef double d2 __attribute__((ext_vector_type(2)));

// The largest entry of every pair of rows in every block of child sizes:
// tab[(node, block)][i / 2] for the interior branches of the program.
__global__ __launch_bounds__(256) void k_block_max(const ReconNode* __restrict__ nodes, const double* __restrict__ mt64,
                                                   int Np, long long slot_elems, int Lq, double* __restrict__ tab)
{
    const int h = blockIdx.x * 256 + threadIdx.x;
    if (2 * h >= Lq) return;
    const int J = blockIdx.y, s = blockIdx.z;
    const double* M = mt64 + (long long)nodes[s].slot * slot_elems + (long long)J * kRecJB * Np + 2 * h;
    double m = 0.0;
#pragma unroll
    for (int jj = 0; jj < kRecJB; ++jj) {   // (rows and columns past N are 0)
        const d2 v = *(const d2*)(M + (long long)jj * Np);
        m = fmax(m, fmax(v[0], v[1]));
    }
    tab[((long long)s * gridDim.y + J) * (Lq / 2) + h] = m;
}

// max over kRecJB / 2 lanes of a DPP row, in the last of them (entries >= 0)
__device__ __forceinline__ double block_max(double v)
{
    auto shr = [](double x, auto ctrl) {
        const unsigned long long u = __builtin_bit_cast(unsigned long long, x);
        const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)u, decltype(ctrl)::value, 0xF, 0xF, false);
        const int hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(u >> 32), decltype(ctrl)::value, 0xF, 0xF, false);
        return __builtin_bit_cast(double, ((unsigned long long)(unsigned)hi << 32) | (unsigned)lo);
    };
    v = fmax(v, shr(v, std::integral_constant<int, 0x111>{}));
    v = fmax(v, shr(v, std::integral_constant<int, 0x112>{}));
    if constexpr (kRecJB == 16) v = fmax(v, shr(v, std::integral_constant<int, 0x114>{}));
    return v;
}

// Families fams[0 .. nf-1] (count row, row of states), FT per workgroup of one
// wave; L_all holds [family rounded up to FT][interior node but the root][Ls].
// tab: k_block_max's (null: no block is skipped).  err[0]: a count outside the
// matrix (a plain store of 1; any family may set it).
template <int FT>
__global__ __launch_bounds__(64) void k_reconstruct(const ReconNode* __restrict__ nodes, int n_prog,
                                                    const ReconKid* __restrict__ kids,
                                                    const double* __restrict__ mt64, int N, int Np,
                                                    long long slot_elems, const double* __restrict__ tab,
                                                    const int* __restrict__ counts_T, int F,
                                                    const int2* __restrict__ fams, int nf,
                                                    const double* __restrict__ prior, int B, int Rr,
                                                    double* L_all, int Lp, int n_nodes, int* states,
                                                    int* __restrict__ err)
{
    const int lane = threadIdx.x;
    const int Lq = (Lp + kRecJB - 1) / kRecJB * kRecJB, nj = Lq / kRecJB, Ls = Lp + (Lp & 1);
    extern __shared__ __align__(16) double s_rec[];
    double* s_prod = s_rec;              // [FT][Lq] the node's products
    double* s_pm = s_rec + FT * Lq;      // [nj][FT] their maxima per block
    int fs[FT];
    bool valid[FT];
    double* L[FT];
    int* st[FT];
#pragma unroll
    for (int f = 0; f < FT; ++f) {
        const int k = (int)blockIdx.x * FT + f;
        valid[f] = k < nf;   // past the last family: the last one again, in rows of its own
        const int kk = valid[f] ? k : nf - 1;
        fs[f] = __builtin_amdgcn_readfirstlane(fams[kk].x);
        L[f] = L_all + (long long)k * (n_prog - 1) * Ls;
        st[f] = states + (long long)__builtin_amdgcn_readfirstlane(fams[kk].y) * n_nodes;
    }
    auto count_of = [&](int leaf_col, int f) {
        const int obs = as_const(counts_T)[(long long)leaf_col * F + fs[f]];
        if (obs >= 0 && obs < N) return obs;
        if (lane == 0) err[0] = 1;   // flagged, read as 0
        return 0;
    };
    // family f's row of a child
    auto row_of = [&](const ReconKid& kd, int f) -> const double* {
        return kd.leaf_col >= 0 ? mt64 + (long long)kd.slot * slot_elems + (long long)count_of(kd.leaf_col, f) * Np
                                : L[f] + (long long)kd.ref * Ls;
    };
    // a node's children: the first two's rows at hand
    struct Family2 {
        const double* r0[FT];
        const double* r1[FT];
    };
    auto children = [&](const ReconNode& nd) {
        const ReconKid k0 = ld_const(kids, nd.kid0), k1 = ld_const(kids, nd.kid0 + (nd.n_kids > 1 ? 1 : 0));
        Family2 r;
#pragma unroll
        for (int f = 0; f < FT; ++f) {
            r.r0[f] = row_of(k0, f);
            r.r1[f] = row_of(k1, f);
        }
        return r;
    };
    // their product at size j (of sizes j and j + 1: V = d2), in descendant order
    auto product = [&](const ReconNode& nd, const Family2& r, int j, auto (&v)[FT]) {
        typedef std::remove_reference_t<decltype(v[0])> V;
        V w[FT];
#pragma unroll
        for (int f = 0; f < FT; ++f) {
            v[f] = *(const V*)(r.r0[f] + j);
            w[f] = *(const V*)(r.r1[f] + j);
        }
        if (nd.n_kids > 1)
#pragma unroll
            for (int f = 0; f < FT; ++f) v[f] *= w[f];
        for (int c = 2; c < nd.n_kids; ++c) {
            const ReconKid kd = ld_const(kids, nd.kid0 + c);
#pragma unroll
            for (int f = 0; f < FT; ++f) v[f] *= *(const V*)(row_of(kd, f) + j);
        }
    };

    for (int s = 0; s + 1 < n_prog; ++s) {
        const ReconNode nd = ld_const(nodes, s);
        const Family2 r = children(nd);
        for (int j0 = 0; j0 < Lq; j0 += 128) {
            const int j = j0 + 2 * lane;
            d2 v[FT];
            product(nd, r, j < Ls ? j : Ls - 2, v);
#pragma unroll
            for (int f = 0; f < FT; ++f) {
                if (j >= Lp) v[f][0] = 0.0;
                if (j + 1 >= Lp) v[f][1] = 0.0;
                const double m = block_max(fmax(v[f][0], v[f][1]));
                if (j < Lq) {
                    *(d2*)(s_prod + f * Lq + j) = v[f];
                    if (2 * lane % kRecJB == kRecJB - 2) s_pm[j / kRecJB * FT + f] = m;
                }
            }
        }
        __syncthreads();   // (one wave: orders its accesses)
        const double* M = mt64 + (long long)nd.slot * slot_elems;
        const double* T = tab ? tab + (long long)s * nj * (Lq / 2) : nullptr;
        // rows 128 g + 2 lane and the next one (past the last block: that one's again)
        for (int i0 = 2 * lane; __builtin_amdgcn_readfirstlane(i0) < Lp; i0 += 128) {
            const int i = i0 < Lq ? i0 : Lq - 2;
            d2 best[FT];
            double low[FT];   // the smaller of the two
#pragma unroll
            for (int f = 0; f < FT; ++f) {
                best[f] = d2{-1, -1};
                low[f] = -1;
            }
            double next = T ? T[i / 2] : 0.0;
            for (int J = 0; J < nj; ++J) {
                const double top = next;
                if (T) next = T[(J + 1 < nj ? J + 1 : J) * (Lq / 2) + i / 2];
                unsigned need = 0;
#pragma unroll
                for (int f = 0; f < FT; ++f)
                    if (__ballot(!T || s_pm[J * FT + f] * top > low[f])) need |= 1u << f;
                if (!need) continue;
                d2 m[kRecJB];
                const double* C = M + (long long)J * kRecJB * Np + i;
#pragma unroll
                for (int jj = 0; jj < kRecJB; ++jj) m[jj] = *(const d2*)(C + jj * Np);
#pragma unroll
                for (int f = 0; f < FT; ++f) {
                    if (!(need >> f & 1)) continue;
                    const d2* p = (const d2*)(s_prod + f * Lq + J * kRecJB);
#pragma unroll
                    for (int jj = 0; jj < kRecJB; jj += 2) {
                        const d2 w = p[jj / 2];
#pragma unroll
                        for (int q = 0; q < 2; ++q) {
                            best[f][q] = fmax(best[f][q], w[0] * m[jj][q]);
                            best[f][q] = fmax(best[f][q], w[1] * m[jj + 1][q]);
                        }
                    }
                    low[f] = fmin(best[f][0], best[f][1]);
                }
            }
            if (i0 < Ls)
#pragma unroll
                for (int f = 0; f < FT; ++f) *(d2*)(L[f] + (long long)s * Ls + i0) = best[f];
        }
        __syncthreads();
    }

    // the root: the first best j = 1..Rr-1 (0 where none exceeds -1)
    {
        const ReconNode nd = ld_const(nodes, n_prog - 1);
        double best[FT];
        int arg[FT];
#pragma unroll
        for (int f = 0; f < FT; ++f) {
            best[f] = -1;
            arg[f] = 0;
        }
        const Family2 r = children(nd);
        for (int j0 = 1; j0 < Rr; j0 += 64) {
            const int j = j0 + lane;
            double v[FT];
            product(nd, r, j < Rr ? j : Rr - 1, v);
            const double pr = prior[j < Rr ? j : Rr - 1];
#pragma unroll
            for (int f = 0; f < FT; ++f) {
                const double val = v[f] * pr;
                if (j < Rr && val > best[f]) {
                    best[f] = val;
                    arg[f] = j;
                }
            }
        }
#pragma unroll
        for (int f = 0; f < FT; ++f) {
            for (int d = 1; d < 64; d <<= 1) {
                const double ob = __shfl_xor(best[f], d);
                const int oa = __shfl_xor(arg[f], d);
                if (ob > best[f] || (ob == best[f] && oa < arg[f])) {
                    best[f] = ob;
                    arg[f] = oa;
                }
            }
            if (valid[f]) st[f][nd.node] = arg[f];
        }
    }
    // parents first: each child's state at its parent's (every lane stores the
    // states it reads back)
    for (int s = n_prog - 1; s >= 0; --s) {
        const ReconNode nd = ld_const(nodes, s);
        int ps[FT];
#pragma unroll
        for (int f = 0; f < FT; ++f) ps[f] = st[f][nd.node];
        for (int c = 0; c < nd.n_kids; ++c) {
            const ReconKid kd = ld_const(kids, nd.kid0 + c);
            if (kd.leaf_col >= 0) {
#pragma unroll
                for (int f = 0; f < FT; ++f)
                    if (valid[f]) st[f][kd.ref] = count_of(kd.leaf_col, f);
                continue;
            }
            const ReconNode ch = ld_const(nodes, kd.ref);
            const Family2 r = children(ch);
            const double* M = mt64 + (long long)kd.slot * slot_elems;
            double want[FT];
            int arg[FT];
            unsigned open = 0;
#pragma unroll
            for (int f = 0; f < FT; ++f) {
                want[f] = L[f][(long long)kd.ref * Ls + ps[f]];
                arg[f] = 0;
                if (valid[f]) open |= 1u << f;
            }
            for (int j0 = 0; j0 < Lp && open; j0 += 64) {
                const int j = j0 + lane < Lp ? j0 + lane : B;   // (B again finds nothing that B did not)
                double v[FT];
                product(ch, r, j, v);
#pragma unroll
                for (int f = 0; f < FT; ++f) {
                    const unsigned long long hit = __ballot(v[f] * M[(long long)j * Np + ps[f]] == want[f]);
                    if (hit && (open >> f & 1)) {
                        arg[f] = min(j0 + __builtin_ctzll(hit), B);
                        open &= ~(1u << f);
                    }
                }
            }
#pragma unroll
            for (int f = 0; f < FT; ++f)
                if (valid[f]) st[f][ch.node] = arg[f];
        }
    }
}

static int block_rows(int Lp) { return (Lp + kRecJB - 1) / kRecJB * kRecJB; }

// Doubles of k_block_max's table.
size_t recon_table_doubles(int n_prog, int Lp)
{
    return (size_t)(n_prog - 1) * (block_rows(Lp) / kRecJB) * (block_rows(Lp) / 2);
}

hipError_t launch_block_max(const ReconNode* nodes, int n_prog, const double* mt64, int Np, long long slot_elems,
                            int Lp, double* tab, hipStream_t st)
{
    const int Lq = block_rows(Lp), nj = Lq / kRecJB;
    for (int s0 = 0; s0 < n_prog - 1; s0 += 65535)   // grid.z
        hipLaunchKernelGGL(k_block_max, dim3((Lq / 2 + 255) / 256, nj, std::min(65535, n_prog - 1 - s0)), dim3(256), 0, st,
                           nodes + s0, mt64, Np, slot_elems, Lq, tab + (size_t)s0 * nj * (Lq / 2));
    return hipGetLastError();
}

hipError_t launch_reconstruct(const ReconNode* nodes, int n_prog, const ReconKid* kids, const double* mt64, int N,
                              int Np, long long slot_elems, const double* tab, const int* counts_T, int F,
                              const int2* fams, int nf, const double* prior, int B, int Rr, double* L_all, int Lp,
                              int n_nodes, int* states, int* err, hipStream_t st)
{
    if (nf <= 0) return hipSuccess;
    const int Lq = block_rows(Lp);
    auto go = [&](auto ft) {
        constexpr int FT = decltype(ft)::value;
        const size_t shm = sizeof(double) * (size_t)FT * (Lq + Lq / kRecJB);
        hipLaunchKernelGGL(k_reconstruct<FT>, dim3((nf + FT - 1) / FT), dim3(64), shm, st, nodes, n_prog, kids, mt64, N,
                           Np, slot_elems, tab, counts_T, F, fams, nf, prior, B, Rr, L_all, Lp, n_nodes, states,
                           err);
        return hipGetLastError();
    };
    return nf >= kRecFew && Lp <= kRecMaxShared ? go(std::integral_constant<int, kRecFT>{}) : go(std::integral_constant<int, 1>{});
}

}  // namespace cafe
