// cluster.hpp -- element forces, assembly and Newmark update of a cluster of
// elements in one kernel (GATHER assembly, wavefront element form).
//
// A cluster is up to CE elements that lie together (2 x 2 x 2 where the mesh
// allows), one workgroup of four wavefronts; a wavefront computes two of the
// elements on 25 lanes each.  A lane owns one line of five points at a time:
// the contractions along xi, eta and zeta each run on whole lines in registers
// with the entries of D as scalar operands, and the lines are exchanged
// through LDS (54 dwords per point and field; one lane per point needs 102).
// The residuals of the cluster's elements are then summed per node in LDS:
//   - interior nodes (regular, in no other cluster) take their Newmark update
//     here; their residual goes to memory only in a run's last step (keep_r),
//     for gfx_solver_get_state;
//   - the others leave one entry per cluster and node in Rl, which the node
//     kernel sums in cluster order.
//
// Why: with one residual entry per element point and one node update for all, a
// step moves 147 bytes per node and field, of which the fused form needs about
// 85 (a 2 x 2 x 2 block has 729 nodes for 1,000 points, 343 of them interior).
// Measured (MI355X; element and node stages of one step, before -> now):
// 131,072 elements, 1 field: 421 -> 321 us; 36,855 elements, 3 fields: 292 ->
// 230 us; 23,328 elements, 24 fields: 1,386 -> 1,072 us.
// Bound: LDS.  At 24 fields its pipes are busy 67 % of the kernel's time (a
// quarter of that bank conflicts, half of them the eta lines' a = 0 and a = 4
// planes meeting; no plane padding within the LDS budget removes both theirs and
// the zeta lines'), VALU 48 %, and the kernel moves 3.3 TB/s.  The contractions
// on the matrix cores took a third of the VALU work out (815 -> 538 instructions
// per wavefront and field).  Loading the next field's displacement before this
// field's stores took 714 -> 610 us: the loads otherwise wait for the stores.
#pragma once

#include <type_traits>

#include "kernels.hpp"

namespace gfx {
namespace dev {

constexpr int CE = 8;                  // elements per cluster
constexpr int CLUSTER_THREADS = 256;   // two elements per wavefront

// One cluster.  Its nodes form two lists (interior, then the others), each
// sorted by the number of the cluster's elements that hold the node, largest
// first; ci[m] / cb[m] = nodes of more than m elements (packed in cnt[m]).  The points to sum
// are stored level by level: for m = 0, 1, ...: the (m+1)-th point of each of
// the first ci[m] interior nodes, then the same for the other list, from ent +
// e0 * 125 (point = element in cluster * 125 + point).  Interior node t is node
// ibase + t; the others' entries in Rl are bdst[boff + t].
struct ClusterHead {
    int32_t e0, ne, ibase, boff;
    uint32_t cnt[8];  // ci[m] | cb[m] << 16
};

// A point's three components in LDS or memory.
struct __attribute__((packed, aligned(4))) F3 {
    float v[3];
};
struct __attribute__((packed, aligned(4))) F5 {
    float v[5];
};

// out[i] = sum_s M[i][s] in[s] for the three components of each lane's line,
// M = D or (TR) its transpose.  Rows 0..3 run on the matrix cores: the 4 x 4 x 1
// FP32 MFMA takes column s of M from the lanes (row lane % 4, in m[s]) and one
// line's value in[s] per lane, and returns rows 0..3 of the lane's own line, so
// five of them are 20 of the line's 25 products at twice the VALU's rate while
// the VALU does row 4 and the other wavefronts' work.  Every lane of the
// wavefront must be active.
typedef float f32x4 __attribute__((ext_vector_type(4)));
template <bool TR>
__device__ __forceinline__ void line_contract(const float* D, const float (&m)[5], const F3 (&in)[5], F3 (&out)[5]) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        float a4 = 0.f;
#pragma unroll
        for (int s = 0; s < 5; ++s) {
            acc = __builtin_amdgcn_mfma_f32_4x4x1f32(m[s], in[s].v[c], acc, 0, 0, 0);
            a4 += (TR ? D[s * 5 + 4] : D[20 + s]) * in[s].v[c];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) out[i].v[c] = acc[i];
        out[4].v[c] = a4;
    }
}

template <int STRIDE>
__device__ __forceinline__ void line_load(const F3* b, F3 (&x)[5]) {
#pragma unroll
    for (int s = 0; s < 5; ++s) x[s] = b[s * STRIDE];
}

template <int STRIDE>
__device__ __forceinline__ void line_store(F3* b, const F3 (&x)[5]) {
#pragma unroll
    for (int s = 0; s < 5; ++s) b[s * STRIDE] = x[s];
}

// Node n of a field (base uniform; the host keeps 12 n below 2^32, so one
// 32-bit offset register addresses it).
__device__ __forceinline__ F3& at_node(float* base, int32_t n) {
    return *reinterpret_cast<F3*>(reinterpret_cast<char*>(base) + uint32_t(n) * 12u);
}
__device__ __forceinline__ const F3& at_node(const float* base, int32_t n) {
    return *reinterpret_cast<const F3*>(reinterpret_cast<const char*>(base) + uint32_t(n) * 12u);
}

enum { CL_FUSED = 0, CL_POINTS = 1 };

// OUT = CL_FUSED: the whole element stage and the interior nodes' update.
// OUT = CL_POINTS: residuals only, one entry per element point (the per-stage
// entry points, whose source injection comes between the two).
template <bool DIAG, int OUT>
__device__ __forceinline__ void cluster_body(const ElemArgs& A, const ClusterHead& H) {
    __shared__ F3 su[CE * NP];  // displacement
    __shared__ F3 sx[CE * NP];  // xi lines: gradient, flux, divergence; then the element residuals
    __shared__ F3 sy[CE * NP];  // eta lines
    __shared__ uint16_t sent[CE * NP];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int ne = H.ne;
    if (OUT == CL_FUSED)
        for (int q = tid; q < ne * NP; q += CLUSTER_THREADS) sent[q] = A.cl_ent[int64_t(H.e0) * NP + q];

    // loads of this wavefront's two elements: 250 consecutive points, four per lane
    const int npt = max(0, min(2, ne - 2 * wv)) * NP;
    const int64_t ptw = int64_t(H.e0 + 2 * wv) * NP;
    int32_t nd[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int i = lane + 64 * q;
        nd[q] = i < npt ? int32_t(__builtin_nontemporal_load(&A.ibool[ptw + i]) & ~FIRST_TOUCH) : -1;
    }
    // lines: lane (element, a, b)
    // (one element per half wavefront: lines of two elements in one half would
    // meet in the LDS banks; the seven lanes left over repeat lines and store nothing)
    const int el = lane >> 5, hl = lane & 31;
    const int qd = hl < 25 ? hl : hl - 7;
    const bool live = hl < 25 && 2 * wv + el < ne;
    const int a5 = qd / 5, b5 = qd - a5 * 5;
    const int eb = (2 * wv + el) * NP;
    const int ew = H.e0 + min(2 * wv + el, ne - 1);
    const int64_t pt0 = int64_t(ew) * NP + qd * 5;
    constexpr int NG9 = DIAG ? 3 : 9;
    F5 g[NG9];
#pragma unroll
    for (int c = 0; c < NG9; ++c) g[c] = *reinterpret_cast<const F5*>(A.G + (DIAG ? c * 4 : c) * A.P + pt0);
    const F5 lam = *reinterpret_cast<const F5*>(A.lam + pt0), mu = *reinterpret_cast<const F5*>(A.mu + pt0);
    // one flag per wavefront: few elements have a source, and with the lists' bounds
    // held over the fields the kernel spilled five registers (131,072 elements,
    // 1 field: 222 -> 212 us)
    const bool src = __any(A.src_off[ew] < A.src_off[ew + 1]);
    const int step = A.ctr[0];
    float md[5], mt[5];  // row lane % 4 of D and of its transpose
#pragma unroll
    for (int s = 0; s < 5; ++s) {
        md[s] = A.D[(lane & 3) * 5 + s];
        mt[s] = A.D[s * 5 + (lane & 3)];
    }
    F3* const xl = sx + eb + qd;               // xi line (j, k) = (a, b): stride 25
    F3* const yl = sy + eb + a5 * 25 + b5;     // eta line (i, k) = (a, b): stride 5
    F3* const ul = su + eb + qd * 5;           // zeta line (i, j) = (a, b): stride 1
    F3* const xk = sx + eb + qd * 5;
    F3* const yk = sy + eb + qd * 5;

    // the cluster's nodes, up to four per lane: where the residual goes and 1/m
    constexpr int NQ = (CE * NP + CLUSTER_THREADS - 1) / CLUSTER_THREADS;
    constexpr int NPRE = 2;  // interior nodes of a lane whose u and w are loaded ahead (343 in a 2 x 2 x 2 block)
    const int n_int = H.cnt[0] & 0xffff, n_all = n_int + (H.cnt[0] >> 16);
    int all_int = 0;  // points of the interior nodes
#pragma unroll
    for (int m = 0; m < CE; ++m) all_int += H.cnt[m] & 0xffff;
    const int nf = A.nf;
    float un[4][3];
    auto load_u = [&](const float* base) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const F3 x = at_node(base, max(nd[q], 0));
            un[q][0] = x.v[0];
            un[q][1] = x.v[1];
            un[q][2] = x.v[2];
        }
    };
    load_u(A.U);

    for (int f = 0; f < nf; ++f) {
        const int64_t fo = int64_t(f) * A.fstride;
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (nd[q] >= 0) su[2 * wv * NP + lane + 64 * q] = F3{un[q][0], un[q][1], un[q][2]};
        wave_sync();
        F3 in[5], out[5], dk[5];
        line_load<25>(su + eb + qd, in);
        line_contract<false>(A.D, md, in, out);
        if (live) line_store<25>(xl, out);
        line_load<5>(su + eb + a5 * 25 + b5, in);
        line_contract<false>(A.D, md, in, out);
        if (live) line_store<5>(yl, out);
        line_load<1>(ul, in);
        line_contract<false>(A.D, md, in, dk);
        wave_sync();
#pragma unroll
        for (int s = 0; s < 5; ++s) {
            const F3 dx = xk[s], dy = yk[s];
            float du[3][3], gg[9], F[9];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                du[c][0] = dx.v[c];
                du[c][1] = dy.v[c];
                du[c][2] = dk[s].v[c];
            }
#pragma unroll
            for (int c = 0; c < 9; ++c) gg[c] = DIAG ? ((c & 3) == 0 ? g[c / 4].v[s] : 0.f) : g[c % NG9].v[s];
            flux_from_du<DIAG>(du, gg, lam.v[s], mu.v[s], F);
            if (live) {
                xk[s] = F3{F[0], F[3], F[6]};
                yk[s] = F3{F[1], F[4], F[7]};
            }
            dk[s] = F3{F[2], F[5], F[8]};
        }
        wave_sync();
        line_load<25>(xl, in);
        line_contract<true>(A.D, mt, in, out);
        if (live) line_store<25>(xl, out);
        line_load<5>(yl, in);
        line_contract<true>(A.D, mt, in, out);
        if (live) line_store<5>(yl, out);
        line_contract<true>(A.D, mt, dk, out);
        wave_sync();
        if (live) {
#pragma unroll
            for (int s = 0; s < 5; ++s) {
                const F3 rx = xk[s], ry = yk[s];
                F3 rv;
#pragma unroll
                for (int c = 0; c < 3; ++c) rv.v[c] = -((rx.v[c] + ry.v[c]) + out[s].v[c]);
                xk[s] = rv;
            }
            if (src)  // point sources, as add_sources
                for (int q = A.src_off[ew], se = A.src_off[ew + 1]; q < se; ++q) {
                    const int4 en = A.src_ent[q];
                    if (en.x != f || step >= A.nstf) continue;
                    const float amp = A.stf[int64_t(f) * A.nstf + step];
                    for (int s = 0; s < 5; ++s) xk[s].v[en.y] += amp * A.src_w[en.z + qd * 5 + s];
                }
            if (OUT == CL_POINTS)
                for (int s = 0; s < 5; ++s)
                    *reinterpret_cast<F3*>(A.Rl + (int64_t(f) * A.PR + A.rdst[pt0 + s]) * 3) = xk[s];
        }
        // the next field's displacement comes in while this one is summed; it is
        // asked for before this field's stores, which the memory counter would
        // otherwise have to see through first
        const float* const next = A.U + fo + (f + 1 < nf ? A.fstride : 0);
        if (OUT == CL_POINTS) {  // su and sx are rewritten only by this wavefront
            load_u(next);
            continue;
        }
        int t0 = tid;
        asm volatile("" : "+v"(t0));  // list positions are made here for every field, not held over the loop
        int32_t dst[NQ];
        float mi[NPRE];
        F3 pw[NPRE];
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const int t = t0 + CLUSTER_THREADS * q;
            dst[q] = t < n_int ? H.ibase + t : t < n_all ? A.cl_bdst[H.boff + t - n_int] : 0;
            if (q < NPRE) {
                const int32_t n = t < n_int ? dst[q] : 0;
                mi[q < NPRE ? q : 0] = A.minv[n];
                pw[q < NPRE ? q : 0] = at_node(A.Ww + fo, n);
            }
        }
        load_u(next);
        __syncthreads();
        // every node's first point, all of a lane's nodes together
        float r[NQ][3], uu[NPRE][3];
        int pos[NQ];
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const int t = t0 + CLUSTER_THREADS * q;
            pos[q] = t < n_int ? t : t < n_all ? all_int + t - n_int : 0;
            const int p = sent[pos[q]];
            const F3 x = sx[p];
#pragma unroll
            for (int c = 0; c < 3; ++c) r[q][c] = 0.f + x.v[c];
            if (q < NPRE) {
                const F3 u = su[p];
#pragma unroll
                for (int c = 0; c < 3; ++c) uu[q < NPRE ? q : 0][c] = u.v[c];
            }
        }
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const int t = t0 + CLUSTER_THREADS * q;
            if (t >= n_all) break;
            const bool in = t < n_int;
            const int i = in ? t : t - n_int;
            // its other points: one, then two, then four at a time (a point that
            // is not there adds nothing); nodes of 2 x 2 x 2 blocks have 1, 2, 4 or 8
            int at = pos[q];
            auto count = [&](int m) { return int(in ? H.cnt[m] & 0xffff : H.cnt[m] >> 16); };
            auto more = [&](auto first, auto n) {
                constexpr int M = decltype(first)::value, N = decltype(n)::value;
                F3 x[N];
                bool have[N];
#pragma unroll
                for (int k = 0; k < N; ++k) {
                    have[k] = i < count(M + k);
                    at += count(M + k - 1);
                    x[k] = sx[sent[have[k] ? at : pos[q]]];
                }
#pragma unroll
                for (int k = 0; k < N; ++k)
#pragma unroll
                    for (int c = 0; c < 3; ++c) r[q][c] += have[k] ? x[k].v[c] : 0.f;
            };
            using std::integral_constant;
            if (i < count(1)) {
                more(integral_constant<int, 1>{}, integral_constant<int, 1>{});
                if (i < count(2)) {
                    more(integral_constant<int, 2>{}, integral_constant<int, 2>{});
                    if (i < count(4)) more(integral_constant<int, 4>{}, integral_constant<int, 4>{});
                }
            }
            if (!in || A.keep_r) at_node(A.Rl + int64_t(f) * A.PR * 3, dst[q]) = F3{r[q][0], r[q][1], r[q][2]};
            if (in) {  // the regular nodes' update
                F3 u, w;
                float m1;
                if (q < NPRE) {
                    constexpr int Q = NPRE - 1;
#pragma unroll
                    for (int c = 0; c < 3; ++c) u.v[c] = uu[q < Q ? q : Q][c];
                    w = pw[q < Q ? q : Q];
                    m1 = mi[q < Q ? q : Q];
                } else {
                    u = su[sent[pos[q]]];
                    w = at_node(A.Ww + fo, dst[q]);
                    m1 = A.minv[dst[q]];
                }
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    const float a1 = r[q][c] * m1;
                    w.v[c] = w.v[c] + A.dt * a1;
                    u.v[c] = u.v[c] + A.dt * w.v[c];
                }
                at_node(A.Ww + fo, dst[q]) = w;
                at_node(A.Uw + fo, dst[q]) = u;
            }
        }
        if (f + 1 < nf) __syncthreads();  // su and sx are rewritten by the next field
    }
}

template <bool DIAG, int OUT>
__global__ void __launch_bounds__(CLUSTER_THREADS, DIAG ? 4 : 3) k_cluster(ElemArgs A, int c0) {
    cluster_body<DIAG, OUT>(A, const_row(A.cl_head, c0 + xcd_block(blockIdx.x, gridDim.x)));
}

// One launch for the clusters of several solvers: map entry (solver, cluster).
template <bool DIAG>
__global__ void __launch_bounds__(CLUSTER_THREADS, DIAG ? 4 : 3)
    k_cluster_grp(const ElemArgs* __restrict__ tab, const int4* __restrict__ map) {
    const int4 E = map[xcd_block(blockIdx.x, gridDim.x)];
    const ElemArgs& A = const_row(tab, E.x);
    cluster_body<DIAG, CL_FUSED>(A, const_row(A.cl_head, E.y));
}

// The nodes the cluster kernel leaves, in one launch: workgroups below
// spec_blocks take 256 special nodes each, the others 256 regular nodes shared
// by clusters.  A lane sums its node's entries itself: with one entry per
// cluster most nodes have none or one beside their own, so little is left to
// stage through LDS (special nodes and their C-PML state hold 85 registers, five
// wavefronts per SIMD; at 23,328 elements, 24 fields the launch moves 5.2 TB/s,
// at 500,000 the special nodes by themselves 4.5: 8.3 ms, where sums staged
// through LDS over entries per point took 7.5; the shared regular nodes 3.2
// against 7.3).
// blockIdx.y: fields [y * chunk, (y + 1) * chunk).  ctr (may be null): the
// launch closes the step as k_advance does (no record kernel follows; nothing
// in the launch reads the counters).
__device__ __forceinline__ void cluster_entries(const NodeArgs& A, int f, int64_t g, int kb, int n, const int32_t (&id)[3],
                                                float* r) {
    const float* const Rl = A.Rl + int64_t(f) * A.PR * 3;
    const F3 a = *reinterpret_cast<const F3*>(Rl + g * 3);
    F3 x[3];
#pragma unroll
    for (int k = 0; k < 3; ++k)
        if (k < n) x[k] = *reinterpret_cast<const F3*>(Rl + int64_t(id[k]) * 3);
#pragma unroll
    for (int c = 0; c < 3; ++c) r[c] = 0.f + a.v[c];
#pragma unroll
    for (int k = 0; k < 3; ++k)
        if (k < n)
#pragma unroll
            for (int c = 0; c < 3; ++c) r[c] += x[k].v[c];
    for (int k = 3; k < n; ++k) {
        const F3 y = *reinterpret_cast<const F3*>(Rl + int64_t(A.pts[kb + k]) * 3);
#pragma unroll
        for (int c = 0; c < 3; ++c) r[c] += y.v[c];
    }
}

__device__ __forceinline__ void cluster_nodes_body(const NodeArgs& A, int blk, int spec_blocks, int f0, int f1) {
    const bool special = blk < spec_blocks;
    const int64_t g = special ? int64_t(blk) * 256 + threadIdx.x : A.Ga + int64_t(blk - spec_blocks) * 256 + threadIdx.x;
    if (g >= (special ? A.Ga : A.G4)) return;
    const int kb = A.off[g], n = A.off[g + 1] - kb;
    int32_t id[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) id[k] = k < n ? A.pts[kb + k] : 0;
    if (special) {
        const SpecialNode N = special_node(A, g);
        for (int f = f0; f < f1; ++f) {
            SpecialState S;
            load_special(A, N, g, f, S);
            float R[3];
            cluster_entries(A, f, g, kb, n, id, R);
            update_special(A, N, g, f, S, R);
        }
    } else {
        const float mi = A.minv[g];
        for (int f = f0; f < f1; ++f) {
            F3* const up = reinterpret_cast<F3*>(A.U + int64_t(f) * A.fstride + g * 3);
            F3* const wp = reinterpret_cast<F3*>(A.W + int64_t(f) * A.fstride + g * 3);
            F3 u = *up, w = *wp;
            float r[3];
            cluster_entries(A, f, g, kb, n, id, r);
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const float a1 = r[c] * mi;
                w.v[c] = w.v[c] + A.dt * a1;
                u.v[c] = u.v[c] + A.dt * w.v[c];
            }
            *wp = w;
            *up = u;
        }
    }
}

__device__ __forceinline__ void advance_step(int* ctr, int stride) {
    const int st = ctr[0];
    if (stride > 0 && st % stride == 0) ctr[1] = ctr[1] + 1;
    ctr[0] = st + 1;
}

__global__ void __launch_bounds__(256) k_cluster_nodes(NodeArgs A, int spec_blocks, int chunk, int* ctr, int stride) {
    if (ctr && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) advance_step(ctr, stride);
    const int f0 = blockIdx.y * chunk;
    cluster_nodes_body(A, blockIdx.x, spec_blocks, f0, min(A.nf, f0 + chunk));
}

// One launch for the nodes of several solvers: map entry (solver, special
// workgroups, first field, workgroup).
__global__ void __launch_bounds__(256)
    k_cluster_nodes_grp(const NodeArgs* __restrict__ tab, const int4* __restrict__ map, int chunk) {
    const int4 E = map[blockIdx.x];
    const NodeArgs& A = const_row(tab, E.x);
    cluster_nodes_body(A, E.w, E.y, E.z, min(A.nf, E.z + chunk));
}

}  // namespace dev
}  // namespace gfx
