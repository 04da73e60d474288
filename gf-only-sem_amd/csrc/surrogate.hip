// surrogate.hip -- strain Green's tensor tiles on the device, the GLL
// interpolation judge, and a Fourier-feature coordinate MLP trained on the
// tiles (BF16 MFMA, FP32 accumulation, hand-written forward / backward / Adam).
//
// Judge: greenfun/gll_interpolator.py:117-227 restated: exact-node shortcut
// (<= 1e-6 m), cell lookup by box with 1e-6 m slack (nearest cell centre
// among the boxes that contain the point), reference coordinates from the
// cell's corner box clipped to [-1, 1], tensor-product GLL Lagrange weights
// renormalised to sum 1, weighted sum of the cell's 125 node values.
//
// MLP: (x, y, z, t) scaled to [-1, 1] -> [sin, cos](2 pi B x) with B ~ N(0,
// sigma^2) (n_freq x 4) -> depth x (Linear(width) + GELU) -> Linear(n_out).
// Every product runs on v_mfma_f32_16x16x32_bf16: operands rounded to BF16
// (round to nearest even), FP32 accumulation; master weights and Adam moments
// stay FP32.
#include <cmath>
#include <cstring>
#include <memory>
#include <random>

#include "device.hpp"
#include "gfx.h"
#include "green.hpp"
#include "gfx_surrogate.h"

namespace gfx {
namespace sur {

constexpr int NP = 125;
constexpr double EXACT_TOL = 1e-6;  // gll_interpolator.py:19

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__host__ __device__ inline uint16_t f2bf(float f) {
    uint32_t u = __builtin_bit_cast(uint32_t, f);
    u += 0x7FFFu + ((u >> 16) & 1u);  // round to nearest even (inputs are finite)
    return uint16_t(u >> 16);
}

// ------------------------------ judge ------------------------------------

__device__ __host__ inline void lagrange5(double xi, double* l) {
    const double x[5] = {-1.0, -0.6546536707079771, 0.0, 0.6546536707079771, 1.0};  // sqrt(3/7)
    for (int i = 0; i < 5; ++i) {
        double v = 1.0;
        for (int j = 0; j < 5; ++j)
            if (j != i) v *= (xi - x[j]) / (x[i] - x[j]);
        l[i] = v;
    }
}

struct JudgeArgs {
    int n_node, n_cell, n_time;
    const float* val;
    const int32_t* cell_idx;
    const double* xyz;
    const double* box;
    int nb0, nb1, nb2;
    double b00, b01, b02, bh0, bh1, bh2;
    const int32_t* bin_off;
    const int32_t* bin_cell;
};

// Containing cell of p (box with slack), nearest centre first; -1 when outside.
__device__ inline int find_cell(const JudgeArgs& A, const double p[3]) {
    int bi[3];
    const int nbv[3] = {A.nb0, A.nb1, A.nb2};
    const double b0[3] = {A.b00, A.b01, A.b02}, bh[3] = {A.bh0, A.bh1, A.bh2};
    for (int d = 0; d < 3; ++d) {
        const double q = (p[d] - b0[d]) / bh[d];
        if (q < -1e-9 || q > nbv[d] + 1e-9) return -1;
        bi[d] = min(max(int(floor(q)), 0), nbv[d] - 1);
    }
    const int b = (bi[2] * A.nb1 + bi[1]) * A.nb0 + bi[0];
    int best = -1;
    double bd = 1e300;
    for (int q = A.bin_off[b]; q < A.bin_off[b + 1]; ++q) {
        const int c = A.bin_cell[q];
        const double* bx = A.box + int64_t(c) * 6;
        if (p[0] < bx[0] - EXACT_TOL || p[0] > bx[1] + EXACT_TOL || p[1] < bx[2] - EXACT_TOL ||
            p[1] > bx[3] + EXACT_TOL || p[2] < bx[4] - EXACT_TOL || p[2] > bx[5] + EXACT_TOL)
            continue;
        const double cx = 0.5 * (bx[0] + bx[1]) - p[0], cy = 0.5 * (bx[2] + bx[3]) - p[1],
                     cz = 0.5 * (bx[4] + bx[5]) - p[2];
        const double dd = cx * cx + cy * cy + cz * cz;
        if (dd < bd || (dd == bd && c < best)) {
            bd = dd;
            best = c;
        }
    }
    return best;
}

// Region (cell, time window) of tile time index t: window t * n_window / n_time.
__host__ __device__ inline int64_t region_of(int cell, int t, int n_time, int n_window) {
    const int w = (t >= 0 && t < n_time) ? int(int64_t(t) * n_window / n_time) : 0;
    return int64_t(cell) * n_window + w;
}

// Lanes of one wavefront exchange data through LDS.
__device__ inline void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Q queries per wavefront: a lane each finds the cells, then the wavefront
// evaluates one query after the other with the 125 nodes of its cell spread over
// the lanes for the exact-node test and the weights; for the sum, 63 lanes take
// seven nodes at a time, nine lanes of two values each.  Q = 1 up to 8,192
// queries, which then all run at once, and grows beyond, so that the search is
// not repeated by 64 lanes.  One lane per query took 97 us for 600 queries (its
// 2,375 dependent loads run one after the other); this takes 14 us.
// policy null: every point is evaluated, NaN where there is no cell or time.
// policy [n_cell][n_window]: out holds other answers; a point keeps them where
// its region says 0, becomes zero at 2, and is evaluated at 1 and outside all
// cells (NaN there); *count is raised by the points evaluated.
constexpr int JQ = 4;  // wavefronts per workgroup

struct JudgeShared {
    double lag[15], w[NP + 3], part[7][18];
};

__device__ inline void judge_eval(const JudgeArgs& A, JudgeShared& S, const double (&p)[3], int c, int t,
                                  float* __restrict__ o) {
    const int lane = threadIdx.x & 63;
    if (c < 0 || t < 0 || t >= A.n_time) {
        if (lane < 18) o[lane] = __builtin_nanf("");
        return;
    }
    const int32_t* ci = A.cell_idx + int64_t(c) * NP;
    const float* vt = A.val + int64_t(t) * A.n_node * 18;
    // exact-node shortcut (gll_interpolator.py:172-177): the first such node
    int hit = -1;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int k = lane + 64 * h;
        bool at = false;
        if (k < NP) {
            const double* x = A.xyz + int64_t(ci[k]) * 3;
            const double dx = x[0] - p[0], dy = x[1] - p[1], dz = x[2] - p[2];
            at = dx * dx + dy * dy + dz * dz < EXACT_TOL * EXACT_TOL;
        }
        const unsigned long long m = __ballot(at);
        if (hit < 0 && m) hit = 64 * h + __ffsll(m) - 1;
    }
    if (hit >= 0) {
        if (lane < 18) o[lane] = vt[int64_t(ci[hit]) * 18 + lane];
        return;
    }
    if (lane < 15) {  // lane (axis d, point a): its Lagrange polynomial at the query
        const double g[5] = {-1.0, -0.6546536707079771, 0.0, 0.6546536707079771, 1.0};  // sqrt(3/7)
        const int d = lane / 5, a = lane - 5 * d;
        const double* bx = A.box + int64_t(c) * 6;
        const double pd = d == 0 ? p[0] : d == 1 ? p[1] : p[2];
        const double lo = bx[2 * d], hi = bx[2 * d + 1];
        const double xi = fmin(1.0, fmax(-1.0, 2.0 * (pd - lo) / (hi - lo) - 1.0));
        const double ga = a == 0 ? g[0] : a == 1 ? g[1] : a == 2 ? g[2] : a == 3 ? g[3] : g[4];
        double v = 1.0;
#pragma unroll
        for (int j = 0; j < 5; ++j)
            if (j != a) v *= (xi - g[j]) / (ga - g[j]);
        S.lag[lane] = v;
    }
    wave_sync();
    double w[2] = {0.0, 0.0}, sw;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int k = lane + 64 * h;
        if (k < NP) w[h] = S.lag[k / 25] * S.lag[5 + (k / 5) % 5] * S.lag[10 + k % 5];
    }
    sw = w[0] + w[1];
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) sw += __shfl_xor(sw, s);
    S.w[lane] = w[0] / sw;
    if (lane + 64 < NP) S.w[lane + 64] = w[1] / sw;
    wave_sync();
    const int sub = lane / 9, pair = lane - 9 * sub;
    if (sub < 7) {
        double a0 = 0.0, a1 = 0.0;
#pragma unroll 6
        for (int k = sub; k < NP; k += 7) {
            const float2 v = *reinterpret_cast<const float2*>(vt + int64_t(ci[k]) * 18 + 2 * pair);
            a0 += S.w[k] * double(v.x);
            a1 += S.w[k] * double(v.y);
        }
        S.part[sub][2 * pair] = a0;
        S.part[sub][2 * pair + 1] = a1;
    }
    wave_sync();
    if (lane < 18) {
        double s = 0.0;
#pragma unroll
        for (int k = 0; k < 7; ++k) s += S.part[k][lane];
        o[lane] = float(s);
    }
    wave_sync();  // S is rewritten by the next query
}

__global__ void __launch_bounds__(64 * JQ)
    k_judge(JudgeArgs A, int n, int Q, const double* __restrict__ q, const int32_t* __restrict__ tix,
            const uint8_t* __restrict__ policy, int n_window, float* __restrict__ out, int32_t* __restrict__ cell_out,
            int* __restrict__ count) {
    __shared__ JudgeShared sh[JQ];
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int64_t base = (int64_t(blockIdx.x) * JQ + wv) * Q;
    const bool mine = lane < Q && base + lane < n;
    double p[3] = {0.0, 0.0, 0.0};
    int c = -1, t = 0, how = 0;
    if (mine) {
        const int64_t i = base + lane;
        for (int d = 0; d < 3; ++d) p[d] = q[3 * i + d];
        t = tix[i];
        c = find_cell(A, p);
        if (cell_out) cell_out[i] = c;
        how = !policy || c < 0 ? 1 : policy[region_of(c, t, A.n_time, n_window)];
        if (how == 2)
            for (int k = 0; k < 18; ++k) out[i * 18 + k] = 0.f;
    }
    unsigned long long todo = __ballot(how == 1);
    if (count && lane == 0 && todo) atomicAdd(count, __popcll(todo));
    while (todo) {
        const int l = __ffsll(todo) - 1;
        todo &= todo - 1;
        const double pq[3] = {__shfl(p[0], l), __shfl(p[1], l), __shfl(p[2], l)};
        judge_eval(A, sh[wv], pq, __shfl(c, l), __shfl(t, l), out + (base + l) * 18);
    }
}

// Queries per wavefront and workgroups for n queries.
int judge_q(int n) { return std::min(64, std::max(1, (n + 8191) / 8192)); }
int judge_blocks(int n) { return int((n + int64_t(JQ) * judge_q(n) - 1) / (int64_t(JQ) * judge_q(n))); }

JudgeArgs judge_args(const gfx_green& G) {
    JudgeArgs a{};
    a.n_node = G.n_node;
    a.n_cell = G.n_cell;
    a.n_time = G.n_time;
    a.val = G.val.p;
    a.cell_idx = G.cell_idx.p;
    a.xyz = G.xyz.p;
    a.box = G.box.p;
    a.nb0 = G.nb[0];
    a.nb1 = G.nb[1];
    a.nb2 = G.nb[2];
    a.b00 = G.b0[0];
    a.b01 = G.b0[1];
    a.b02 = G.b0[2];
    a.bh0 = G.bh[0];
    a.bh1 = G.bh[1];
    a.bh2 = G.bh[2];
    a.bin_off = G.bin_off.p;
    a.bin_cell = G.bin_cell.p;
    return a;
}

// -------------------------------- MLP -------------------------------------
//
// Every product is one form: C(m, n) = sum_k A[m][k] B[n][k] with both operands
// BF16 and k-contiguous, leading dimensions padded to 64 with zeros.  Whoever
// makes an operand (features, a layer's GELU, its gradient, Adam) rounds it to
// BF16 once (nearest even) in the layout, or the two layouts, in which products
// read it: activations and gradients [row][unit] for the next product along the
// network and [unit][row] for the weight gradients, weights both ways.  Sums,
// biases, pre-activations, master weights and moments stay FP32.
//
// Bound: at 131,072 rows a hidden layer takes 61 us, of which erff is more than
// half (33.5 M values); its traffic would take 26 us.  At a training batch of
// 8,192 rows the launches are latency bound (9 to 11 us a layer and direction,
// traffic 2 to 4).  One Adam iteration of the default network: 212 us (204 of them
// in its 20 kernels), with FP32 operands rounded and transposed while staging, separate bias and GELU passes and
// 256-term sums by single lanes 1,380 us; 150,000 queries: 0.8 ms of kernels (2.9 ms).

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
constexpr int GK = 64;        // k per stage, and the padding of leading dimensions
constexpr int GKP = GK + 8;   // LDS row: 144 bytes, so the 16 lanes of a read phase meet distinct banks

inline int pad64(int n) { return (n + 63) / 64 * 64; }

// What a product's tile turns into.
enum {
    EPI_HIDDEN = 0,  // z = acc + bias; optionally Z = z; gelu(z) as BF16, one or two layouts
    EPI_OUT = 1,     // acc + bias, FP32
    EPI_BACK = 2,    // acc * gelu'(Z) as BF16, both layouts, and its column sums (bias gradient)
    EPI_PART = 3     // acc, FP32 partial product of one k range
};

struct GemmArgs {
    const uint16_t* A;
    const uint16_t* B;
    int lda, ldb;
    int M, N, K;          // K a multiple of 64 (zero padded)
    const float* bias;    // [N]
    float* Z;             // [M][ldz] pre-activations (written by EPI_HIDDEN when set, read by EPI_BACK)
    int ldz;              // padded to 64
    uint16_t* H;          // [M][ldh], may be null
    int ldh;
    uint16_t* Ht;         // [N][ldt] transposed, rows m in [M, ldt) zero; may be null
    int ldt;
    float* out;           // EPI_OUT [M][N]; EPI_PART [z][M][N]; EPI_BACK [row tile][N] column sums
};

// The weight gradients of all layers as one launch: block -> (layer, tile).
struct GradArgs {
    static constexpr int MAX = 33;
    GemmArgs g[MAX];
    int tile0[MAX + 1];  // first block of each layer
    int n, kc;           // layers; k per split
};
static_assert(sizeof(GradArgs) <= 4096, "kernel arguments");

__device__ inline float gelu(float z) { return 0.5f * z * (1.f + erff(z * 0.70710678118654752f)); }
__device__ inline float gelu_d(float z) {
    return 0.5f * (1.f + erff(z * 0.70710678118654752f)) + z * 0.39894228040143268f * expf(-0.5f * z * z);
}

// One T x T tile of C (T = 128 or 64) by four wavefronts of T/2 x T/2 each, on
// v_mfma_f32_16x16x32_bf16 with B as the first operand: lane l feeds row l % 16
// of A and of B with k = 8 (l / 16) .. + 7 and receives row l % 16 of C, columns
// 4 (l / 16) .. + 3.  A stage of 64 k comes in as 16-byte loads, one stage ahead
// of the products.
template <int EPI, int T>
__device__ __forceinline__ void gemm_tile(const GemmArgs& G, int mt, int nt, int kbeg, int kend, int z) {
    constexpr int F = T / 32;       // 16 x 16 tiles per wavefront and side
    constexpr int L = T * GK / 8 / 256;  // 16-byte pieces per lane, operand and stage
    // the stages of both operands; the epilogue's transposed tile and column sums
    constexpr int STAGE = 2 * T * GKP, EPIL = T * (T + 8) + 4 * T;
    __shared__ __attribute__((aligned(16))) uint16_t sA[STAGE > EPIL ? STAGE : EPIL];
    uint16_t* const sB = sA + T * GKP;
    const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
    const int mb = mt * T, nb = nt * T;
    const int wm = (wave >> 1) * (T / 2), wn = (wave & 1) * (T / 2);
    const int r16 = lane & 15, kq = (lane >> 4) * 8;
    // Built-in vectors: as an array of uint4 structs the stage went to scratch, and
    // eight Adam iterations of 8,192 rows took 2.7 instead of 1.8 ms.  Two or four
    // stages ahead (four are a whole layer of 256 units) were no faster: 1.70 and
    // 1.80 ms against 1.69.
    u32x4 ra[L], rb[L];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int q = 0; q < L; ++q) {
            const int i = t + 256 * q, row = i >> 3, kk = (i & 7) * 8;
            // rows past the end repeat the last one; their results are not stored
            ra[q] = *reinterpret_cast<const u32x4*>(G.A + int64_t(min(mb + row, G.M - 1)) * G.lda + k0 + kk);
            rb[q] = *reinterpret_cast<const u32x4*>(G.B + int64_t(min(nb + row, G.N - 1)) * G.ldb + k0 + kk);
        }
    };
    f32x4 acc[F][F];
#pragma unroll
    for (int i = 0; i < F; ++i)
#pragma unroll
        for (int j = 0; j < F; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    fetch(kbeg);
    for (int k0 = kbeg; k0 < kend; k0 += GK) {
        __syncthreads();  // the previous stage has been read
#pragma unroll
        for (int q = 0; q < L; ++q) {
            const int i = t + 256 * q, row = i >> 3, kk = (i & 7) * 8;
            *reinterpret_cast<u32x4*>(&sA[row * GKP + kk]) = ra[q];
            *reinterpret_cast<u32x4*>(&sB[row * GKP + kk]) = rb[q];
        }
        __syncthreads();
        if (k0 + GK < kend) fetch(k0 + GK);
#pragma unroll
        for (int kk = 0; kk < GK; kk += 32) {
            bf16x8 a[F], b[F];
#pragma unroll
            for (int i = 0; i < F; ++i) a[i] = *reinterpret_cast<const bf16x8*>(&sA[(wm + i * 16 + r16) * GKP + kk + kq]);
#pragma unroll
            for (int j = 0; j < F; ++j) b[j] = *reinterpret_cast<const bf16x8*>(&sB[(wn + j * 16 + r16) * GKP + kk + kq]);
#pragma unroll
            for (int i = 0; i < F; ++i)
#pragma unroll
                for (int j = 0; j < F; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j], a[i], acc[i][j], 0, 0, 0);
        }
    }
    // a lane holds row m of the tile and four neighbouring columns: results go out
    // in 8- and 16-byte pieces, the transposed copy through LDS
    const bool back = EPI == EPI_BACK;
    const bool transpose = (EPI == EPI_HIDDEN || back) && G.Ht;  // uniform
    if (back || transpose) __syncthreads();  // the stages have been read
    uint16_t* const sT = sA;                       // [T columns][T + 8 rows]
    float* const sum = reinterpret_cast<float*>(sA + T * (T + 8));  // column sums of the two row halves
#pragma unroll
    for (int j = 0; j < F; ++j) {
        const int nl = wn + j * 16 + (lane >> 4) * 4, n0 = nb + nl;
        float bias[4], col[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            bias[q] = (EPI == EPI_HIDDEN || EPI == EPI_OUT) && n0 + q < G.N ? G.bias[n0 + q] : 0.f;
            col[q] = 0.f;
        }
#pragma unroll
        for (int i = 0; i < F; ++i) {
            const int ml = wm + i * 16 + r16, m = mb + ml;
            float v[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) v[q] = acc[i][j][q];
            if (EPI == EPI_OUT || EPI == EPI_PART) {
                if (EPI == EPI_PART && G.N % 4 == 0) {  // 16-byte aligned: the layers before have whole rows of four
                    if (m < G.M && n0 < G.N)
                        *reinterpret_cast<float4*>(G.out + (int64_t(z) * G.M + m) * G.N + n0) = make_float4(v[0], v[1], v[2], v[3]);
                    continue;
                }
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (m < G.M && n0 + q < G.N) G.out[(int64_t(z) * G.M + m) * G.N + n0 + q] = v[q] + bias[q];
                continue;
            }
            const bool row = m < G.M;
            if (EPI == EPI_HIDDEN) {
#pragma unroll
                for (int q = 0; q < 4; ++q) v[q] += bias[q];
                if (row && G.Z && n0 < G.ldz) *reinterpret_cast<float4*>(G.Z + int64_t(m) * G.ldz + n0) = make_float4(v[0], v[1], v[2], v[3]);
#pragma unroll
                for (int q = 0; q < 4; ++q) v[q] = row && n0 + q < G.N ? gelu(v[q]) : 0.f;
            } else {
                const float4 zz = row && n0 < G.ldz ? *reinterpret_cast<const float4*>(G.Z + int64_t(m) * G.ldz + n0) : make_float4(0.f, 0.f, 0.f, 0.f);
                const float zq[4] = {zz.x, zz.y, zz.z, zz.w};
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    v[q] = row && n0 + q < G.N ? v[q] * gelu_d(zq[q]) : 0.f;
                    col[q] += v[q];
                }
            }
            uint32_t h[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) h[q] = f2bf(v[q]);
            if (G.H && row && n0 < G.ldh)  // columns past N: zero
                *reinterpret_cast<uint2*>(G.H + int64_t(m) * G.ldh + n0) = make_uint2(h[0] | h[1] << 16, h[2] | h[3] << 16);
            if (transpose)
#pragma unroll
                for (int q = 0; q < 4; ++q) sT[(nl + q) * (T + 8) + ml] = uint16_t(h[q]);
        }
        if (back)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
#pragma unroll
                for (int x = 1; x < 16; x <<= 1) col[q] += __shfl_xor(col[q], x);
                if (r16 == 0) sum[(wave >> 1) * T + nl + q] = col[q];
            }
    }
    if (back || transpose) __syncthreads();
    if (transpose)
        for (int c = t; c < T * T / 8; c += 256) {  // rows past M: zero, up to ldt
            const int n = c / (T / 8), m = (c - n * (T / 8)) * 8;
            if (nb + n < G.N && mb + m < G.ldt)
                *reinterpret_cast<uint4*>(G.Ht + int64_t(nb + n) * G.ldt + mb + m) =
                    *reinterpret_cast<const uint4*>(&sT[n * (T + 8) + m]);
        }
    if (back)
        for (int n = t; n < T; n += 256)
            if (nb + n < G.N) G.out[int64_t(mt) * G.N + nb + n] = sum[n] + sum[T + n];
}

template <int EPI, int T>
__global__ void __launch_bounds__(256) k_gemm(GemmArgs G) {
    gemm_tile<EPI, T>(G, blockIdx.y, blockIdx.x, 0, G.K, 0);
}

// dW = H^T dZ of every layer: the rows split over blockIdx.y, partial products
// summed afterwards in split order.
__global__ void __launch_bounds__(256) k_gemm_grads(GradArgs W) {
    int l = 0;
    while (l + 1 < W.n && int(blockIdx.x) >= W.tile0[l + 1]) ++l;
    const GemmArgs& G = W.g[l];
    const int tile = blockIdx.x - W.tile0[l], tn = (G.N + 63) / 64;
    const int kbeg = blockIdx.y * W.kc;
    gemm_tile<EPI_PART, 64>(G, tile / tn, tile % tn, kbeg, min(G.K, kbeg + W.kc), blockIdx.y);
}

// Gradient of every parameter from its partial sums, in order: W (layer l, i)
// from `splits` products, b from the row tiles' column sums.
struct ReduceArgs {
    int n;                       // layers
    int64_t w_off[GradArgs::MAX];   // its weights, then its biases
    int64_t w_part[GradArgs::MAX];  // first partial product of the layer
    int64_t b_part[GradArgs::MAX];
    int size[GradArgs::MAX], cols[GradArgs::MAX], tiles[GradArgs::MAX];
    int blk0[GradArgs::MAX];  // first workgroup of the layer
    int splits;
};
// 64 parameters of one layer per workgroup, four lanes each, so that the many row
// tiles of a bias do not run as one serial chain; the four sums are added in lane
// order.  The layer is the workgroup's: its table is read by scalar loads, where a
// search per lane read the kernel's arguments entry after entry.
__global__ void __launch_bounds__(256) k_reduce_grads(ReduceArgs R, const float* __restrict__ wp,
                                                      const float* __restrict__ bp, float* __restrict__ g) {
    __shared__ float sh[4][64];
    const int c = threadIdx.x & 63, part = threadIdx.x >> 6;
    int l = 0;
    while (l + 1 < R.n && int(blockIdx.x) >= R.blk0[l + 1]) ++l;
    const int i = (int(blockIdx.x) - R.blk0[l]) * 64 + c, size = R.size[l], cols = R.cols[l];
    float s = 0.f;
    if (i < size + cols) {
        const bool bias = i >= size;
        const int cnt = bias ? R.tiles[l] : R.splits;
        const int64_t stride = bias ? cols : size;
        const float* src = bias ? bp + R.b_part[l] + (i - size) : wp + R.w_part[l] + i;
        const int q = (cnt + 3) / 4;
#pragma unroll 4
        for (int z = part * q; z < min(cnt, part * q + q); ++z) s += src[z * stride];
    }
    sh[part][c] = s;
    __syncthreads();
    if (part == 0 && i < size + cols) g[R.w_off[l] + i] = ((sh[0][c] + sh[1][c]) + sh[2][c]) + sh[3][c];
}

// features [sin, cos](2 pi B x) as BF16, [row][ld] (columns past 2 n_freq zero)
// and, when set, transposed [feature][ldt] with rows past the end zero; X in
// [rows][4] scaled to [-1, 1].  A lane makes eight frequencies of one row, so
// that rows are written in 16-byte pieces (n_freq a multiple of 8) and the
// transposed layout a wavefront's 64 rows at a time.
__global__ void __launch_bounds__(256) k_fourier(const float* __restrict__ X, int rows, const float* __restrict__ Bf,
                                                 int n_freq, uint16_t* __restrict__ H, int ld,
                                                 uint16_t* __restrict__ Ht, int ldt) {
    const int r = blockIdx.x * 64 + (threadIdx.x & 63);
    if (r >= max(rows, Ht ? ldt : 0)) return;
    const bool in = r < rows;
    float x[4] = {0.f, 0.f, 0.f, 0.f};
    if (in)
        for (int d = 0; d < 4; ++d) x[d] = X[int64_t(r) * 4 + d];
    uint16_t* const row = H + int64_t(r) * ld;
    const bool wide = n_freq % 8 == 0;
    const int first = (blockIdx.y * 4 + (threadIdx.x >> 6)) * 8;
    for (int j0 = first; j0 < n_freq; j0 += gridDim.y * 32) {
        uint32_t s[4] = {}, c[4] = {};
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int j = j0 + q;
            if (j >= n_freq) break;
            float v = 0.f;
            for (int d = 0; d < 4; ++d) v += Bf[j * 4 + d] * x[d];
            v *= 6.283185307179586f;
            const uint32_t a = in ? f2bf(sinf(v)) : 0u, b = in ? f2bf(cosf(v)) : 0u;
            s[q / 2] |= a << (16 * (q & 1));
            c[q / 2] |= b << (16 * (q & 1));
            if (!wide && in) {
                row[j] = uint16_t(a);
                row[n_freq + j] = uint16_t(b);
            }
            if (Ht) {
                Ht[int64_t(j) * ldt + r] = uint16_t(a);
                Ht[int64_t(n_freq + j) * ldt + r] = uint16_t(b);
            }
        }
        if (wide && in) {
            *reinterpret_cast<uint4*>(row + j0) = make_uint4(s[0], s[1], s[2], s[3]);
            *reinterpret_cast<uint4*>(row + n_freq + j0) = make_uint4(c[0], c[1], c[2], c[3]);
        }
    }
    if (in && first == 0)
        for (int j = 2 * n_freq; j < ld; ++j) row[j] = 0;
}

// Squared error of 64 rows and its gradient as BF16 (both layouts), with the
// gradient's column sums per 64 rows.  out, y: [rows][18].  One wavefront per
// workgroup: with 256 rows each, 8,192 rows were 32 workgroups and took 11 us.
constexpr int NO = 18;
constexpr int MSE_ROWS = 64;
__global__ void __launch_bounds__(MSE_ROWS) k_mse(const float* __restrict__ out, const float* __restrict__ y, int rows,
                                                  float inv_n, uint16_t* __restrict__ D, int ld, uint16_t* __restrict__ Dt,
                                                  int ldt, float* __restrict__ col, float* __restrict__ loss) {
    const int lane = threadIdx.x, r = blockIdx.x * MSE_ROWS + lane;
    const bool in = r < rows;
    float e = 0.f, c[NO];
#pragma unroll
    for (int k = 0; k < NO; ++k) c[k] = 0.f;
    if (in)
#pragma unroll
        for (int k = 0; k < NO; ++k) {
            const float d = out[int64_t(r) * NO + k] - y[int64_t(r) * NO + k];
            e += d * d;
            c[k] = 2.f * d * inv_n;
            D[int64_t(r) * ld + k] = f2bf(c[k]);
        }
    if (r < ldt)
#pragma unroll
        for (int k = 0; k < NO; ++k) Dt[int64_t(k) * ldt + r] = f2bf(c[k]);
    for (int s = 32; s > 0; s >>= 1) {
        e += __shfl_xor(e, s);
#pragma unroll
        for (int k = 0; k < NO; ++k) c[k] += __shfl_xor(c[k], s);
    }
    if (lane == 0) {
        loss[blockIdx.x] = e;
#pragma unroll
        for (int k = 0; k < NO; ++k) col[int64_t(blockIdx.x) * NO + k] = c[k];
    }
}

// The batch's loss in FP64 by one wavefront: the workgroups' sums, always in the
// same order.
__global__ void __launch_bounds__(64) k_loss(const float* __restrict__ part, int n, double inv_n, double* __restrict__ dst) {
    double s = 0.0;
    for (int i = threadIdx.x; i < n; i += 64) s += part[i];
    for (int x = 32; x > 0; x >>= 1) s += __shfl_xor(s, x);
    if (threadIdx.x == 0) *dst = s * inv_n;
}

// One layer's place in the parameter array and its BF16 copies: Wt [out][ld_in]
// (forward) and Wn [in][ld_out] (backward).
struct Layers {
    int n;
    int64_t w_off[GradArgs::MAX], b_off[GradArgs::MAX];
    int in[GradArgs::MAX], out[GradArgs::MAX];
    int64_t wt[GradArgs::MAX], wn[GradArgs::MAX];  // offsets in the copies' buffer
};

__device__ inline void round_weight(const Layers& Y, int64_t i, float w, uint16_t* __restrict__ copies) {
    int l = 0;
    while (l + 1 < Y.n && i >= Y.w_off[l + 1]) ++l;
    if (i >= Y.b_off[l]) return;  // biases are added in FP32
    const int q = int(i - Y.w_off[l]), a = q / Y.out[l], b = q - a * Y.out[l];
    const uint16_t h = f2bf(w);
    copies[Y.wt[l] + int64_t(b) * ((Y.in[l] + 63) / 64 * 64) + a] = h;
    copies[Y.wn[l] + int64_t(a) * ((Y.out[l] + 63) / 64 * 64) + b] = h;
}

__global__ void k_round_weights(const float* __restrict__ w, int64_t n, Layers Y, uint16_t* __restrict__ copies) {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) round_weight(Y, i, w[i], copies);
}

__global__ void k_adam(float* __restrict__ w, const float* __restrict__ g, float* __restrict__ m, float* __restrict__ v,
                       int64_t n, float lr, float b1, float b2, float eps, float c1, float c2, Layers Y,
                       uint16_t* __restrict__ copies) {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    w[i] = wi;
    round_weight(Y, i, wi, copies);
}

// Output envelope e(r), r = horizontal distance from (cx, cy): piecewise
// linear through env[i] at r_i = (i + 0.5) h, h = r_max / n, constant outside
// [r_0, r_{n-1}]; 1 when n == 0.
// The network's time input is the retarded time t - slowness * r (moveout).
struct Envelope {
    const float* env;  // device or host array of n knots
    int n;
    double cx, cy, r_max, slowness;
};

__host__ __device__ inline double retarded_time(const Envelope& E, double x, double y, double t) {
    if (E.slowness == 0.0) return t;
    return t - E.slowness * sqrt((x - E.cx) * (x - E.cx) + (y - E.cy) * (y - E.cy));
}

__host__ __device__ inline float envelope_at(const Envelope& E, double x, double y) {
    if (E.n <= 0) return 1.f;
    const double r = sqrt((x - E.cx) * (x - E.cx) + (y - E.cy) * (y - E.cy));
    const double u = r * E.n / E.r_max - 0.5;
    if (u <= 0.0) return E.env[0];
    if (u >= E.n - 1) return E.env[E.n - 1];
    const int i = int(u);
    const float f = float(u - i);
    return E.env[i] * (1.f - f) + E.env[i + 1] * f;
}

__device__ inline uint64_t mix64(uint64_t z) {
    z += 0x9E3779B97F4A7C15ULL;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
}

// training batch from a tile: random (node, time) pairs; inputs scaled to
// [-1, 1], targets divided by the per-output scale and the envelope
__global__ void k_sample_tile(const float* __restrict__ val, const double* __restrict__ xyz, int n_node, int n_time,
                              double t0, double dt, const double* __restrict__ lo, const double* __restrict__ hi,
                              const float* __restrict__ inv_scale, Envelope E, uint64_t seed, int rows,
                              float* __restrict__ X, float* __restrict__ Y) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= rows) return;
    const uint64_t h = mix64(seed ^ (uint64_t(r) * 0xD1B54A32D192ED03ULL));
    const int node = int(h % uint64_t(n_node));
    const int t = int((h >> 32) % uint64_t(n_time));
    const double px = xyz[int64_t(node) * 3], py = xyz[int64_t(node) * 3 + 1];
    const double in[4] = {px, py, xyz[int64_t(node) * 3 + 2], retarded_time(E, px, py, t0 + t * dt)};
    for (int d = 0; d < 4; ++d) X[int64_t(r) * 4 + d] = float(2.0 * (in[d] - lo[d]) / (hi[d] - lo[d]) - 1.0);
    const float ie = 1.f / envelope_at(E, px, py);
    const float* v = val + (int64_t(t) * n_node + node) * 18;
    for (int k = 0; k < 18; ++k) Y[int64_t(r) * 18 + k] = v[k] * inv_scale[k] * ie;
}

// raw (x, y, z, t) -> scaled inputs, the time retarded; t from t0 + tix dt when
// tix is given (q then holds x, y, z).  No contraction: the values the host rounds.
__global__ void k_inputs(const double* __restrict__ q, const int32_t* __restrict__ tix, double t0, double dt, int rows,
                         const double* __restrict__ lo, const double* __restrict__ hi, Envelope E,
                         float* __restrict__ X) {
#pragma clang fp contract(off)
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= rows) return;
    const double* p = q + int64_t(r) * (tix ? 3 : 4);
    const double t = tix ? t0 + tix[r] * dt : p[3];
    const double in[4] = {p[0], p[1], p[2], retarded_time(E, p[0], p[1], t)};
    for (int d = 0; d < 4; ++d) X[int64_t(r) * 4 + d] = float(2.0 * (in[d] - lo[d]) / (hi[d] - lo[d]) - 1.0);
}

// network outputs -> values: times the output scale and the envelope
__global__ void k_outputs(const float* __restrict__ out, const double* __restrict__ q, int stride, int rows,
                          const double* __restrict__ scale, Envelope E, float* __restrict__ y) {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= int64_t(rows) * NO) return;
    const int64_t r = i / NO;
    const double e = envelope_at(E, q[r * stride], q[r * stride + 1]);
    y[i] = float(out[i] * scale[i - r * NO] * e);
}

}  // namespace sur
}  // namespace gfx

struct gfx_mlp {
    gfx_mlp_config cfg{};
    int n_feat = 0;
    std::vector<int> lin_in, lin_out;        // per linear layer
    std::vector<int64_t> w_off, b_off;       // offsets in the flat parameter array
    int64_t n_params = 0;
    gfx::DevBuf<float> w, g, m, v, Bf;
    gfx::DevBuf<double> lo, hi, scale;
    gfx::DevBuf<float> inv_scale;
    std::vector<double> h_scale;
    // output envelope (knots on the host and the device)
    std::vector<float> h_env;
    gfx::DevBuf<float> env;
    double env_cx = 0, env_cy = 0, env_rmax = 1, slowness = 0;
    gfx::sur::Envelope envelope(bool device) const {
        return gfx::sur::Envelope{device ? env.p : h_env.data(), int(h_env.size()), env_cx, env_cy, env_rmax,
                                  slowness};
    }
    // BF16 copies of the weights, both ways, for every layer
    gfx::sur::Layers layers{};
    gfx::DevBuf<uint16_t> copies;
    // inputs and outputs of a call, and the activations on the way (grown to the
    // largest chunk or batch used, freed with the network)
    int cap = 0;
    gfx::DevBuf<float> X, out;
    gfx::DevBuf<uint16_t> ha, hb;      // activations of two consecutive layers
    gfx::DevBuf<double> raw;
    gfx::DevBuf<int32_t> tix;
    gfx::DevBuf<float> y;
    gfx::DevBuf<uint8_t> policy;       // a query's answer per region
    gfx::DevBuf<int> count;            // points the judge answered
    // training: per layer pre-activations, transposed activations and gradients
    int train_cap = 0;
    gfx::DevBuf<float> Y, Z, w_part, b_part, lossp;
    gfx::DevBuf<uint16_t> H, Ht, D, Dt, dout;
    gfx::DevBuf<double> losses;
    int64_t adam_t = 0;
    hipStream_t stream = nullptr;
    ~gfx_mlp() {
        if (stream) (void)hipStreamDestroy(stream);
    }
};

namespace gfx {
namespace sur {
namespace {

constexpr int CHUNK = 131072;  // rows per pass of a forward call

// Widest padded layer input / output.
int wide(const gfx_mlp& M) { return std::max(pad64(M.n_feat), pad64(M.cfg.width)); }

void ensure_rows(gfx_mlp& M, int rows) {
    if (rows <= M.cap) return;
    const int cap = (rows + 255) / 256 * 256;
    GFX_HIP(hipStreamSynchronize(M.stream));  // the old buffers may still be in use
    M.cap = 0;
    M.X.alloc(size_t(cap) * 4);
    M.out.alloc(size_t(cap) * NO);
    M.y.alloc(size_t(cap) * NO);
    M.raw.alloc(size_t(cap) * 4);
    M.tix.alloc(size_t(cap));
    M.ha.alloc(size_t(cap) * wide(M));
    M.hb.alloc(size_t(cap) * wide(M));
    M.ha.zero(M.stream);  // features past 2 n_freq stay zero
    M.hb.zero(M.stream);
    M.cap = cap;
}

// Row splits of the weight gradients: about a thousand workgroups, at least 256 rows each.
int grad_splits(const gfx_mlp& M, int rows) {
    int tiles = 0;
    for (size_t l = 0; l < M.lin_in.size(); ++l) tiles += ((M.lin_in[l] + 63) / 64) * ((M.lin_out[l] + 63) / 64);
    return std::max(1, std::min((1024 + tiles - 1) / tiles, rows / 256));
}

// Buffers of forward and backward over one batch of rows.
struct Train {
    int ldt;                        // padded rows
    std::vector<int64_t> z, h, ht;  // per layer input l: offsets of Z (l >= 1), H, Ht
    std::vector<int64_t> dt;        // per layer output: offset of Dt
};
Train train_layout(const gfx_mlp& M, int rows) {
    Train T;
    T.ldt = pad64(rows);
    int64_t z = 0, h = 0, ht = 0, dt = 0;
    for (size_t l = 0; l < M.lin_in.size(); ++l) {
        T.z.push_back(z);
        T.h.push_back(h);
        T.ht.push_back(ht);
        T.dt.push_back(dt);
        z += int64_t(T.ldt) * pad64(M.lin_in[l]);
        h += int64_t(T.ldt) * pad64(M.lin_in[l]);
        ht += int64_t(T.ldt) * M.lin_in[l];
        dt += int64_t(T.ldt) * M.lin_out[l];
    }
    T.z.push_back(z);
    T.h.push_back(h);
    T.ht.push_back(ht);
    T.dt.push_back(dt);
    return T;
}

void ensure_train(gfx_mlp& M, int rows) {
    ensure_rows(M, rows);
    if (rows == M.train_cap) return;  // leading dimensions belong to the batch size
    GFX_HIP(hipStreamSynchronize(M.stream));
    M.train_cap = 0;
    const Train T = train_layout(M, rows);
    M.Y.alloc(size_t(rows) * NO);
    M.Z.alloc(T.z.back());
    M.H.alloc(T.h.back());
    M.Ht.alloc(T.ht.back());
    M.D.alloc(size_t(2) * T.ldt * pad64(M.cfg.width));
    M.Dt.alloc(T.dt.back());
    M.H.zero(M.stream);  // padding columns stay zero
    M.D.zero(M.stream);
    M.w_part.alloc(size_t(grad_splits(M, rows)) * M.n_params);
    M.b_part.alloc(size_t(T.ldt / 64) * (size_t(M.cfg.width) * M.cfg.depth + NO));
    M.dout.alloc(size_t(T.ldt) * pad64(NO));
    M.dout.zero(M.stream);
    M.lossp.alloc((rows + MSE_ROWS - 1) / MSE_ROWS);
    M.train_cap = rows;
}

// One product, 128 x 128 tiles where they give every CU two workgroups, else 64 x 64:
// a layer of 256 units over 131,072 rows takes 61 us in tiles of 128 and 66 in
// tiles of 64; over 8,192 rows tiles of 128 would be 128 workgroups for 256 CUs.
template <int EPI>
int gemm(gfx_mlp& M, const GemmArgs& G) {
    const int big = ((G.M + 127) / 128) * ((G.N + 127) / 128);
    if (big >= 512) {
        k_gemm<EPI, 128><<<dim3((G.N + 127) / 128, (G.M + 127) / 128), 256, 0, M.stream>>>(G);
        return 128;
    }
    k_gemm<EPI, 64><<<dim3((G.N + 63) / 64, (G.M + 63) / 64), 256, 0, M.stream>>>(G);
    return 64;
}

void features(gfx_mlp& M, int rows, uint16_t* H, uint16_t* Ht, int ldt) {
    const int nf = M.cfg.n_freq;
    const int n = Ht ? ldt : rows;
    k_fourier<<<dim3((n + 63) / 64, (nf + 31) / 32), 256, 0, M.stream>>>(M.X.p, rows, M.Bf.p, nf, H,
                                                                                     pad64(M.n_feat), Ht, ldt);
}

// forward of rows scaled inputs in M.X; output (scaled) in M.out
void forward(gfx_mlp& M, int rows) {
    uint16_t *in = M.ha.p, *next = M.hb.p;
    features(M, rows, in, nullptr, 0);
    const int d = M.cfg.depth;
    for (int l = 0; l <= d; ++l) {
        GemmArgs G{};
        G.A = in;
        G.lda = G.ldb = G.K = pad64(M.lin_in[l]);
        G.B = M.copies.p + M.layers.wt[l];
        G.M = rows;
        G.N = M.lin_out[l];
        G.bias = M.w.p + M.b_off[l];
        if (l == d) {
            G.out = M.out.p;
            gemm<EPI_OUT>(M, G);
        } else {
            G.H = next;
            G.ldh = pad64(M.lin_out[l]);
            gemm<EPI_HIDDEN>(M, G);
            std::swap(in, next);
        }
    }
    GFX_HIP(hipGetLastError());
}

// Forward and backward of the batch in M.X, M.Y: gradient into M.g, loss (mean
// over rows x n_out of the squared scaled error) into *loss on the device.
void gradient(gfx_mlp& M, int rows, double* loss) {
    const Train T = train_layout(M, rows);
    const int d = M.cfg.depth;
    features(M, rows, M.H.p, M.Ht.p, T.ldt);
    for (int l = 0; l <= d; ++l) {
        GemmArgs G{};
        G.A = M.H.p + T.h[l];
        G.lda = G.ldb = G.K = pad64(M.lin_in[l]);
        G.B = M.copies.p + M.layers.wt[l];
        G.M = rows;
        G.N = M.lin_out[l];
        G.bias = M.w.p + M.b_off[l];
        if (l == d) {
            G.out = M.out.p;
            gemm<EPI_OUT>(M, G);
        } else {
            G.Z = M.Z.p + T.z[l + 1];
            G.ldz = pad64(M.lin_out[l]);
            G.H = M.H.p + T.h[l + 1];
            G.ldh = pad64(M.lin_out[l]);
            G.Ht = M.Ht.p + T.ht[l + 1];
            G.ldt = T.ldt;
            gemm<EPI_HIDDEN>(M, G);
        }
    }
    // bias sums: one row per row tile, layer after layer
    ReduceArgs R{};
    R.n = d + 1;
    R.splits = grad_splits(M, rows);
    int64_t bp = 0, wp = 0;
    uint16_t *dcur = M.D.p, *dnext = M.D.p + int64_t(T.ldt) * pad64(M.cfg.width);
    const int64_t n = int64_t(rows) * NO;
    const int mb = (rows + MSE_ROWS - 1) / MSE_ROWS;
    k_mse<<<mb, MSE_ROWS, 0, M.stream>>>(M.out.p, M.Y.p, rows, 1.f / float(n), M.dout.p, pad64(NO), M.Dt.p + T.dt[d],
                                         T.ldt, M.b_part.p, M.lossp.p);
    k_loss<<<1, 64, 0, M.stream>>>(M.lossp.p, mb, 1.0 / double(n), loss);
    R.b_part[d] = 0;
    R.tiles[d] = mb;
    bp = int64_t(mb) * NO;
    const uint16_t* grad = M.dout.p;
    for (int l = d; l >= 1; --l) {  // dZ_{l-1} = (dZ_l W_l^T) gelu'(Z_{l-1})
        GemmArgs G{};
        G.A = grad;
        G.lda = G.ldb = G.K = pad64(M.lin_out[l]);
        G.B = M.copies.p + M.layers.wn[l];
        G.M = rows;
        G.N = M.lin_in[l];
        G.Z = M.Z.p + T.z[l];
        G.ldz = pad64(M.lin_in[l]);
        G.H = l > 1 ? dcur : nullptr;
        G.ldh = pad64(M.lin_in[l]);
        G.Ht = M.Dt.p + T.dt[l - 1];
        G.ldt = T.ldt;
        G.out = M.b_part.p + bp;
        const int tile = gemm<EPI_BACK>(M, G);
        R.b_part[l - 1] = bp;
        R.tiles[l - 1] = (rows + tile - 1) / tile;
        bp += int64_t(R.tiles[l - 1]) * M.lin_in[l];
        grad = dcur;
        std::swap(dcur, dnext);
    }
    GradArgs W{};
    W.n = d + 1;
    W.kc = (T.ldt / 64 + R.splits - 1) / R.splits * 64;
    R.splits = (T.ldt + W.kc - 1) / W.kc;
    int tiles = 0, blocks = 0;
    for (int l = 0; l <= d; ++l) {
        GemmArgs& G = W.g[l];
        G.A = M.Ht.p + T.ht[l];
        G.B = M.Dt.p + T.dt[l];
        G.lda = G.ldb = G.K = T.ldt;
        G.M = M.lin_in[l];
        G.N = M.lin_out[l];
        G.out = M.w_part.p + wp;
        W.tile0[l] = tiles;
        tiles += ((G.M + 63) / 64) * ((G.N + 63) / 64);
        R.w_off[l] = M.w_off[l];
        R.w_part[l] = wp;
        R.size[l] = G.M * G.N;
        R.cols[l] = G.N;
        R.blk0[l] = blocks;
        blocks += (R.size[l] + G.N + 63) / 64;
        wp += int64_t(R.splits) * R.size[l];
    }
    W.tile0[d + 1] = tiles;
    k_gemm_grads<<<dim3(tiles, R.splits), 256, 0, M.stream>>>(W);
    k_reduce_grads<<<blocks, 256, 0, M.stream>>>(R, M.w_part.p, M.b_part.p, M.g.p);
    GFX_HIP(hipGetLastError());
}

// BF16 copies of the weights after they changed outside Adam.
void round_weights(gfx_mlp& M) {
    k_round_weights<<<int((M.n_params + 255) / 256), 256, 0, M.stream>>>(M.w.p, M.n_params, M.layers, M.copies.p);
    GFX_HIP(hipGetLastError());
}

void adam(gfx_mlp& M, float lr) {
    ++M.adam_t;
    const float b1 = M.cfg.beta1, b2 = M.cfg.beta2;
    const float c1 = 1.f - std::pow(b1, float(M.adam_t)), c2 = 1.f - std::pow(b2, float(M.adam_t));
    sur::k_adam<<<int((M.n_params + 255) / 256), 256, 0, M.stream>>>(M.w.p, M.g.p, M.m.p, M.v.p, M.n_params,
                                                                      lr, b1, b2, M.cfg.eps, c1, c2, M.layers,
                                                                      M.copies.p);
}

}  // namespace
}  // namespace sur
}  // namespace gfx

using namespace gfx;

// ------------------------------ C ABI: tiles -------------------------------

extern "C" gfx_status gfx_green_create(int n_time, int n_node, const double* node_xyz, int n_cell,
                                       const int32_t* cell_node_index, gfx_green** out) {
    return guarded([&] {
        require(out && node_xyz && cell_node_index, "null argument");
        require(n_time >= 1 && n_node >= 1 && n_cell >= 1, "empty tile");
        *out = nullptr;
        auto G = std::make_unique<gfx_green>();
        G->n_time = n_time;
        G->n_node = n_node;
        G->n_cell = n_cell;
        G->h_xyz.assign(node_xyz, node_xyz + size_t(n_node) * 3);
        G->h_cell.assign(cell_node_index, cell_node_index + size_t(n_cell) * sur::NP);
        for (int32_t k : G->h_cell) require(k >= 0 && k < n_node, "cell node index out of range");
        // corner boxes (gll_interpolator.py:80-105)
        const int corner[8] = {0, 4, 20, 24, 100, 104, 120, 124};
        G->h_box.resize(size_t(n_cell) * 6);
        double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
        double ext[3] = {0, 0, 0};
        for (int c = 0; c < n_cell; ++c) {
            double* b = &G->h_box[size_t(c) * 6];
            for (int d = 0; d < 3; ++d) {
                b[2 * d] = 1e300;
                b[2 * d + 1] = -1e300;
            }
            for (int k : corner) {
                const double* x = &G->h_xyz[size_t(G->h_cell[size_t(c) * sur::NP + k]) * 3];
                for (int d = 0; d < 3; ++d) {
                    b[2 * d] = std::min(b[2 * d], x[d]);
                    b[2 * d + 1] = std::max(b[2 * d + 1], x[d]);
                }
            }
            for (int d = 0; d < 3; ++d) {
                lo[d] = std::min(lo[d], b[2 * d]);
                hi[d] = std::max(hi[d], b[2 * d + 1]);
                ext[d] = std::max(ext[d], b[2 * d + 1] - b[2 * d]);
            }
        }
        // bins about one cell wide
        for (int d = 0; d < 3; ++d) {
            const double span = std::max(hi[d] - lo[d], 1e-9);
            G->nb[d] = std::max(1, std::min(4096, int(span / std::max(ext[d], 1e-9))));
            G->b0[d] = lo[d] - 2 * sur::EXACT_TOL;
            G->bh[d] = (span + 4 * sur::EXACT_TOL) / G->nb[d];
        }
        const int64_t nbins = int64_t(G->nb[0]) * G->nb[1] * G->nb[2];
        std::vector<std::vector<int32_t>> bins(nbins);
        for (int c = 0; c < n_cell; ++c) {
            const double* b = &G->h_box[size_t(c) * 6];
            int r0[3], r1[3];
            for (int d = 0; d < 3; ++d) {
                r0[d] = std::max(0, int(std::floor((b[2 * d] - sur::EXACT_TOL - G->b0[d]) / G->bh[d])));
                r1[d] = std::min(G->nb[d] - 1, int(std::floor((b[2 * d + 1] + sur::EXACT_TOL - G->b0[d]) / G->bh[d])));
            }
            for (int z = r0[2]; z <= r1[2]; ++z)
                for (int y = r0[1]; y <= r1[1]; ++y)
                    for (int x = r0[0]; x <= r1[0]; ++x)
                        bins[(int64_t(z) * G->nb[1] + y) * G->nb[0] + x].push_back(c);
        }
        std::vector<int32_t> off(nbins + 1, 0), cells;
        for (int64_t b = 0; b < nbins; ++b) {
            off[b + 1] = off[b] + int32_t(bins[b].size());
            cells.insert(cells.end(), bins[b].begin(), bins[b].end());
        }
        GFX_HIP(hipStreamCreateWithFlags(&G->stream, hipStreamNonBlocking));
        G->val.alloc(size_t(n_time) * n_node * 18);
        G->val.zero(G->stream);
        G->cell_idx.upload(G->h_cell);
        G->xyz.upload(G->h_xyz);
        G->box.upload(G->h_box);
        G->bin_off.upload(off);
        G->bin_cell.upload(cells);
        GFX_HIP(hipStreamSynchronize(G->stream));
        *out = G.release();
    });
}

extern "C" gfx_status gfx_green_destroy(gfx_green* g) {
    return guarded([&] { delete g; });
}

extern "C" gfx_status gfx_green_set_values(gfx_green* g, int t, const float* v) {
    return guarded([&] {
        require(g && v, "null argument");
        require(t >= 0 && t < g->n_time, "time index out of range");
        GFX_HIP(hipMemcpy(g->val.p + int64_t(t) * g->n_node * 18, v, size_t(g->n_node) * 18 * 4,
                          hipMemcpyHostToDevice));
    });
}

extern "C" gfx_status gfx_green_get_values(const gfx_green* g, int t, float* v) {
    return guarded([&] {
        require(g && v, "null argument");
        require(t >= 0 && t < g->n_time, "time index out of range");
        GFX_HIP(hipStreamSynchronize(g->stream));
        GFX_HIP(hipMemcpy(v, g->val.p + int64_t(t) * g->n_node * 18, size_t(g->n_node) * 18 * 4,
                          hipMemcpyDeviceToHost));
    });
}

extern "C" gfx_status gfx_green_interpolate(const gfx_green* g, int n, const double* xyz, const int32_t* tix,
                                            float* out, int32_t* cell) {
    return guarded([&] {
        require(g && xyz && tix && out && n >= 0, "null argument");
        if (n == 0) return;
        std::lock_guard<std::mutex> lock(g->work_mu);
        gfx_green::Work& w = g->work;
        struct Trim {
            gfx_green::Work& w;
            ~Trim() { w.trim(); }
        } trim{w};  // also when the call fails
        w.fit(n);
        GFX_HIP(hipMemcpyAsync(w.q.p, xyz, size_t(n) * 24, hipMemcpyHostToDevice, g->stream));
        GFX_HIP(hipMemcpyAsync(w.t.p, tix, size_t(n) * 4, hipMemcpyHostToDevice, g->stream));
        sur::k_judge<<<sur::judge_blocks(n), 64 * sur::JQ, 0, g->stream>>>(
            sur::judge_args(*g), n, sur::judge_q(n), w.q.p, w.t.p, nullptr, 1, w.o.p, cell ? w.c.p : nullptr, nullptr);
        GFX_HIP(hipGetLastError());
        GFX_HIP(hipMemcpyAsync(out, w.o.p, size_t(n) * 18 * 4, hipMemcpyDeviceToHost, g->stream));
        if (cell) GFX_HIP(hipMemcpyAsync(cell, w.c.p, size_t(n) * 4, hipMemcpyDeviceToHost, g->stream));
        GFX_HIP(hipStreamSynchronize(g->stream));
    });
}

// Host FP64 restatement of GLLInterpolator.interpolate for one point over
// node values [n_node][nv]; returns GFX_ERR_INVALID when the point lies
// outside all cells (the reference raises ValueError).
extern "C" gfx_status gfx_gll_interpolate_host(int n_node, const double* node_xyz, int n_cell,
                                               const int32_t* cell_node_index, int nv, const double* values,
                                               const double* point, double* out) {
    return guarded([&] {
        require(node_xyz && cell_node_index && values && point && out && nv >= 1, "null argument");
        const double p[3] = {point[0], point[1], point[2]};
        // exact-node shortcut over all nodes
        int best_node = -1;
        double bd = 1e300;
        for (int k = 0; k < n_node; ++k) {
            const double* x = node_xyz + size_t(k) * 3;
            const double dd = (x[0] - p[0]) * (x[0] - p[0]) + (x[1] - p[1]) * (x[1] - p[1]) + (x[2] - p[2]) * (x[2] - p[2]);
            if (dd < bd) {
                bd = dd;
                best_node = k;
            }
        }
        if (best_node >= 0 && std::sqrt(bd) < sur::EXACT_TOL) {
            std::memcpy(out, values + size_t(best_node) * nv, size_t(nv) * 8);
            return;
        }
        const int corner[8] = {0, 4, 20, 24, 100, 104, 120, 124};
        int cell = -1;
        double cdist = 1e300, cb[6] = {0, 0, 0, 0, 0, 0};
        for (int c = 0; c < n_cell; ++c) {
            double b[6] = {1e300, -1e300, 1e300, -1e300, 1e300, -1e300};
            for (int k : corner) {
                const double* x = node_xyz + size_t(cell_node_index[size_t(c) * sur::NP + k]) * 3;
                for (int d = 0; d < 3; ++d) {
                    b[2 * d] = std::min(b[2 * d], x[d]);
                    b[2 * d + 1] = std::max(b[2 * d + 1], x[d]);
                }
            }
            bool in = true;
            for (int d = 0; d < 3; ++d)
                in = in && p[d] >= b[2 * d] - sur::EXACT_TOL && p[d] <= b[2 * d + 1] + sur::EXACT_TOL;
            if (!in) continue;
            double dd = 0;
            for (int d = 0; d < 3; ++d) dd += (0.5 * (b[2 * d] + b[2 * d + 1]) - p[d]) * (0.5 * (b[2 * d] + b[2 * d + 1]) - p[d]);
            if (dd < cdist) {
                cdist = dd;
                cell = c;
                std::memcpy(cb, b, sizeof(b));
            }
        }
        if (cell < 0) throw Error(GFX_ERR_INVALID, "query point is outside all recording cells");
        double xi[3], l[3][5];
        for (int d = 0; d < 3; ++d) {
            xi[d] = std::min(1.0, std::max(-1.0, 2.0 * (p[d] - cb[2 * d]) / (cb[2 * d + 1] - cb[2 * d]) - 1.0));
            sur::lagrange5(xi[d], l[d]);
        }
        double sw = 0;
        for (int a = 0; a < 5; ++a)
            for (int b = 0; b < 5; ++b)
                for (int k = 0; k < 5; ++k) sw += l[0][a] * l[1][b] * l[2][k];
        for (int m = 0; m < nv; ++m) out[m] = 0.0;
        for (int a = 0; a < 5; ++a)
            for (int b = 0; b < 5; ++b)
                for (int k = 0; k < 5; ++k) {
                    const double w = l[0][a] * l[1][b] * l[2][k] / sw;
                    const double* v = values + size_t(cell_node_index[size_t(cell) * sur::NP + (a * 5 + b) * 5 + k]) * nv;
                    for (int m = 0; m < nv; ++m) out[m] += w * v[m];
                }
    });
}

// ------------------------------ C ABI: MLP ---------------------------------

extern "C" gfx_status gfx_mlp_config_default(gfx_mlp_config* c) {
    return guarded([&] {
        require(c != nullptr, "null argument");
        *c = gfx_mlp_config{};
        c->n_freq = 64;
        c->width = 256;
        c->depth = 6;
        c->n_out = 18;
        c->sigma = 2.0f;
        c->seed = 5;
        c->lr = 1e-3f;
        c->beta1 = 0.9f;
        c->beta2 = 0.999f;
        c->eps = 1e-8f;
        c->batch = 8192;
        c->lr_final = 5e-5f;
    });
}

extern "C" gfx_status gfx_mlp_create(const gfx_mlp_config* cfg, const double* in_lo, const double* in_hi,
                                     const double* out_scale, gfx_mlp** out) {
    return guarded([&] {
        require(cfg && in_lo && in_hi && out_scale && out, "null argument");
        require(cfg->n_freq >= 1 && cfg->n_freq <= 1024 && cfg->width >= 16 && cfg->width <= 4096 &&
                    cfg->depth >= 1 && cfg->depth <= 32 && cfg->n_out == 18,
                "bad MLP shape (n_out must be 18: 6 strain components x 3 force directions)");
        for (int d = 0; d < 4; ++d) require(in_hi[d] > in_lo[d], "input range must be non-empty");
        require(cfg->lr > 0 && cfg->lr_final > 0 && cfg->lr_final <= cfg->lr, "need 0 < lr_final <= lr");
        *out = nullptr;
        auto M = std::make_unique<gfx_mlp>();
        M->cfg = *cfg;
        M->n_feat = 2 * cfg->n_freq;
        int iw = M->n_feat;
        for (int l = 0; l <= cfg->depth; ++l) {
            const int ow = (l == cfg->depth) ? cfg->n_out : cfg->width;
            M->lin_in.push_back(iw);
            M->lin_out.push_back(ow);
            M->w_off.push_back(M->n_params);
            M->n_params += int64_t(iw) * ow;
            M->b_off.push_back(M->n_params);
            M->n_params += ow;
            iw = ow;
        }
        // init: weights U(-sqrt(6/(in+out)), ...) (Glorot), biases 0, B ~ N(0, sigma^2)
        std::mt19937_64 rng(cfg->seed);
        std::vector<float> hw(M->n_params, 0.f);
        for (size_t l = 0; l < M->lin_in.size(); ++l) {
            const double a = std::sqrt(6.0 / (M->lin_in[l] + M->lin_out[l]));
            std::uniform_real_distribution<double> U(-a, a);
            for (int64_t i = 0; i < int64_t(M->lin_in[l]) * M->lin_out[l]; ++i) hw[M->w_off[l] + i] = float(U(rng));
        }
        std::normal_distribution<double> Nd(0.0, cfg->sigma);
        std::vector<float> hb(size_t(cfg->n_freq) * 4);
        for (auto& x : hb) x = float(Nd(rng));
        GFX_HIP(hipStreamCreateWithFlags(&M->stream, hipStreamNonBlocking));
        M->w.upload(hw);
        M->g.alloc(M->n_params);
        M->m.alloc(M->n_params);
        M->v.alloc(M->n_params);
        M->m.zero(M->stream);
        M->v.zero(M->stream);
        M->Bf.upload(hb);
        {
            int64_t at = 0;
            M->layers.n = int(M->lin_in.size());
            for (int l = 0; l < M->layers.n; ++l) {
                sur::Layers& Y = M->layers;
                Y.w_off[l] = M->w_off[l];
                Y.b_off[l] = M->b_off[l];
                Y.in[l] = M->lin_in[l];
                Y.out[l] = M->lin_out[l];
                Y.wt[l] = at;
                at += int64_t(Y.out[l]) * sur::pad64(Y.in[l]);
                Y.wn[l] = at;
                at += int64_t(Y.in[l]) * sur::pad64(Y.out[l]);
            }
            M->copies.alloc(at);
            M->copies.zero(M->stream);  // padding stays zero
            sur::round_weights(*M);
        }
        M->lo.upload(std::vector<double>(in_lo, in_lo + 4));
        M->hi.upload(std::vector<double>(in_hi, in_hi + 4));
        M->h_scale.assign(out_scale, out_scale + 18);
        M->scale.upload(M->h_scale);
        std::vector<float> inv(18);
        for (int k = 0; k < 18; ++k) {
            require(out_scale[k] > 0, "output scales must be > 0");
            inv[k] = float(1.0 / out_scale[k]);
        }
        M->inv_scale.upload(inv);
        GFX_HIP(hipStreamSynchronize(M->stream));
        *out = M.release();
    });
}

extern "C" gfx_status gfx_mlp_destroy(gfx_mlp* m) {
    return guarded([&] { delete m; });
}

extern "C" gfx_status gfx_mlp_n_params(const gfx_mlp* m, size_t* n) {
    return guarded([&] {
        require(m && n, "null argument");
        *n = size_t(m->n_params);
    });
}

extern "C" gfx_status gfx_mlp_get_params(const gfx_mlp* m, float* w, size_t n, float* fourier) {
    return guarded([&] {
        require(m && w && n == size_t(m->n_params), "parameter buffer must hold n_params floats");
        GFX_HIP(hipStreamSynchronize(m->stream));
        GFX_HIP(hipMemcpy(w, m->w.p, n * 4, hipMemcpyDeviceToHost));
        if (fourier) GFX_HIP(hipMemcpy(fourier, m->Bf.p, size_t(m->cfg.n_freq) * 16, hipMemcpyDeviceToHost));
    });
}

extern "C" gfx_status gfx_mlp_set_params(gfx_mlp* m, const float* w, size_t n) {
    return guarded([&] {
        require(m && w && n == size_t(m->n_params), "parameter buffer must hold n_params floats");
        GFX_HIP(hipStreamSynchronize(m->stream));
        GFX_HIP(hipMemcpy(m->w.p, w, n * 4, hipMemcpyHostToDevice));
        sur::round_weights(*m);
    });
}

extern "C" gfx_status gfx_mlp_set_envelope(gfx_mlp* m, double cx, double cy, double slowness, double r_max,
                                           int n_bins, const float* env) {
    return guarded([&] {
        require(m != nullptr, "null argument");
        require(n_bins >= 0 && n_bins <= 65536, "n_bins must be in [0, 65536]");
        require(std::isfinite(slowness) && slowness >= 0, "slowness must be >= 0");
        GFX_HIP(hipStreamSynchronize(m->stream));
        m->env_cx = cx;
        m->env_cy = cy;
        m->slowness = slowness;
        if (n_bins == 0) {
            m->h_env.clear();
            m->env.release();
            return;
        }
        require(env != nullptr && r_max > 0, "envelope needs knots and r_max > 0");
        for (int i = 0; i < n_bins; ++i) require(env[i] > 0.f && std::isfinite(env[i]), "envelope knots must be > 0");
        m->h_env.assign(env, env + n_bins);
        m->env.upload(m->h_env);
        m->env_rmax = r_max;
    });
}

// inputs raw (x, y, z, t) [n][4] FP64; outputs unscaled [n][18]
extern "C" gfx_status gfx_mlp_forward(gfx_mlp* m, int n, const double* x, float* y) {
    return guarded([&] {
        require(m && x && y && n >= 0, "null argument");
        const sur::Envelope E = m->envelope(true);
        for (int b = 0; b < n; b += sur::CHUNK) {
            const int rows = std::min(sur::CHUNK, n - b);
            sur::ensure_rows(*m, rows);
            GFX_HIP(hipMemcpyAsync(m->raw.p, x + size_t(b) * 4, size_t(rows) * 32, hipMemcpyHostToDevice, m->stream));
            sur::k_inputs<<<(rows + 255) / 256, 256, 0, m->stream>>>(m->raw.p, nullptr, 0.0, 0.0, rows, m->lo.p, m->hi.p,
                                                                     E, m->X.p);
            sur::forward(*m, rows);
            sur::k_outputs<<<(rows * sur::NO + 255) / 256, 256, 0, m->stream>>>(m->out.p, m->raw.p, 4, rows, m->scale.p,
                                                                               E, m->y.p);
            GFX_HIP(hipGetLastError());
            GFX_HIP(hipMemcpyAsync(y + size_t(b) * 18, m->y.p, size_t(rows) * 72, hipMemcpyDeviceToHost, m->stream));
        }
        GFX_HIP(hipStreamSynchronize(m->stream));
    });
}

// Gradient of the scaled MSE for given samples (checking against a CPU model):
// x raw [n][4] FP64, y unscaled targets [n][18]; grad [n_params]
extern "C" gfx_status gfx_mlp_gradient(gfx_mlp* m, int n, const double* x, const float* y, float* grad,
                                       double* loss) {
    return guarded([&] {
        require(m && x && y && grad && loss && n >= 1, "null argument");
        sur::ensure_train(*m, n);
        GFX_HIP(hipStreamSynchronize(m->stream));
        GFX_HIP(hipMemcpy(m->raw.p, x, size_t(n) * 32, hipMemcpyHostToDevice));
        std::vector<float> ys(size_t(n) * 18);
        const sur::Envelope E = m->envelope(false);
        for (int r = 0; r < n; ++r) {
            const double e = sur::envelope_at(E, x[size_t(r) * 4], x[size_t(r) * 4 + 1]);
            for (int k = 0; k < 18; ++k) ys[size_t(r) * 18 + k] = float(y[size_t(r) * 18 + k] / (m->h_scale[k] * e));
        }
        GFX_HIP(hipMemcpy(m->Y.p, ys.data(), ys.size() * 4, hipMemcpyHostToDevice));
        if (m->losses.n < 1) m->losses.alloc(1);
        sur::k_inputs<<<(n + 255) / 256, 256, 0, m->stream>>>(m->raw.p, nullptr, 0.0, 0.0, n, m->lo.p, m->hi.p,
                                                              m->envelope(true), m->X.p);
        sur::gradient(*m, n, m->losses.p);
        GFX_HIP(hipStreamSynchronize(m->stream));
        GFX_HIP(hipMemcpy(loss, m->losses.p, sizeof(double), hipMemcpyDeviceToHost));
        GFX_HIP(hipMemcpy(grad, m->g.p, size_t(m->n_params) * 4, hipMemcpyDeviceToHost));
    });
}

// Adam training on random (node, time) samples of a tile; the tile's time
// index k maps to t = t0 + k * dt.  *loss receives the mean scaled loss of the
// last 10 % of the iterations.
extern "C" gfx_status gfx_mlp_train(gfx_mlp* m, const gfx_green* g, double t0, double dt, int iters, uint64_t seed,
                                    double* loss) {
    return guarded([&] {
        require(m && g && loss && iters >= 0, "null argument");
        const int rows = m->cfg.batch;
        require(rows >= 64, "batch must be >= 64");
        sur::ensure_train(*m, rows);
        GFX_HIP(hipStreamSynchronize(g->stream));
        if (m->losses.n < size_t(std::max(iters, 1))) {
            GFX_HIP(hipStreamSynchronize(m->stream));
            m->losses.alloc(std::max(iters, 1));
        }
        const sur::Envelope E = m->envelope(true);
        const double lr0 = m->cfg.lr, lr1 = m->cfg.lr_final;
        for (int it = 0; it < iters; ++it) {
            sur::k_sample_tile<<<(rows + 255) / 256, 256, 0, m->stream>>>(
                g->val.p, g->xyz.p, g->n_node, g->n_time, t0, dt, m->lo.p, m->hi.p, m->inv_scale.p, E,
                seed * 0x9E3779B97F4A7C15ULL + uint64_t(it), rows, m->X.p, m->Y.p);
            sur::gradient(*m, rows, m->losses.p + it);
            // cosine decay from lr to lr_final over this call
            const double ph = iters > 1 ? double(it) / double(iters - 1) : 1.0;
            sur::adam(*m, float(lr1 + 0.5 * (lr0 - lr1) * (1.0 + std::cos(3.14159265358979323846 * ph))));
        }
        GFX_HIP(hipStreamSynchronize(m->stream));
        const int nt = iters > 0 ? std::max(1, iters / 10) : 0;
        std::vector<double> tail(nt);
        if (nt)
            GFX_HIP(hipMemcpy(tail.data(), m->losses.p + (iters - nt), nt * sizeof(double), hipMemcpyDeviceToHost));
        double sum = 0.0;
        for (double l : tail) sum += l;
        *loss = nt ? sum / nt : 0.0;
    });
}

// Surrogate query: the MLP everywhere, the judge for points in (cell, time
// window) regions marked for fallback (or outside the tile).  *n_fallback
// counts judge answers.
extern "C" gfx_status gfx_surrogate_query(gfx_mlp* m, const gfx_green* g, const uint8_t* fallback, int n_window,
                                          double t0, double dt, int n, const double* xyz, const int32_t* tix,
                                          float* out, int* n_fallback) {
    return guarded([&] {
        require(m && g && fallback && xyz && tix && out && n_fallback && n >= 0, "null argument");
        require(n_window >= 1 && n_window <= g->n_time, "n_window must be in [1, n_time]");
        if (n == 0) {
            *n_fallback = 0;
            return;
        }
        const size_t nreg = size_t(g->n_cell) * n_window;
        GFX_HIP(hipStreamSynchronize(g->stream));  // the tile's values are in place
        if (m->policy.n < nreg) {
            GFX_HIP(hipStreamSynchronize(m->stream));
            m->policy.alloc(nreg);
        }
        if (m->count.n < 1) m->count.alloc(1);
        GFX_HIP(hipMemcpyAsync(m->policy.p, fallback, nreg, hipMemcpyHostToDevice, m->stream));
        m->count.zero(m->stream);
        const sur::Envelope E = m->envelope(true);
        for (int b = 0; b < n; b += sur::CHUNK) {
            const int rows = std::min(sur::CHUNK, n - b);
            sur::ensure_rows(*m, rows);
            GFX_HIP(hipMemcpyAsync(m->raw.p, xyz + size_t(b) * 3, size_t(rows) * 24, hipMemcpyHostToDevice, m->stream));
            GFX_HIP(hipMemcpyAsync(m->tix.p, tix + b, size_t(rows) * 4, hipMemcpyHostToDevice, m->stream));
            sur::k_inputs<<<(rows + 255) / 256, 256, 0, m->stream>>>(m->raw.p, m->tix.p, t0, dt, rows, m->lo.p, m->hi.p, E,
                                                                     m->X.p);
            sur::forward(*m, rows);
            sur::k_outputs<<<(rows * sur::NO + 255) / 256, 256, 0, m->stream>>>(m->out.p, m->raw.p, 3, rows, m->scale.p,
                                                                               E, m->y.p);
            // the judge's answers, and zeros, over the network's
            sur::k_judge<<<sur::judge_blocks(rows), 64 * sur::JQ, 0, m->stream>>>(
                sur::judge_args(*g), rows, sur::judge_q(rows), m->raw.p, m->tix.p, m->policy.p, n_window, m->y.p, nullptr, m->count.p);
            GFX_HIP(hipGetLastError());
            GFX_HIP(hipMemcpyAsync(out + size_t(b) * 18, m->y.p, size_t(rows) * 72, hipMemcpyDeviceToHost, m->stream));
        }
        GFX_HIP(hipMemcpyAsync(n_fallback, m->count.p, sizeof(int), hipMemcpyDeviceToHost, m->stream));
        GFX_HIP(hipStreamSynchronize(m->stream));
    });
}
