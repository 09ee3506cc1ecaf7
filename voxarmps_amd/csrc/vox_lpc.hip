// vox_lpc.hip — learned PPE preconditioner on gfx950: a message-passing
// network over the PPE matrix graph, its training on the GPU, and the
// coupling operator it parameterises for flexible CG (vox_cg.hip).
//
// No reference code: the reference solves the PPE with IC(0)-CG only
// (functions.cu:1139-1200, 506-716). The preconditioner is
//   z_r = g_r w_r / A_rr + sqrt(c_r) sum_{k in S(r)} O_rk / (A_rr A_kk) sqrt(c_k) w_k
// with O = -offdiag(A) >= 0 and S the strong couplings O_rk >= theta * O_ref
// (O_ref the coupling of two particles one spacing apart, theta = 0.25: a
// symmetric pattern, about the neighbours within 2.3 spacings). g = c = 1 is
// the Neumann series D^-1 + D^-1 O_S D^-1 truncated after one term on S; the
// network sets g and c per unknown from local features.
//
// Network (per unknown r, hidden 64, messages 16; bf16 operands on the matrix
// cores, FP32 accumulation; weights packed as in voxarmps.h):
//   h0 = relu(W0 f + b0)
//   for l = 1..3: s = P_l h_{l-1};  m_r = (sum_k O_rk s_k) / sum_k O_rk
//                 h_l = relu(U_l h_{l-1} + V_l m + c_l)
//   o = Wo h3 + bo;  g = exp(0.5 tanh o0);  c = 2.5 sigmoid(o1 - ln 1.5)
// Features f: n_r/n0, wall flag, sum_k O_rk / A_rr, the first moments
// sum_k O_rk (x_k - x_r) / re / sum_k O_rk (three axes), 0, 0.
//
// Layout: rows of activations are contiguous (64 bf16 = 128 bytes of hidden
// state, 16 bf16 = 32 bytes of message per row), so the aggregation gathers
// one 32-byte message per matrix entry; matrix and coupling operator are
// SELL-64 (mx_index). The dense layers run one wavefront per 16-row tile:
// v_mfma_f32_16x16x32_bf16 with the weights held in registers for the whole
// launch, the 16 x 64 output tile staged in LDS for the coalesced store and
// for the message product that follows in the same kernel.
//
// Row walks take 4 or 8 lanes per row, each with its own channels (or probe, or
// moment): the lanes of a row read one gathered record side by side (one cache
// lookup instead of one a lane), every sum stays one chain in the row's order,
// and a system of a few thousand rows still fills the chip.
//
// Training (mean over probes w of ||A M w - w||^2 / ||w||^2, Adam): the four
// probes go through one walk of each operator, and the backward pass runs in
// FP32, its dense products and weight gradients on v_mfma_f32_16x16x4_f32, with
// weight gradients reduced in a fixed order (deterministic).
#include <algorithm>
#include <cstring>
#include <numeric>

#include "vox_internal.hpp"

namespace vox {

constexpr int LF = 8, LH = 64, LM = 16, LO = 2, LNL = 3;
constexpr int OFF_W0 = 0, OFF_B0 = OFF_W0 + LH * LF;
constexpr int LAYER_SZ = LM * LH + LH * LH + LH * LM + LH;
__host__ __device__ constexpr int off_P(int l) { return OFF_B0 + LH + (l - 1) * LAYER_SZ; }
__host__ __device__ constexpr int off_U(int l) { return off_P(l) + LM * LH; }
__host__ __device__ constexpr int off_V(int l) { return off_U(l) + LH * LH; }
__host__ __device__ constexpr int off_c(int l) { return off_V(l) + LH * LM; }
constexpr int OFF_WO = off_P(LNL + 1), OFF_BO = OFF_WO + LO * LH, NPARAM = OFF_BO + LO;
static_assert(NPARAM == VOX_LPC_NPARAM, "parameter count");
constexpr float kCMax = 2.5f;
constexpr float kBeta = -0.40546510810816438f;   // -ln(1.5): c = 1 at zero output
constexpr int kProbes = 4;
constexpr int kOuterBlocks = 256;

// ---- bf16 (round to nearest even; inputs are finite) -----------------------
__device__ __forceinline__ uint16_t f2bf(float x)
{
    uint32_t b = __float_as_uint(x);
    b += 0x7FFFu + ((b >> 16) & 1u);
    return (uint16_t)(b >> 16);
}
__device__ __forceinline__ float bf2f(uint32_t h) { return __uint_as_float(h << 16); }
__device__ __forceinline__ float bf_lo(int32_t x) { return __uint_as_float((uint32_t)x << 16); }
__device__ __forceinline__ float bf_hi(int32_t x) { return __uint_as_float((uint32_t)x & 0xFFFF0000u); }

__device__ __forceinline__ double rademacher(uint64_t seed, int probe, int r)
{
    uint64_t z = seed + ((uint64_t)probe << 32) + (uint64_t)(r + 1) * 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z = z ^ (z >> 31);
    return (z >> 63) ? -1.0 : 1.0;
}

// ---- row walks ---------------------------------------------------------------
// The first `len` entries of row r of a SELL-64 matrix in order: f(column, value,
// gathered) for each, gathered = get(column). U entries' gathers are in flight
// together, and the next U columns and values are loaded before they are used;
// loads past the row's end take its last entry again, so none sits in a branch.
// A wave's rows are of one slice, whose start is a scalar: a lane's offsets in it
// (256 bytes an entry) are 32 bits for column and value alike. With 64-bit
// addresses of each load, a third of the loop's instructions, the walks of 14.6k
// rows took 6 to 14 % longer. (Loads that leave no cache lines: 22 to 45 % slower,
// the four or eight lanes of a row then fetch an entry's line again.)
template <int U, class Get, class F>
__device__ __forceinline__ void walk_row(const int32_t* __restrict__ cols, const float* __restrict__ vals,
                                         int r, int cap, int len, Get get, F f)
{
    if (len <= 0) return;
    const long slice = mx_index((long)__builtin_amdgcn_readfirstlane(r >> 6) << 6, 0, cap);
    const char* __restrict__ col = reinterpret_cast<const char*>(cols + slice);
    const char* __restrict__ val = reinterpret_cast<const char*>(vals + slice);
    const uint32_t first = 4u * (r & 63), last = first + 256u * (uint32_t)(len - 1);
    int32_t c[U], cn[U];
    float v[U], vn[U];
    auto next = [&](int k) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t i = min(first + 256u * (uint32_t)(k + u), last);
            cn[u] = *reinterpret_cast<const int32_t*>(col + i);
            vn[u] = *reinterpret_cast<const float*>(val + i);
        }
    };
    decltype(get(0)) x[U];
    auto gather = [&]() {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            c[u] = cn[u];
            v[u] = vn[u];
            x[u] = get(c[u]);
        }
    };
    next(0);
    int k = 0;
    for (; k + U <= len; k += U) {
        gather();
        next(k + U);
#pragma unroll
        for (int u = 0; u < U; ++u) f(c[u], v[u], x[u]);
    }
    gather();
#pragma unroll
    for (int u = 0; u < U; ++u)
        if (k + u < len) f(c[u], v[u], x[u]);
}

// ---- features and strong couplings ------------------------------------------
// Per-row preparation: FP32 position of the unknown's particle, 1/A_rr, and
// the two features that need no neighbours (n/n0, wall flag); padding rows
// get zero features.
struct PrepArgs {
    int nu, rows, dim;
    double n0;
    const double* __restrict__ adiag;
    const int32_t* __restrict__ urow;
    const int32_t* __restrict__ ptype;
    const double *x, *y, *z, *pnd;
    v4f* upos;
    float* invd;
    float* feat;
};

__global__ __launch_bounds__(kBlock) void k_lpc_rowprep(PrepArgs a)
{
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= a.rows) return;
    float* f = a.feat + 8L * r;
    if (r >= a.nu) {
        for (int q = 0; q < 8; ++q) f[q] = 0.f;
        return;
    }
    const int i = a.urow[r];
    a.upos[r] = v4f{(float)a.x[i], (float)a.y[i], a.dim == 3 ? (float)a.z[i] : 0.f, 0.f};
    a.invd[r] = (float)(1.0 / a.adiag[r]);
    f[0] = (float)(a.pnd[i] / a.n0);
    f[1] = (a.ptype[i] == 0) ? 1.f : 0.f;
}

// Row sums over the FP32 off-diagonal magnitudes O_rk = -a_rk (sum and the
// first moments of the FP32 neighbour offsets: features 2..7), and the strong
// couplings O_rk >= thr of the row (column and O_rk, in matrix order).
struct FeatArgs {
    int nu, cap;
    float inv_re;
    float thr;                  // the smallest float not below the threshold
    const int32_t* __restrict__ rowlen;
    const int32_t* __restrict__ acol;
    const float* __restrict__ aval;
    const v4f* __restrict__ upos;
    const float* __restrict__ invd;
    float* feat;
    float* inv_osum;
    int32_t* slen;
    int32_t* scol;
    float* sval;
};

// Four lanes per row: x, y, z moments and the sum of magnitudes. Strong
// couplings wait in LDS for whole-line stores at the end (a wave's stores hold up
// its next gathers), written without a branch: an entry that is not strong is
// overwritten by the next. A row's 61st and later are stored as they come; a
// lattice has up to 56 within the threshold's distance, and 31 KB leave 5 blocks
// to a CU. 107k rows of 215 entries: 240 us (one thread per row), 254 (stores in
// the walk), 150 (a branch per strong entry), 135 (48 slots), 120.
constexpr int kStrongLds = 60;
__global__ __launch_bounds__(kBlock) void k_lpc_features(FeatArgs a)
{
    __shared__ uint32_t qs[kStrongLds + 1][kWave][2];  // column, value; the last slot is not read
    __shared__ int sn[kWave];
    const int q = threadIdx.x & 3, lr = threadIdx.x >> 2;
    const int row0 = xcd_block() * kWave, r = row0 + lr;
    if (r < a.nu) {
        const float* __restrict__ pos = reinterpret_cast<const float*>(a.upos);
        const float own = pos[4L * r + q];
        const long b = mx_index(r, 0, a.cap);
        uint32_t* __restrict__ out = (q & 1) ? reinterpret_cast<uint32_t*>(a.sval + b)
                                             : reinterpret_cast<uint32_t*>(a.scol + b);
        const int far = q < 2 ? kStrongLds : INT_MAX;  // lanes 2 and 3 hold 0's and 1's words
        float acc = 0.f;
        int n = 0;
        walk_row<8>(a.acol, a.aval, r, a.cap, a.rowlen[r], [&](int c) { return pos[4L * c + q]; },
                    [&](int c, float v, float x) {
                        const float o = -v;
                        acc = fmaf(o, q < 3 ? x - own : 1.f, acc);
                        const bool strong = o >= a.thr;
                        const uint32_t w = (q & 1) ? __float_as_uint(o) : (uint32_t)c;
                        qs[min(n, kStrongLds)][lr][q & 1] = w;
                        if (strong && n >= far) out[64L * n] = w;
                        n += strong;
                    });
        const float osum = __shfl(acc, 3, 4);
        const float inv = (osum > 0.f) ? 1.f / osum : 0.f;
        float* f = a.feat + 8L * r;
        if (q < 3) {
            f[3 + q] = acc * inv * a.inv_re;
            if (q < 2) f[6 + q] = 0.f;
        } else {
            a.slen[r] = n;
            f[2] = osum * a.invd[r];
            a.inv_osum[r] = inv;
        }
        if (q == 0) sn[lr] = min(n, kStrongLds);
    } else if (q == 0) {
        sn[lr] = 0;
    }
    __syncthreads();
    const int i = threadIdx.x & (kWave - 1), n = sn[i];
    const long b = mx_index(row0 + i, 0, a.cap);
    for (int k = threadIdx.x >> 6; k < n; k += kBlock / kWave) {
        a.scol[b + 64L * k] = (int32_t)qs[k][i][0];
        a.sval[b + 64L * k] = __uint_as_float(qs[k][i][1]);
    }
}

// Training-set coupling values: O_rk / (A_rr A_kk) as (O_rk * (1/A_rr)) * (1/A_kk).
__global__ __launch_bounds__(kBlock) void k_lpc_oh(int nu, int cap, const int32_t* __restrict__ slen,
                                                   const int32_t* __restrict__ scol,
                                                   const float* __restrict__ invd, float* sval)
{
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= nu) return;
    const long b = mx_index(r, 0, cap);
    const float ir = invd[r];
    for (int k = 0; k < slen[r]; ++k) sval[b + 64L * k] = (sval[b + 64L * k] * ir) * invd[scol[b + 64L * k]];
}

// FP64 -> FP32 right-hand side and diagonal of a dumped system.
__global__ void k_lpc_dump_rows(int nu, const double* __restrict__ adiag, const double* __restrict__ rhs,
                                float* diag32, float* rhs32)
{
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= nu) return;
    diag32[r] = (float)adiag[r];
    rhs32[r] = (float)rhs[r];
}

// ---- network forward --------------------------------------------------------
struct AggArgs {
    int nu, cap;
    const int32_t* __restrict__ rowlen;
    const int32_t* __restrict__ acol;
    const float* __restrict__ aval;
    const float* __restrict__ inv_osum;
    const uint16_t* __restrict__ s;
    uint16_t* m;
};

// m_r = (sum_k O_rk s_k) / sum_k O_rk over the matrix row: G lanes per row, each
// with 16 / G of the message's channels.
// Bound by the gathers' cache lookups: one thread per row, 32 bytes an entry,
// made two a row and entry, the lanes of a row make one between them. 107k rows
// of 215 entries 176 -> 102 us (8 lanes: the same within 3 %), 14.6k rows 134 ->
// 19 us. 16 entries a batch and 3 to 6 waves a SIMD measured the same, 4 entries
// slower, 8 waves 6 to 20 % slower (107k rows, blocks of 128 to 1024 threads).
template <int G>
__global__ __launch_bounds__(kBlock) void k_lpc_agg(AggArgs a)
{
    constexpr int D = LM / G / 2;                      // dwords (channel pairs) of a lane
    const int q = threadIdx.x & (G - 1);
    const int r = xcd_block() * (kBlock / G) + threadIdx.x / G;
    if (r >= a.nu) return;
    struct Part { uint32_t w[D]; };
    const Part* __restrict__ s = reinterpret_cast<const Part*>(a.s);
    float acc[2 * D] = {};
    walk_row<8>(a.acol, a.aval, r, a.cap, a.rowlen[r], [&](int c) { return s[(long)G * c + q]; },
                [&](int, float v, const Part& x) {
#pragma unroll
                    for (int t = 0; t < D; ++t) {
                        acc[2 * t] = fmaf(-v, bf_lo(x.w[t]), acc[2 * t]);
                        acc[2 * t + 1] = fmaf(-v, bf_hi(x.w[t]), acc[2 * t + 1]);
                    }
                });
    const float io = a.inv_osum[r];
    Part o;
#pragma unroll
    for (int t = 0; t < D; ++t)
        o.w[t] = (uint32_t)f2bf(acc[2 * t] * io) | ((uint32_t)f2bf(acc[2 * t + 1] * io) << 16);
    reinterpret_cast<Part*>(a.m)[(long)G * r + q] = o;
}

// Inference: t_r = sqrt(c_r) / A_rr, gd_r = g_r / A_rr from the network
// output, then coupling values (O_rk t_r) t_k.
__global__ void k_lpc_gc_inf(int nu, const float* __restrict__ o, const float* __restrict__ invd, float* gd,
                             float* t)
{
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= nu) return;
    const float gv = expf(0.5f * tanhf(o[2 * r]));
    const float cv = kCMax / (1.f + expf(-(o[2 * r + 1] + kBeta)));
    gd[r] = gv * invd[r];
    t[r] = sqrtf(cv) * invd[r];
}

// (4 threads per row, 64 rows side by side; 31 -> 20 us at 107k rows)
__global__ __launch_bounds__(kBlock) void k_lpc_scale(int nu, int cap, const int32_t* __restrict__ slen,
                                                      const int32_t* __restrict__ scol,
                                                      const float* __restrict__ t, float* sval)
{
    const int r = xcd_block() * kWave + (threadIdx.x & (kWave - 1));
    if (r >= nu) return;
    const long b = mx_index(r, 0, cap);
    const float tr = t[r];
    const int len = slen[r];
    for (int k = threadIdx.x >> 6; k < len; k += kBlock / kWave)
        sval[b + 64L * k] = (sval[b + 64L * k] * tr) * t[scol[b + 64L * k]];
}

struct DenseArgs {
    int rows, layer;            // rows: multiple of 16; layer 0 = encoder
    const uint16_t* __restrict__ w16;
    const float* __restrict__ w32;
    const float* __restrict__ feat;
    const uint16_t* __restrict__ hin;
    const uint16_t* __restrict__ min;
    uint16_t* hout;
    uint16_t* sout;             // next layer's messages (layer < 3)
    float* o;                   // network output (layer 3)
};

typedef short v8s __attribute__((ext_vector_type(8)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

__device__ __forceinline__ v8s ld8(const uint16_t* p) { return *reinterpret_cast<const v8s*>(p); }

// D += A B on gfx950's 16 x 16 x 32 bf16 matrix instruction.
__device__ __forceinline__ v4f mfma32(v8s x, v8s y, v4f acc)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, x),
                                                   __builtin_bit_cast(v8bf, y), acc, 0, 0, 0);
}

// One 16-row tile per wavefront. Operand layouts of v_mfma_f32_16x16x32_bf16:
// lane l supplies A[row l%16][k 8*(l/16)..+7] and B[k 8*(l/16)..+7][col l%16]
// and receives D[row 4*(l/16)+i][col l%16], i = 0..3. Rows are graph rows,
// columns are output features, k runs over input features: the encoder's 8
// features are one instruction (k 8..31 zero), a message layer's 64 hidden
// inputs two and its 16 messages one (k 16..31 zero), the message
// projection's 64 inputs two.
template <int MODE>   // 0: encoder (features in), 1: message layer
__global__ __launch_bounds__(kBlock) void k_lpc_dense(DenseArgs a)
{
    __shared__ __align__(16) uint16_t th[4][16][LH + 8];
    __shared__ __align__(16) uint16_t ts[4][16][LM];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int cl = lane & 15, gp = lane >> 4;
    constexpr int KB = (MODE == 0) ? 1 : 3;
    const v8s zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
    const int l = a.layer;
    v8s bw[KB][4];
    float bias[4];
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
        const int o = nt * 16 + cl;
        if (MODE == 0) {
            bw[0][nt] = (gp == 0) ? ld8(a.w16 + OFF_W0 + o * LF) : zero8;
            bias[nt] = a.w32[OFF_B0 + o];
        } else {
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) bw[kb][nt] = ld8(a.w16 + off_U(l) + o * LH + kb * 32 + 8 * gp);
            bw[KB - 1][nt] = (gp < 2) ? ld8(a.w16 + off_V(l) + o * LM + 8 * gp) : zero8;
            bias[nt] = a.w32[off_c(l) + o];
        }
    }
    const bool next = (l < LNL);
    v8s bp[2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
        bp[kb] = next ? ld8(a.w16 + off_P(l + 1) + cl * LH + kb * 32 + 8 * gp) : zero8;
    float wo[2][LH / 2];   // head weights of this lane's output (lanes < 32)
    if (!next) {
        const int q = lane & 1;
#pragma unroll
        for (int k = 0; k < LH / 2; ++k) {
            wo[0][k] = a.w32[OFF_WO + q * LH + k];
            wo[1][k] = a.w32[OFF_WO + q * LH + LH / 2 + k];
        }
    }
    const int ntile = a.rows / 16;
    for (int base = blockIdx.x * 4; base < ntile; base += gridDim.x * 4) {
        const int tile = base + wv;
        const bool act = tile < ntile;
        const long row0 = (long)tile * 16;
        if (act) {
            v8s af[KB];
            if (MODE == 0) {
                if (gp == 0) {
                    const float* f = a.feat + (row0 + cl) * LF;
                    af[0] = v8s{(short)f2bf(f[0]), (short)f2bf(f[1]), (short)f2bf(f[2]),
                                (short)f2bf(f[3]), (short)f2bf(f[4]), (short)f2bf(f[5]),
                                (short)f2bf(f[6]), (short)f2bf(f[7])};
                } else {
                    af[0] = zero8;
                }
            } else {
#pragma unroll
                for (int kb = 0; kb < 2; ++kb) af[kb] = ld8(a.hin + (row0 + cl) * LH + kb * 32 + 8 * gp);
                if (gp < 2) af[KB - 1] = ld8(a.min + (row0 + cl) * LM + 8 * gp);
                else af[KB - 1] = zero8;
            }
#pragma unroll
            for (int nt = 0; nt < 4; ++nt) {
                v4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int kb = 0; kb < KB; ++kb) acc = mfma32(af[kb], bw[kb][nt], acc);
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    th[wv][4 * gp + i][nt * 16 + cl] = f2bf(fmaxf(acc[i] + bias[nt], 0.f));
            }
        }
        __syncthreads();
        if (act) {
            const int nd = lane >> 2, pt = lane & 3;
            const v4i* src = reinterpret_cast<const v4i*>(&th[wv][nd][pt * 16]);
            v4i* dst = reinterpret_cast<v4i*>(a.hout + (row0 + nd) * LH + pt * 16);
            dst[0] = src[0];
            dst[1] = src[1];
            if (next) {
                v4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int kb = 0; kb < 2; ++kb) {
                    const v8s x = *reinterpret_cast<const v8s*>(&th[wv][cl][kb * 32 + 8 * gp]);
                    acc = mfma32(x, bp[kb], acc);
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) ts[wv][4 * gp + i][cl] = f2bf(acc[i]);
            } else if (lane < 32) {
                // head: lane = 2 * row + output
                const int nd2 = lane >> 1, q = lane & 1;
                float acc = a.w32[OFF_BO + q];
#pragma unroll
                for (int k = 0; k < LH / 2; ++k) acc = fmaf(wo[0][k], bf2f(th[wv][nd2][k]), acc);
#pragma unroll
                for (int k = 0; k < LH / 2; ++k) acc = fmaf(wo[1][k], bf2f(th[wv][nd2][LH / 2 + k]), acc);
                a.o[(row0 + nd2) * LO + q] = acc;
            }
        }
        __syncthreads();
        if (act && next && lane < 32) {
            const int nd = lane >> 1, hf = lane & 1;
            *reinterpret_cast<v4i*>(a.sout + (row0 + nd) * LM + hf * 8) =
                *reinterpret_cast<const v4i*>(&ts[wv][nd][hf * 8]);
        }
        __syncthreads();
    }
}

// g, sqrt(c) (and c) from the network output.
__global__ void k_lpc_gc(int nu, const float* __restrict__ o, float* g, float* c, float* sc)
{
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= nu) return;
    const float gv = expf(0.5f * tanhf(o[2 * r]));
    const float cv = kCMax / (1.f + expf(-(o[2 * r + 1] + kBeta)));
    g[r] = gv;
    if (c) c[r] = cv;
    sc[r] = sqrtf(cv);
}

// ---- training: probes and the loss gradient with respect to g and c --------
// Vectors of the four probes are interleaved: element 4 r + p.
enum { LS_NN = 0, LS_COEF = kProbes, LS_LOSS = 2 * kProbes, LS_EPOCH, LS_COUNT };

// w = right-hand side, then three Rademacher vectors; v = sc w; partial ||rhs||^2.
__global__ __launch_bounds__(kBlock) void k_lpc_probe(int nu, uint64_t seed, const float* __restrict__ rhs,
                                                      const float* __restrict__ sc, v4f* w, v4f* v,
                                                      double* part)
{
    __shared__ double lds[kBlock];
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    double s = 0.0;
    if (r < nu) {
        const v4f x = {rhs[r], (float)rademacher(seed, 1, r), (float)rademacher(seed, 2, r),
                       (float)rademacher(seed, 3, r)};
        w[r] = x;
        v[r] = x * sc[r];
        s = (double)x.x * (double)x.x;
    }
    s = block_sum(s, lds);
    if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// From the partial ||rhs||^2 (n1) and ||A M w - w||^2 (n2 a probe): each probe's
// norm and gradient factor 2 / (probes ||w||^2), and the loss.
__global__ __launch_bounds__(kBlock) void k_lpc_fin(int nu, const double* __restrict__ part, int n1,
                                                    const double* __restrict__ epart, int n2, double* scal)
{
    __shared__ double lds[kBlock];
    double loss = 0.0;
    for (int p = 0; p < kProbes; ++p) {
        double s = 0.0, e = 0.0;
        if (p == 0) {
            for (int k = threadIdx.x; k < n1; k += kBlock) s = s + part[k];
            s = block_sum(s, lds);
        } else {
            s = (double)nu;
        }
        for (int k = threadIdx.x; k < n2; k += kBlock) e = e + epart[(long)p * n2 + k];
        e = block_sum(e, lds);
        if (threadIdx.x != 0) continue;
        scal[LS_NN + p] = s;
        scal[LS_COEF + p] = s > 0 ? 2.0 / (kProbes * s) : 0.0;
        loss += s > 0 ? e / (kProbes * s) : 0.0;
    }
    if (threadIdx.x == 0) scal[LS_LOSS] = loss;
}

__global__ void k_lpc_set(double* scal, int slot, double v) { scal[slot] = v; }
__global__ void k_lpc_epoch(double* scal) { scal[LS_EPOCH] += scal[LS_LOSS]; }

struct OpView {   // a SELL-64 operator: rows, cap, lengths, columns, values
    int nu, cap;
    const int32_t* __restrict__ len;
    const int32_t* __restrict__ col;
    const float* __restrict__ val;
};

// init + sum_k a_rk x_k of row r for probe p.
__device__ __forceinline__ float row_product(const OpView& A, int r, int p, const float* __restrict__ x,
                                             float init)
{
    float acc = init;
    walk_row<8>(A.col, A.val, r, A.cap, A.len[r], [&](int c) { return x[4L * c + p]; },
                [&](int, float v, float y) { acc = fmaf(v, y, acc); });
    return acc;
}

// One lane per row and probe in the kernels that follow, so that an operator is
// walked once for the four probes and a gather takes their 16 bytes together.
// 14.6k rows of 215 entries, all four probes: residual 4 x 87 -> 17 us, adjoint
// 4 x 87 -> 15, mprobe 4 x 22 -> 7, dgc 4 x 36 -> 8.
// t = Oh (sc w); z = g w / A_rr + sc t
__global__ __launch_bounds__(kBlock) void k_lpc_mprobe(OpView S, const float* __restrict__ sc,
                                                       const float* __restrict__ g,
                                                       const float* __restrict__ inv_d,
                                                       const float* __restrict__ w,
                                                       const float* __restrict__ v, float* t, float* z)
{
    const int e = xcd_tid(), r = e >> 2;
    if (r >= S.nu) return;
    const float acc = row_product(S, r, e & 3, v, 0.f);
    t[e] = acc;
    z[e] = fmaf(sc[r], acc, (g[r] * inv_d[r]) * w[e]);
}

// e = A z - w, partial ||e||^2 per block and probe
__global__ __launch_bounds__(kBlock) void k_lpc_residual(OpView A, const float* __restrict__ diag,
                                                         const float* __restrict__ z,
                                                         const float* __restrict__ w, float* out,
                                                         double* epart)
{
    __shared__ double lds[kBlock];
    const int e = xcd_tid(), r = e >> 2, t = threadIdx.x;
    double ee = 0.0;
    if (r < A.nu) {
        const float d = row_product(A, r, e & 3, z, diag[r] * z[e]) - w[e];
        out[e] = d;
        ee = (double)d * (double)d;
    }
    lds[t] = ee;
    __syncthreads();
    for (int s = kBlock / 2; s >= kProbes; s >>= 1) {
        if (t < s) lds[t] = lds[t] + lds[t + s];
        __syncthreads();
    }
    if (t < kProbes) epart[(long)t * gridDim.x + blockIdx.x] = lds[t];
}

// y = coef A e and sc y
__global__ __launch_bounds__(kBlock) void k_lpc_adjoint(OpView A, const float* __restrict__ diag,
                                                        const float* __restrict__ x,
                                                        const float* __restrict__ sc,
                                                        const double* __restrict__ scal, float* y, float* ys)
{
    const int e = xcd_tid(), r = e >> 2;
    if (r >= A.nu) return;
    const float acc = row_product(A, r, e & 3, x, diag[r] * x[e]);
    const float v = (float)(scal[LS_COEF + (e & 3)] * (double)acc);
    y[e] = v;
    ys[e] = sc[r] * v;
}

// u = Oh (sc y); dL/dg = sum over probes of y w / A_rr; dL/dc = (y t + w u) / (2 sc);
// then through the output functions (dO) and the head's weights (dh).
__global__ __launch_bounds__(kBlock) void k_lpc_dgc(OpView S, const float* __restrict__ sc,
                                                    const float* __restrict__ inv_d,
                                                    const float* __restrict__ w,
                                                    const float* __restrict__ t,
                                                    const float* __restrict__ y,
                                                    const float* __restrict__ ys,
                                                    const float* __restrict__ w32,
                                                    const float* __restrict__ o,
                                                    const float* __restrict__ g, float* dO, float* dh)
{
    const int e = xcd_tid(), r = e >> 2, p = e & 3;
    if (r >= S.nu) return;
    const float u = row_product(S, r, p, ys, 0.f);
    const float dgp = y[e] * w[e] * inv_d[r];
    const float dcp = (0.5f / sc[r]) * (y[e] * t[e] + w[e] * u);
    float dg = __shfl(dgp, 0, 4), dc = __shfl(dcp, 0, 4);
#pragma unroll
    for (int k = 1; k < kProbes; ++k) {
        dg += __shfl(dgp, k, 4);
        dc += __shfl(dcp, k, 4);
    }
    const float th = tanhf(o[2 * r]);
    const float s = 1.f / (1.f + expf(-(o[2 * r + 1] + kBeta)));
    const float d0 = dg * g[r] * 0.5f * (1.f - th * th);
    const float d1 = dc * kCMax * s * (1.f - s);
    if (p < LO) dO[2 * r + p] = p ? d1 : d0;
#pragma unroll
    for (int j = 0; j < LH / 16; ++j) {
        const int k = 16 * j + 4 * p;
        v4f v;
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = fmaf(d0, w32[OFF_WO + k + i], d1 * w32[OFF_WO + LH + k + i]);
        *reinterpret_cast<v4f*>(dh + LH * (long)r + k) = v;
    }
}

// ---- training: backward through the network (FP32) -------------------------
// dpre = dh * [h > 0] is formed where it is read.
__device__ __forceinline__ float relu_grad(float dh, uint16_t h) { return bf2f(h) > 0.f ? dh : 0.f; }

// dh_prev = dpre U (the direct part) and dmh = (dpre V) / sum_k O_rk (the
// aggregation's input gradient, scaled) of layer l >= 1: one 16-row tile per
// wave, 80 output columns, on v_mfma_f32_16x16x4_f32 (operands: lane l holds
// A[row l%16][k l/16] and B[k l/16][col l%16], D[row 4*(l/16)+i][col l%16]). k is
// taken so that lane group g holds inputs 16 g .. 16 g + 15: contiguous loads.
// 14.6k rows 57 (one thread per row, weights read from LDS) -> 7.4 us.
__global__ __launch_bounds__(kBlock) void k_lpc_dense_bwd(int nu, int l, const uint16_t* __restrict__ w16,
                                                          const uint16_t* __restrict__ h,
                                                          const float* __restrict__ dh,
                                                          const float* __restrict__ inv_osum, float* dmh,
                                                          float* dh_prev)
{
    constexpr int NC = LH + LM;
    __shared__ __align__(16) uint16_t wt[NC][LH + 8];  // [output column][input]
    for (int k = threadIdx.x; k < LH * NC / 8; k += kBlock) {
        const int o = k / (NC / 8), c = (k % (NC / 8)) * 8;
        const v8s v = c < LH ? ld8(w16 + off_U(l) + o * LH + c) : ld8(w16 + off_V(l) + o * LM + (c - LH));
#pragma unroll
        for (int i = 0; i < 8; ++i) wt[c + i][o] = (uint16_t)v[i];
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
    const int row0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * 16;
    if (row0 >= nu) return;
    const long in = LH * (long)min(row0 + n, nu - 1) + 16 * g;
    float dp[16];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const v4f v = *reinterpret_cast<const v4f*>(dh + in + 4 * q);
#pragma unroll
        for (int i = 0; i < 4; ++i) dp[4 * q + i] = v[i];
    }
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const v8s v = ld8(h + in + 8 * q);
#pragma unroll
        for (int i = 0; i < 8; ++i) dp[8 * q + i] = relu_grad(dp[8 * q + i], (uint16_t)v[i]);
    }
    for (int nt = 0; nt < NC / 16; ++nt) {
        v4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const v8s v = *reinterpret_cast<const v8s*>(&wt[16 * nt + n][16 * g + 8 * q]);
#pragma unroll
            for (int i = 0; i < 8; ++i)
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(dp[8 * q + i], bf2f((uint16_t)v[i]), acc, 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = row0 + 4 * g + i;
            if (r >= nu) continue;
            if (nt < LH / 16) dh_prev[LH * (long)r + 16 * nt + n] = acc[i];
            else dmh[LM * (long)r + n] = acc[i] * inv_osum[r];
        }
    }
}

// ds_k = sum_r O_kr dmh_r (transpose of the aggregation; O is symmetric), 8
// lanes per row with 2 of the 16 channels each, and dh_prev_k += ds_k P_l.
// 14.6k rows 165 (one thread per row) -> 30 us.
__global__ __launch_bounds__(kBlock) void k_lpc_agg_bwd(int nu, int cap, const int32_t* __restrict__ rowlen,
                                                        const int32_t* __restrict__ acol,
                                                        const float* __restrict__ aval, int l,
                                                        const uint16_t* __restrict__ w16,
                                                        const float* __restrict__ dmh, float* ds,
                                                        float* dh_prev)
{
    constexpr int R = kBlock / 8;                      // rows of a block
    __shared__ float sP[LM * LH];
    __shared__ float sd[R][LM];
    for (int k = threadIdx.x; k < LM * LH; k += kBlock) sP[k] = bf2f(w16[off_P(l) + k]);
    const int q = threadIdx.x & 7, lr = threadIdx.x >> 3;
    const int row0 = xcd_block() * R, r = row0 + lr;
    float a0 = 0.f, a1 = 0.f;
    if (r < nu) {
        const float2* __restrict__ d = reinterpret_cast<const float2*>(dmh);
        walk_row<8>(acol, aval, r, cap, rowlen[r], [&](int c) { return d[8L * c + q]; },
                    [&](int, float v, float2 x) {
                        a0 = fmaf(-v, x.x, a0);
                        a1 = fmaf(-v, x.y, a1);
                    });
        *reinterpret_cast<float2*>(ds + LM * (long)r + 2 * q) = make_float2(a0, a1);
    }
    sd[lr][2 * q] = a0;
    sd[lr][2 * q + 1] = a1;
    __syncthreads();
    for (int k = threadIdx.x; k < R * LH; k += kBlock) {
        const int i = k / LH, c = k % LH;
        if (row0 + i >= nu) break;
        float v = dh_prev[LH * (long)(row0 + i) + c];
#pragma unroll
        for (int j = 0; j < LM; ++j) v = fmaf(sd[i][j], sP[j * LH + c], v);
        dh_prev[LH * (long)(row0 + i) + c] = v;
    }
}

// Weight gradients of one layer over a block's rows, all in one launch: sums of
// outer products of row vectors, matrix products with the graph's rows as the
// inner index (4 rows an instruction); wave w takes the 16 outputs 16 w .. 16 w
// + 15. MODE 0: encoder (dpre x features, bias); 1: message layer (dpre x h, dpre
// x m, bias, ds x h); 2: head (dO x h, bias). Partials in the parameters' order.
// 14.6k rows, a message layer: four products and their reductions 270 -> 11 us,
// the one reduction of all layers' partials 50 a product -> 6 us.
struct WGradArgs {
    int nu, chunk, layer;
    const float* __restrict__ dh;          // gradient of the layer's output
    const uint16_t* __restrict__ hl;       // the layer's output
    const uint16_t* __restrict__ hp;       // the layer's input
    const uint16_t* __restrict__ mp;       // and messages
    const float* __restrict__ ds;
    const float* __restrict__ feat;
    float* part;
};

template <int MODE>
__global__ __launch_bounds__(kBlock) void k_lpc_wgrad(WGradArgs a)
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, n = lane & 15, g = lane >> 4;
    const int r0 = blockIdx.x * a.chunk, r1 = min(a.nu, r0 + a.chunk);
    constexpr int NU = MODE == 1 ? 4 : 1;
    v4f cu[NU], cv = {0.f, 0.f, 0.f, 0.f}, cp = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < NU; ++t) cu[t] = v4f{0.f, 0.f, 0.f, 0.f};
    float bias = 0.f;
#pragma unroll 8
    for (int s = r0; s < r1; s += 4) {
        const bool ok = s + g < r1;
        const long r = ok ? s + g : r0;
        float x;
        if (MODE == 2) x = a.dh[LO * r + (n & (LO - 1))];
        else x = relu_grad(a.dh[LH * r + 16 * w + n], a.hl[LH * r + 16 * w + n]);
        if (!ok || (MODE == 2 && n >= LO)) x = 0.f;
        bias += x;
        if (MODE == 0) {
            float y = bf2f(f2bf(a.feat[LF * r + (n & (LF - 1))]));
            if (n >= LF) y = 0.f;
            cu[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(x, y, cu[0], 0, 0, 0);
        } else if (MODE == 2) {
            cu[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(x, bf2f(a.hp[LH * r + 16 * w + n]), cu[0], 0, 0, 0);
        } else {
#pragma unroll
            for (int t = 0; t < NU; ++t)
                cu[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(x, bf2f(a.hp[LH * r + 16 * t + n]), cu[t], 0, 0, 0);
            cv = __builtin_amdgcn_mfma_f32_16x16x4f32(x, bf2f(a.mp[LM * r + n]), cv, 0, 0, 0);
            float d = a.ds[LM * r + n];
            if (!ok) d = 0.f;
            cp = __builtin_amdgcn_mfma_f32_16x16x4f32(d, bf2f(a.hp[LH * r + 16 * w + n]), cp, 0, 0, 0);
        }
    }
    bias += __shfl_xor(bias, 16);
    bias += __shfl_xor(bias, 32);
    float* __restrict__ p = a.part + (long)blockIdx.x * NPARAM;
    const int l = a.layer;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int q = 4 * g + i, o = 16 * w + q;
        if (MODE == 0) {
            if (n < LF) p[OFF_W0 + o * LF + n] = cu[0][i];
        } else if (MODE == 2) {
            if (q < LO) p[OFF_WO + q * LH + 16 * w + n] = cu[0][i];
        } else {
#pragma unroll
            for (int t = 0; t < NU; ++t) p[off_U(l) + o * LH + 16 * t + n] = cu[t][i];
            p[off_V(l) + o * LM + n] = cv[i];
            p[off_P(l) + q * LH + 16 * w + n] = cp[i];
        }
    }
    if (g != 0) return;
    if (MODE == 0) p[OFF_B0 + 16 * w + n] = bias;
    if (MODE == 1) p[off_c(l) + 16 * w + n] = bias;
    if (MODE == 2 && w == 0 && n < LO) p[OFF_BO + n] = bias;
}

// The gradient: FP64 sums of the blocks' partials, 64 parameters x 16 shares of
// the blocks a block.
__global__ __launch_bounds__(1024) void k_lpc_reduce(int nblk, const float* __restrict__ part, float* out)
{
    __shared__ double lds[16][kWave];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int e = blockIdx.x * kWave + lane;
    double s = 0.0;
    if (e < NPARAM)
#pragma unroll 4
        for (int b = w; b < nblk; b += 16) s += (double)part[(long)b * NPARAM + e];
    lds[w][lane] = s;
    __syncthreads();
    if (w != 0 || e >= NPARAM) return;
    for (int k = 1; k < 16; ++k) s += lds[k][lane];
    out[e] = (float)s;
}

__global__ void k_lpc_adam(int n, float* w, const float* __restrict__ g, float* m, float* v, float lr,
                           float b1, float b2, float eps, float bc1, float bc2, uint16_t* w16)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const float gk = g[k];
    const float mk = b1 * m[k] + (1.f - b1) * gk;
    const float vk = b2 * v[k] + (1.f - b2) * gk * gk;
    m[k] = mk;
    v[k] = vk;
    const float wk = w[k] - lr * (mk / bc1) / (sqrtf(vk / bc2) + eps);
    w[k] = wk;
    w16[k] = f2bf(wk);
}

__global__ void k_lpc_cast(int n, const float* __restrict__ w, uint16_t* w16)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) w16[k] = f2bf(w[k]);
}

}  // namespace vox

// ---- the network object -------------------------------------------------------
namespace {

struct LpcSys {
    int nu = 0, rows = 0, cap = 0;
    int32_t *rowlen = nullptr, *acol = nullptr, *slen = nullptr, *scol = nullptr;
    float *aval = nullptr, *diag = nullptr, *inv_d = nullptr, *inv_osum = nullptr, *feat = nullptr,
          *rhs = nullptr, *sval = nullptr;
};

}  // namespace

struct vox_lpc {
    int device = 0;
    hipStream_t stream = nullptr;
    float *w32 = nullptr, *grad = nullptr, *am = nullptr, *av = nullptr, *gpart = nullptr;
    uint16_t* w16 = nullptr;
    double *dpart = nullptr, *dscal = nullptr, *hscal = nullptr;
    float* hgrad = nullptr;        // pinned: a pageable copy of the gradient takes 25 us
    std::mutex hgrad_m;
    std::vector<LpcSys> sys;
    int rows_cap = 0;
    uint16_t *h[4] = {}, *s[3] = {}, *m[3] = {};
    float *o = nullptr, *g = nullptr, *c = nullptr, *sc = nullptr;
    float *wv = nullptr, *vv = nullptr, *t = nullptr, *z = nullptr, *e = nullptr, *y = nullptr,
          *ys = nullptr, *dO = nullptr, *dh[2] = {}, *dmh = nullptr, *ds = nullptr;
    double* epart = nullptr;
    long adam_t = 0;
};

namespace vox {

// Zeroed memory for kernels on `stream`, cleared in that stream's order: the streams
// here do not wait for the null stream, on which a clear of hundreds of megabytes would
// still run when the first kernels write there.
template <class T>
static int lalloc(hipStream_t stream, T** p, size_t n)
{
    if (n == 0) n = 1;
    VOX_HIP(hipMalloc((void**)p, sizeof(T) * n));
    VOX_HIP(hipMemsetAsync(*p, 0, sizeof(T) * n, stream));
    return VOX_OK;
}
template <class T>
static void lfree(T*& p)
{
    if (p) (void)hipFree(p);
    p = nullptr;
}
static int round64(int n) { return (n + 63) & ~63; }

// He-uniform weights from SplitMix64(seed) in the packed order; biases zero,
// the output layer scaled by 0.1 (outputs start near g = c = 1).
static void init_weights(uint64_t seed, std::vector<float>& w)
{
    w.assign(NPARAM, 0.f);
    uint64_t st = seed;
    auto next = [&]() {
        uint64_t z = (st += 0x9E3779B97F4A7C15ull);
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        z = z ^ (z >> 31);
        return (double)(z >> 11) * (1.0 / 9007199254740992.0);
    };
    auto fill = [&](int off, int rows, int cols, double gain) {
        const double lim = gain * std::sqrt(6.0 / cols);
        for (int k = 0; k < rows * cols; ++k) w[off + k] = (float)((2.0 * next() - 1.0) * lim);
    };
    fill(OFF_W0, LH, LF, 1.0);
    for (int l = 1; l <= LNL; ++l) {
        fill(off_P(l), LM, LH, 1.0);
        fill(off_U(l), LH, LH, 1.0);
        fill(off_V(l), LH, LM, 1.0);
    }
    fill(OFF_WO, LO, LH, 0.1);
}

static int lpc_training_buffers(vox_lpc* L, int rows)
{
    if (rows <= L->rows_cap) return VOX_OK;
    for (auto*& p : L->h) lfree(p);
    for (auto*& p : L->s) lfree(p);
    for (auto*& p : L->m) lfree(p);
    for (float** p : {&L->o, &L->g, &L->c, &L->sc, &L->wv, &L->vv, &L->t, &L->z, &L->e, &L->y, &L->ys,
                      &L->dO, &L->dh[0], &L->dh[1], &L->dmh, &L->ds})
        lfree(*p);
    lfree(L->epart);
    const size_t n = (size_t)rows;
    auto alloc = [&](auto** p, size_t k) { return lalloc(L->stream, p, k); };
    for (auto*& p : L->h) VOX_TRY(alloc(&p, n * LH));
    for (auto*& p : L->s) VOX_TRY(alloc(&p, n * LM));
    for (auto*& p : L->m) VOX_TRY(alloc(&p, n * LM));
    VOX_TRY(alloc(&L->o, n * LO));
    for (float** p : {&L->g, &L->c, &L->sc}) VOX_TRY(alloc(p, n));
    for (float** p : {&L->wv, &L->vv, &L->t, &L->z, &L->e, &L->y, &L->ys}) VOX_TRY(alloc(p, n * kProbes));
    VOX_TRY(alloc(&L->epart, (size_t)kProbes * grid_for((long)kProbes * rows)));
    VOX_TRY(alloc(&L->dO, n * 2));
    VOX_TRY(alloc(&L->dh[0], n * LH));
    VOX_TRY(alloc(&L->dh[1], n * LH));
    VOX_TRY(alloc(&L->dmh, n * LM));
    VOX_TRY(alloc(&L->ds, n * LM));
    L->rows_cap = rows;
    return VOX_OK;
}

// Rows from which the aggregation takes 4 lanes a row (fewer instructions an
// entry) instead of 8 (more waves).
constexpr int kAggRows = 32768;

// Network forward over `rows` rows (multiple of 64) of a graph with nu rows;
// h[0..3], s[0..2], m[0..2] may alias as long as layer l's inputs differ from
// its outputs.
static int lpc_forward(hipStream_t st, const vox_lpc* L, int rows, AggArgs ag, const float* feat,
                       uint16_t* const h[4], uint16_t* const s[3], uint16_t* const m[3], float* o)
{
    const int ntile = rows / 16;
    const int nblk = std::max(1, std::min(2048, (ntile + 3) / 4));
    DenseArgs d{};
    d.rows = rows; d.w16 = L->w16; d.w32 = L->w32; d.feat = feat;
    d.layer = 0; d.hout = h[0]; d.sout = s[0]; d.o = o;
    k_lpc_dense<0><<<nblk, kBlock, 0, st>>>(d);
    for (int l = 1; l <= LNL; ++l) {
        ag.s = s[l - 1];
        ag.m = m[l - 1];
        if (ag.nu < kAggRows) k_lpc_agg<8><<<grid_for(8L * ag.nu), kBlock, 0, st>>>(ag);
        else k_lpc_agg<4><<<grid_for(4L * ag.nu), kBlock, 0, st>>>(ag);
        d.layer = l; d.hin = h[l - 1]; d.min = m[l - 1]; d.hout = h[l];
        d.sout = (l < LNL) ? s[l] : nullptr;
        k_lpc_dense<1><<<nblk, kBlock, 0, st>>>(d);
    }
    VOX_HIP(hipGetLastError());
    return VOX_OK;
}

static int lpc_forward_sys(vox_lpc* L, const LpcSys& S)
{
    AggArgs ag{};
    ag.nu = S.nu; ag.cap = S.cap; ag.rowlen = S.rowlen; ag.acol = S.acol; ag.aval = S.aval;
    ag.inv_osum = S.inv_osum;
    VOX_TRY(lpc_forward(L->stream, L, S.rows, ag, S.feat, L->h, L->s, L->m, L->o));
    k_lpc_gc<<<grid_for(S.nu), kBlock, 0, L->stream>>>(S.nu, L->o, L->g, L->c, L->sc);
    VOX_HIP(hipGetLastError());
    return VOX_OK;
}

// Loss (into dscal[LS_LOSS]) and gradient (into L->grad) on one system.
static int lpc_loss_grad_sys(vox_lpc* L, const LpcSys& S, uint64_t seed)
{
    hipStream_t st = L->stream;
    const int nu = S.nu;
    if (grid_for(nu) > kMaxPartials) return fail(VOX_ERR_ARG, "training system too large");
    VOX_TRY(lpc_forward_sys(L, S));
    const OpView SO{nu, S.cap, S.slen, S.scol, S.sval};
    const OpView AO{nu, S.cap, S.rowlen, S.acol, S.aval};
    const int nb = grid_for(nu), nb4 = grid_for((long)kProbes * nu);
    k_lpc_probe<<<nb, kBlock, 0, st>>>(nu, seed, S.rhs, L->sc, reinterpret_cast<v4f*>(L->wv),
                                       reinterpret_cast<v4f*>(L->vv), L->dpart);
    k_lpc_mprobe<<<nb4, kBlock, 0, st>>>(SO, L->sc, L->g, S.inv_d, L->wv, L->vv, L->t, L->z);
    k_lpc_residual<<<nb4, kBlock, 0, st>>>(AO, S.diag, L->z, L->wv, L->e, L->epart);
    k_lpc_fin<<<1, kBlock, 0, st>>>(nu, L->dpart, nb, L->epart, nb4, L->dscal);
    k_lpc_adjoint<<<nb4, kBlock, 0, st>>>(AO, S.diag, L->e, L->sc, L->dscal, L->y, L->ys);
    k_lpc_dgc<<<nb4, kBlock, 0, st>>>(SO, L->sc, S.inv_d, L->wv, L->t, L->y, L->ys, L->w32, L->o, L->g,
                                      L->dO, L->dh[0]);
    VOX_HIP(hipGetLastError());
    // weight gradients: a block sums at least 64 rows, a multiple of 4
    WGradArgs wg{};
    wg.nu = nu;
    wg.chunk = ((std::max(64, (nu + kOuterBlocks - 1) / kOuterBlocks)) + 3) & ~3;
    wg.part = L->gpart;
    const int nw = grid_for(nu, wg.chunk);
    wg.dh = L->dO; wg.hp = L->h[LNL];
    k_lpc_wgrad<2><<<nw, kBlock, 0, st>>>(wg);
    int cur = 0;
    for (int l = LNL; l >= 1; --l) {
        float* dh = L->dh[cur];
        float* dhp = L->dh[cur ^ 1];
        k_lpc_dense_bwd<<<grid_for(nu, 64), kBlock, 0, st>>>(nu, l, L->w16, L->h[l], dh, S.inv_osum, L->dmh,
                                                             dhp);
        k_lpc_agg_bwd<<<grid_for(8L * nu), kBlock, 0, st>>>(nu, S.cap, S.rowlen, S.acol, S.aval, l, L->w16,
                                                            L->dmh, L->ds, dhp);
        wg.layer = l; wg.dh = dh; wg.hl = L->h[l]; wg.hp = L->h[l - 1]; wg.mp = L->m[l - 1]; wg.ds = L->ds;
        k_lpc_wgrad<1><<<nw, kBlock, 0, st>>>(wg);
        cur ^= 1;
    }
    wg.layer = 0; wg.dh = L->dh[cur]; wg.hl = L->h[0]; wg.feat = S.feat;
    k_lpc_wgrad<0><<<nw, kBlock, 0, st>>>(wg);
    k_lpc_reduce<<<grid_for(NPARAM, kWave), 1024, 0, st>>>(nw, L->gpart, L->grad);
    VOX_HIP(hipGetLastError());
    return VOX_OK;
}

static int check_lpc(vox_lpc* L)
{
    if (!L) return fail(VOX_ERR_ARG, "null learned preconditioner");
    VOX_HIP(hipSetDevice(L->device));
    return VOX_OK;
}

static int check_index(vox_lpc* L, int index)
{
    if (index < 0 || index >= (int)L->sys.size()) return fail(VOX_ERR_ARG, "no stored system of that index");
    return VOX_OK;
}

// ---- inference for a context ------------------------------------------------
void lpc_free_ctx(vox_ctx* c)
{
    lfree(c->lpc_feat); lfree(c->lpc_inv_osum); lfree(c->lpc_t); lfree(c->lpc_invd);
    lfree(c->lpc_upos);
    lfree(c->lpc_h[0]); lfree(c->lpc_h[1]); lfree(c->lpc_s); lfree(c->lpc_m); lfree(c->lpc_o);
    lfree(c->lpc_gd); lfree(c->lpc_slen); lfree(c->lpc_scol);
    lfree(c->lpc_sval); lfree(c->cg_z); lfree(c->cg_z32);
    c->lpc_rows = 0;
    c->lpc_scap = 0;
}

// Strong-coupling threshold: theta times the coupling of two particles one
// spacing dl apart, ((2 dim / lambda) W(dl) / n0) / rho1 as the assembly forms
// it (W of functions.cu:32-70).
static double lpc_threshold(const vox_ctx* c)
{
    const vox_params& p = c->p;
    const double q = p.dl / p.re_l;
    double w = 0.0;
    if (p.ktype == 2) w = (q < 1.0) ? (1 / q) - 1 : 0.0;
    else if (p.ktype == 6) w = (q <= 1.0) ? (1 - q) * (1 - q) * (1 - q) : 0.0;
    else if (p.ktype == 1) w = (q < 0.5) ? 2.0 - 4.0 * (q * q) : (q <= 1.0 ? (2 * q - 2) * (2 * q - 2) : 0.0);
    else if (p.ktype == 5) w = (q <= 1.0) ? 1.5 * std::log(1 / (q + 0.000001)) : 0.0;
    return 0.25 * ((2.0 * p.dim / p.lambda * w / c->n0l) / p.rho1);
}

// Features and raw strong couplings of the context's assembled PPE (FP32
// values): feat (rows x 8), inv_osum, invd, slen/scol/sval; upos is scratch.
static void ctx_features(vox_ctx* c, int rows, v4f* upos, float* invd, float* feat, float* inv_osum,
                         int32_t* slen, int32_t* scol, float* sval)
{
    PrepArgs pa;
    pa.nu = c->nu; pa.rows = rows; pa.dim = c->p.dim; pa.n0 = c->n0l;
    pa.adiag = c->adiag; pa.urow = c->urow; pa.ptype = c->ptype;
    pa.x = c->f[VOX_F_X]; pa.y = c->f[VOX_F_Y]; pa.z = c->f[VOX_F_Z]; pa.pnd = c->f[VOX_F_N];
    pa.upos = upos; pa.invd = invd; pa.feat = feat;
    k_lpc_rowprep<<<grid_for(rows), kBlock, 0, c->stream>>>(pa);
    FeatArgs fa;
    fa.nu = c->nu; fa.cap = c->a_cap; fa.inv_re = (float)(1.0 / c->p.re_l);
    const double thr = lpc_threshold(c);
    fa.thr = (float)thr;
    if ((double)fa.thr < thr) fa.thr = std::nextafter(fa.thr, INFINITY);
    fa.rowlen = c->rowlen; fa.acol = c->acol; fa.aval = c->aval32; fa.upos = upos; fa.invd = invd;
    fa.feat = feat; fa.inv_osum = inv_osum; fa.slen = slen; fa.scol = scol; fa.sval = sval;
    k_lpc_features<<<grid_for(4L * c->nu), kBlock, 0, c->stream>>>(fa);
}

int lpc_prepare(vox_ctx* c)
{
    VOX_TRY(ensure_acol(c));
    if (!c->lpc) return fail(VOX_ERR_STATE, "learned solver without an attached vox_lpc");
    if (!c->aval32_ok) VOX_TRY(ppe_make_aval32(c));
    ProfScope ps(c, KC_LPC_NET);
    const int nu = c->nu;
    const int rows = round64(c->tp);
    if (c->lpc_rows < rows) {
        lpc_free_ctx(c);
        const size_t n = (size_t)rows;
        auto alloc = [&](auto** p, size_t k) { return lalloc(c->stream, p, k); };
        VOX_TRY(alloc(&c->lpc_feat, n * LF));
        VOX_TRY(alloc(&c->lpc_inv_osum, n));
        VOX_TRY(alloc(&c->lpc_t, n));
        VOX_TRY(alloc(&c->lpc_invd, n));
        VOX_TRY(alloc(&c->lpc_upos, n));
        VOX_TRY(alloc(&c->lpc_h[0], n * LH));
        VOX_TRY(alloc(&c->lpc_h[1], n * LH));
        VOX_TRY(alloc(&c->lpc_s, n * LM));
        VOX_TRY(alloc(&c->lpc_m, n * LM));
        VOX_TRY(alloc(&c->lpc_o, n * LO));
        VOX_TRY(alloc(&c->lpc_gd, n));
        VOX_TRY(alloc(&c->lpc_slen, n));
        VOX_TRY(alloc(&c->cg_z, n));
        VOX_TRY(alloc(&c->cg_z32, n));
        c->lpc_rows = rows;
    }
    if (c->lpc_scap != c->a_cap) {
        lfree(c->lpc_scol);
        lfree(c->lpc_sval);
        VOX_TRY(lalloc(c->stream, &c->lpc_scol, (size_t)sl_size(c->tp, c->a_cap)));
        VOX_TRY(lalloc(c->stream, &c->lpc_sval, (size_t)sl_size(c->tp, c->a_cap)));
        c->lpc_scap = c->a_cap;
    }
    if (nu == 0) return VOX_OK;
    const int frows = round64(nu);
    ctx_features(c, frows, c->lpc_upos, c->lpc_invd, c->lpc_feat, c->lpc_inv_osum, c->lpc_slen,
                 c->lpc_scol, c->lpc_sval);
    AggArgs ag{};
    ag.nu = nu; ag.cap = c->a_cap; ag.rowlen = c->rowlen; ag.acol = c->acol; ag.aval = c->aval32;
    ag.inv_osum = c->lpc_inv_osum;
    uint16_t* const h[4] = {c->lpc_h[0], c->lpc_h[1], c->lpc_h[0], c->lpc_h[1]};
    uint16_t* const s[3] = {c->lpc_s, c->lpc_s, c->lpc_s};
    uint16_t* const m[3] = {c->lpc_m, c->lpc_m, c->lpc_m};
    VOX_TRY(lpc_forward(c->stream, c->lpc, frows, ag, c->lpc_feat, h, s, m, c->lpc_o));
    k_lpc_gc_inf<<<grid_for(nu), kBlock, 0, c->stream>>>(nu, c->lpc_o, c->lpc_invd, c->lpc_gd, c->lpc_t);
    k_lpc_scale<<<grid_for(nu, kWave), kBlock, 0, c->stream>>>(nu, c->a_cap, c->lpc_slen, c->lpc_scol, c->lpc_t,
                                                        c->lpc_sval);
    VOX_HIP(hipGetLastError());
    return VOX_OK;
}

}  // namespace vox

using namespace vox;

extern "C" {

int vox_lpc_create(vox_lpc** out, uint64_t seed)
{
    if (!out) return fail(VOX_ERR_ARG, "null argument");
    *out = nullptr;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return fail(VOX_ERR_HIP, "no HIP device available");
    vox_lpc* L = new vox_lpc();
    auto bail = [&](int rc) { vox_lpc_destroy(L); return rc; };
    if (hipGetDevice(&L->device) != hipSuccess) return bail(fail(VOX_ERR_HIP, "hipGetDevice"));
    if (hipStreamCreateWithFlags(&L->stream, hipStreamNonBlocking) != hipSuccess)
        return bail(fail(VOX_ERR_HIP, "hipStreamCreate"));
    int rc;
    auto alloc = [&](auto** p, size_t n) { return lalloc(L->stream, p, n); };
    if ((rc = alloc(&L->w32, NPARAM)) || (rc = alloc(&L->grad, NPARAM)) || (rc = alloc(&L->am, NPARAM)) ||
        (rc = alloc(&L->av, NPARAM)) || (rc = alloc(&L->w16, NPARAM)) ||
        (rc = alloc(&L->gpart, (size_t)kOuterBlocks * NPARAM)) || (rc = alloc(&L->dpart, (size_t)kMaxPartials)) ||
        (rc = alloc(&L->dscal, LS_COUNT)))
        return bail(rc);
    if (hipHostMalloc((void**)&L->hscal, sizeof(double) * LS_COUNT, hipHostMallocDefault) != hipSuccess ||
        hipHostMalloc((void**)&L->hgrad, sizeof(float) * NPARAM, hipHostMallocDefault) != hipSuccess)
        return bail(fail(VOX_ERR_HIP, "hipHostMalloc"));
    std::vector<float> w;
    init_weights(seed, w);
    if ((rc = vox_lpc_set_weights(L, w.data()))) return bail(rc);
    *out = L;
    return VOX_OK;
}

int vox_lpc_destroy(vox_lpc* L)
{
    if (!L) return VOX_OK;
    (void)hipSetDevice(L->device);
    if (L->stream) (void)hipStreamSynchronize(L->stream);
    for (auto& S : L->sys) {
        lfree(S.rowlen); lfree(S.acol); lfree(S.slen); lfree(S.scol); lfree(S.aval); lfree(S.diag);
        lfree(S.inv_d); lfree(S.inv_osum); lfree(S.feat); lfree(S.rhs); lfree(S.sval);
    }
    for (auto*& p : L->h) lfree(p);
    for (auto*& p : L->s) lfree(p);
    for (auto*& p : L->m) lfree(p);
    for (float** p : {&L->o, &L->g, &L->c, &L->sc, &L->wv, &L->vv, &L->t, &L->z, &L->e, &L->y, &L->ys,
                      &L->dO, &L->dh[0], &L->dh[1], &L->dmh, &L->ds, &L->w32, &L->grad, &L->am, &L->av,
                      &L->gpart})
        lfree(*p);
    lfree(L->epart);
    lfree(L->w16); lfree(L->dpart); lfree(L->dscal);
    if (L->hscal) (void)hipHostFree(L->hscal);
    if (L->hgrad) (void)hipHostFree(L->hgrad);
    if (L->stream) (void)hipStreamDestroy(L->stream);
    delete L;
    return VOX_OK;
}

int vox_lpc_get_weights(vox_lpc* L, float* w)
{
    VOX_TRY(check_lpc(L));
    if (!w) return fail(VOX_ERR_ARG, "null weights");
    VOX_HIP(hipMemcpyAsync(w, L->w32, sizeof(float) * NPARAM, hipMemcpyDeviceToHost, L->stream));
    VOX_HIP(hipStreamSynchronize(L->stream));
    return VOX_OK;
}

int vox_lpc_set_weights(vox_lpc* L, const float* w)
{
    VOX_TRY(check_lpc(L));
    if (!w) return fail(VOX_ERR_ARG, "null weights");
    for (int k = 0; k < NPARAM; ++k)
        if (!std::isfinite(w[k])) return fail(VOX_ERR_ARG, "non-finite weight");
    VOX_HIP(hipMemcpyAsync(L->w32, w, sizeof(float) * NPARAM, hipMemcpyHostToDevice, L->stream));
    k_lpc_cast<<<grid_for(NPARAM), kBlock, 0, L->stream>>>(NPARAM, L->w32, L->w16);
    VOX_HIP(hipGetLastError());
    // a fresh set of weights restarts the optimiser
    VOX_HIP(hipMemsetAsync(L->am, 0, sizeof(float) * NPARAM, L->stream));
    VOX_HIP(hipMemsetAsync(L->av, 0, sizeof(float) * NPARAM, L->stream));
    VOX_HIP(hipStreamSynchronize(L->stream));
    L->adam_t = 0;
    return VOX_OK;
}

int vox_lpc_dump(vox_lpc* L, vox_ctx* c, int32_t* index)
{
    VOX_TRY(check_lpc(L));
    if (!c) return fail(VOX_ERR_ARG, "null context");
    if (c->device != L->device) return fail(VOX_ERR_ARG, "context and network on different devices");
    if (!c->acol || c->nu <= 0) return fail(VOX_ERR_STATE, "no assembled PPE in the context");
    if (c->uorder_cells) {
        // training systems are dumped with the unknowns in particle order, the
        // order of vox_ppe_export: the system is assembled again in that order
        c->uorder_particles = true;
        const int rc0 = ppe_assemble(c);
        c->uorder_particles = false;
        VOX_TRY(rc0);
    }
    if (!c->aval32_ok) VOX_TRY(ppe_make_aval32(c));
    VOX_TRY(ensure_acol(c));
    LpcSys S;
    S.nu = c->nu; S.rows = round64(c->nu); S.cap = c->a_cap;
    const size_t nn = (size_t)S.rows, mat = (size_t)sl_size(S.nu, S.cap);
    int rc;
    v4f* upos = nullptr;
    auto cleanup = [&]() {
        lfree(S.rowlen); lfree(S.acol); lfree(S.slen); lfree(S.scol); lfree(S.aval); lfree(S.diag);
        lfree(S.inv_d); lfree(S.inv_osum); lfree(S.feat); lfree(S.rhs); lfree(S.sval); lfree(upos);
    };
    auto alloc = [&](auto** p, size_t n) { return lalloc(c->stream, p, n); };
    if ((rc = alloc(&S.rowlen, nn)) || (rc = alloc(&S.acol, mat)) || (rc = alloc(&S.aval, mat)) ||
        (rc = alloc(&S.slen, nn)) || (rc = alloc(&S.scol, mat)) || (rc = alloc(&S.sval, mat)) ||
        (rc = alloc(&S.diag, nn)) || (rc = alloc(&S.inv_d, nn)) || (rc = alloc(&S.inv_osum, nn)) ||
        (rc = alloc(&S.feat, nn * LF)) || (rc = alloc(&S.rhs, nn)) || (rc = alloc(&upos, nn))) {
        cleanup();
        return rc;
    }
    hipStream_t st = c->stream;
    if (hipMemcpyAsync(S.rowlen, c->rowlen, sizeof(int32_t) * S.nu, hipMemcpyDeviceToDevice, st) != hipSuccess ||
        hipMemcpyAsync(S.acol, c->acol, sizeof(int32_t) * mat, hipMemcpyDeviceToDevice, st) != hipSuccess ||
        hipMemcpyAsync(S.aval, c->aval32, sizeof(float) * mat, hipMemcpyDeviceToDevice, st) != hipSuccess) {
        cleanup();
        return fail(VOX_ERR_HIP, "dump copy");
    }
    k_lpc_dump_rows<<<grid_for(S.nu), kBlock, 0, st>>>(S.nu, c->adiag, c->rhs, S.diag, S.rhs);
    ctx_features(c, S.rows, upos, S.inv_d, S.feat, S.inv_osum, S.slen, S.scol, S.sval);
    k_lpc_oh<<<grid_for(S.nu), kBlock, 0, st>>>(S.nu, S.cap, S.slen, S.scol, S.inv_d, S.sval);
    if (hipGetLastError() != hipSuccess || hipStreamSynchronize(st) != hipSuccess) {
        cleanup();
        return fail(VOX_ERR_HIP, "dump kernels");
    }
    lfree(upos);
    if ((rc = lpc_training_buffers(L, S.rows))) {
        cleanup();
        return rc;
    }
    L->sys.push_back(S);
    if (index) *index = (int32_t)L->sys.size() - 1;
    return VOX_OK;
}

int vox_lpc_count(vox_lpc* L, int32_t* systems, int64_t* rows)
{
    VOX_TRY(check_lpc(L));
    if (systems) *systems = (int32_t)L->sys.size();
    if (rows) {
        int64_t t = 0;
        for (auto& S : L->sys) t += S.nu;
        *rows = t;
    }
    return VOX_OK;
}

int vox_lpc_eval(vox_lpc* L, int32_t index, float* feat, float* g, float* c)
{
    VOX_TRY(check_lpc(L));
    VOX_TRY(check_index(L, index));
    const LpcSys& S = L->sys[index];
    VOX_TRY(lpc_forward_sys(L, S));
    if (feat) VOX_HIP(hipMemcpyAsync(feat, S.feat, sizeof(float) * LF * S.nu, hipMemcpyDeviceToHost, L->stream));
    if (g) VOX_HIP(hipMemcpyAsync(g, L->g, sizeof(float) * S.nu, hipMemcpyDeviceToHost, L->stream));
    if (c) VOX_HIP(hipMemcpyAsync(c, L->c, sizeof(float) * S.nu, hipMemcpyDeviceToHost, L->stream));
    VOX_HIP(hipStreamSynchronize(L->stream));
    return VOX_OK;
}

int vox_lpc_loss_grad(vox_lpc* L, int32_t index, uint64_t seed, double* loss, float* grad)
{
    VOX_TRY(check_lpc(L));
    VOX_TRY(check_index(L, index));
    VOX_TRY(lpc_loss_grad_sys(L, L->sys[index], seed));
    VOX_HIP(hipMemcpyAsync(L->hscal, L->dscal, sizeof(double) * LS_COUNT, hipMemcpyDeviceToHost, L->stream));
    std::lock_guard<std::mutex> lock(L->hgrad_m);
    if (grad) VOX_HIP(hipMemcpyAsync(L->hgrad, L->grad, sizeof(float) * NPARAM, hipMemcpyDeviceToHost, L->stream));
    VOX_HIP(hipStreamSynchronize(L->stream));
    if (grad) std::memcpy(grad, L->hgrad, sizeof(float) * NPARAM);
    if (loss) *loss = L->hscal[LS_LOSS];
    return VOX_OK;
}

int vox_lpc_train(vox_lpc* L, int32_t epochs, double lr, uint64_t seed, double* loss_first, double* loss_last)
{
    VOX_TRY(check_lpc(L));
    if (epochs < 1 || !(lr > 0)) return fail(VOX_ERR_ARG, "epochs >= 1 and lr > 0 required");
    const int ns = (int)L->sys.size();
    if (ns == 0) return fail(VOX_ERR_STATE, "no stored systems to train on");
    std::vector<int> order(ns);
    std::iota(order.begin(), order.end(), 0);
    uint64_t st = seed ^ 0xD1B54A32D192ED03ull;
    auto next = [&]() {
        uint64_t z = (st += 0x9E3779B97F4A7C15ull);
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        return z ^ (z >> 31);
    };
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    for (int ep = 0; ep < epochs; ++ep) {
        for (int k = ns - 1; k > 0; --k) std::swap(order[k], order[(int)(next() % (uint64_t)(k + 1))]);
        k_lpc_set<<<1, 1, 0, L->stream>>>(L->dscal, LS_EPOCH, 0.0);
        for (int k = 0; k < ns; ++k) {
            const int i = order[k];
            VOX_TRY(lpc_loss_grad_sys(L, L->sys[i], seed + (uint64_t)ep * 1000003ull + (uint64_t)i));
            k_lpc_epoch<<<1, 1, 0, L->stream>>>(L->dscal);
            ++L->adam_t;
            const float bc1 = 1.f - std::pow(b1, (float)L->adam_t);
            const float bc2 = 1.f - std::pow(b2, (float)L->adam_t);
            k_lpc_adam<<<grid_for(NPARAM), kBlock, 0, L->stream>>>(NPARAM, L->w32, L->grad, L->am, L->av,
                                                                   (float)lr, b1, b2, eps, bc1, bc2, L->w16);
            VOX_HIP(hipGetLastError());
        }
        VOX_HIP(hipMemcpyAsync(L->hscal, L->dscal, sizeof(double) * LS_COUNT, hipMemcpyDeviceToHost, L->stream));
        VOX_HIP(hipStreamSynchronize(L->stream));
        const double mean = L->hscal[LS_EPOCH] / ns;
        if (!std::isfinite(mean)) return fail(VOX_ERR_SOLVER, "training loss is not finite");
        if (ep == 0 && loss_first) *loss_first = mean;
        if (loss_last) *loss_last = mean;
    }
    return VOX_OK;
}

int vox_attach_lpc(vox_ctx* c, vox_lpc* L)
{
    if (!c) return fail(VOX_ERR_ARG, "null context");
    if (L && L->device != c->device) return fail(VOX_ERR_ARG, "context and network on different devices");
    c->lpc = L;
    c->lpc_baseline = 0;
    return VOX_OK;
}

}  // extern "C"
