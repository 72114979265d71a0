// gfx950 kernels of the radial-descriptor MLP potential (mlp_kernels.hpp).
//
// The network runs on MFMA v_mfma_f32_16x16x16_bf16 with the activations kept
// transposed (features x particles): a layer's 16x16 output block in the
// accumulator layout (lane l holds rows 4(l/16)..4(l/16)+3 of column l%16) is
// exactly the B-operand layout of the next layer's K block, so no data moves
// between layers.  Weights are the A operands, converted to BF16 once per wave
// and held in registers while the wave walks its 16-particle tiles.  The
// first layer (and its transpose in the input gradient) carries each operand
// as a pair of BF16 values hi + lo, three MFMAs per block: the energy is a
// nearly linear function of correlated descriptors, and single-BF16 inputs
// cost more accuracy than the network gains over a linear fit.
// The library is compiled with -ffp-contract=off; the FP32 math here uses
// explicit fmaf where a fused multiply-add is wanted.
#include <algorithm>

#include "md_segment.hpp"
#include "mlp_kernels.hpp"

namespace pk {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// FP32 -> BF16, round to nearest even: the hardware's conversion of two values
typedef __bf16 hwbf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack2(float a, float b) {
    const f32x2 f = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, hwbf16x2));
}
__device__ __forceinline__ short f2bf(float f) { return (short) pack2(f, f); }
__device__ __forceinline__ bf16x4 pack4(float a, float b, float c, float d) {
    const uint2 u = make_uint2(pack2(a, b), pack2(c, d));
    return __builtin_bit_cast(bf16x4, u);
}
__device__ __forceinline__ bf16x4 pack4(const f32x4 &x) { return pack4(x[0], x[1], x[2], x[3]); }
__device__ __forceinline__ float bf2f(short b) { return __uint_as_float(((uint32_t) (uint16_t) b) << 16); }
// x = hi + lo with hi = bf16(x), lo = bf16(x - hi): a pair carries 16 mantissa bits
__device__ __forceinline__ void split4(float a, float b, float c, float d, bf16x4 &hi, bf16x4 &lo) {
    hi = pack4(a, b, c, d);
    lo = pack4(a - bf2f(hi[0]), b - bf2f(hi[1]), c - bf2f(hi[2]), d - bf2f(hi[3]));
}
__device__ __forceinline__ void split4(const f32x4 &x, bf16x4 &hi, bf16x4 &lo) { split4(x[0], x[1], x[2], x[3], hi, lo); }

__device__ __forceinline__ f32x4 mfma16(bf16x4 a, bf16x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

// SiLU and its derivative
__device__ __forceinline__ void silu(float z, float &h, float &dh) {
    const float sg = __builtin_amdgcn_rcpf(1.0f + __expf(-z));
    h = z * sg;
    dh = sg * fmaf(z, 1.0f - sg, 1.0f);
}

// ---------------------------------------------------------------- network tile

// The network of a workgroup in LDS: the A operands of every MFMA, converted
// to BF16 once and laid out by fragment and lane (lane l: q = l / 16, col = l %
// 16), and the FP32 constants.  In registers, one set per wave, they took 96 of
// 243 registers and left two waves on a SIMD; a read from LDS is one
// conflict-free 8-byte access per fragment and four waves fit (k_mlp_eval,
// 131072 rows: 22.3 -> 18.1 us).
enum {
    NF_A1 = 0,     // W1 rows 16c + col, columns 4q..4q+3 (high BF16 part)
    NF_A1L = 4,    // W1 - a1 (low part: the first layer runs at ~16-bit precision)
    NF_A2 = 8,     // W2 [c][kc]: rows 16c + col, columns 16kc + 4q..
    NF_A2T = 24,   // W2^T [c][kc]: W2[16kc + 4q + v][16c + col]
    NF_A1T = 40,   // W1^T [kc]: W1[16kc + 4q + v][col] (high part)
    NF_A1TL = 44,  // its low part
    NF_COUNT = 48
};
struct MLPNet {
    bf16x4 f[NF_COUNT][64];
    f32x4 b1[4][4], b2[4][4], w3[4][4];  // [c][q]: rows 16c + 4q + v
    f32x4 gm[4], gi[4];                  // [q]: features 4q + v
    float b3, em, es;
};

// the waves of a workgroup of NT threads convert the fragments in turn, every
// load in flight before the first conversion; ends with a barrier
template <bool BACK, int NT>
__device__ __forceinline__ void mlp_stage(MLPNet &N, const float *__restrict__ p, const float *__restrict__ sc) {
    constexpr int NF = BACK ? NF_COUNT : NF_A2T, IT = (NF * 64 + NT - 1) / NT;
    const int lane = threadIdx.x & 63, q = lane >> 4, col = lane & 15;
    const int wl = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    float w[IT][4], c[5] = {0.f, 0.f, 0.f, 0.f, 0.f}, y[3] = {0.f, 0.f, 0.f};
#pragma unroll
    for (int it = 0; it < IT; it++) {
        const int f = it * (NT / 64) + wl;
        if (f >= NF) break;
        const bool rows = f < NF_A2T;  // of W, else of W^T
        const float *m;
        if (f < NF_A2) m = p + MLP_W1 + (16 * (f & 3) + col) * MLP_ND + 4 * q;
        else if (rows) m = p + MLP_W2 + (16 * ((f - NF_A2) >> 2) + col) * MLP_H + 16 * (f & 3) + 4 * q;
        else if (f < NF_A1T) m = p + MLP_W2 + (16 * (f & 3) + 4 * q) * MLP_H + 16 * ((f - NF_A2T) >> 2) + col;
        else m = p + MLP_W1 + (16 * (f & 3) + 4 * q) * MLP_ND + col;
        const int step = rows ? 1 : f < NF_A1T ? MLP_H : MLP_ND;
#pragma unroll
        for (int v = 0; v < 4; v++) w[it][v] = m[v * step];
    }
    if (wl == 0) {
        c[0] = p[MLP_B1 + lane]; c[1] = p[MLP_B2 + lane]; c[2] = p[MLP_W3 + lane];
        if (lane < 16) { c[3] = sc[MLP_GMEAN + lane]; c[4] = sc[MLP_GISTD + lane]; }
        y[0] = p[MLP_B3]; y[1] = sc[MLP_EMEAN]; y[2] = sc[MLP_ESTD];
    }
#pragma unroll
    for (int it = 0; it < IT; it++) {
        const int f = it * (NT / 64) + wl;
        if (f >= NF) break;
        bf16x4 hi, lo;
        split4(w[it][0], w[it][1], w[it][2], w[it][3], hi, lo);
        N.f[f][lane] = (f >= NF_A1L && f < NF_A2) || f >= NF_A1TL ? lo : hi;
    }
    if (wl == 0) {
        ((float *) N.b1)[lane] = c[0]; ((float *) N.b2)[lane] = c[1]; ((float *) N.w3)[lane] = c[2];
        if (lane < 16) { ((float *) N.gm)[lane] = c[3]; ((float *) N.gi)[lane] = c[4]; }
        if (lane == 0) { N.b3 = y[0]; N.em = y[1]; N.es = y[2]; }
    }
    __syncthreads();
}

// keeps the compiler from hoisting a tile loop's LDS reads into registers
__device__ __forceinline__ void mlp_keep_in_lds() { asm volatile("" ::: "memory"); }

// one lane's view of the network
struct MLPView {
    const MLPNet &N;
    int lane, q;
    __device__ __forceinline__ bf16x4 f(int k) const { return N.f[k][lane]; }
    __device__ __forceinline__ f32x4 b1(int c) const { return N.b1[c][q]; }
    __device__ __forceinline__ f32x4 b2(int c) const { return N.b2[c][q]; }
    __device__ __forceinline__ f32x4 w3(int c) const { return N.w3[c][q]; }
    __device__ __forceinline__ float4 gi() const {
        const f32x4 g = N.gi[q];
        return make_float4(g[0], g[1], g[2], g[3]);
    }
};

// standardised descriptors of the lane's particle, features 4q..4q+3
__device__ __forceinline__ f32x4 mlp_input(const MLPView &R, float4 g) {
    const f32x4 gm = R.N.gm[R.q], gi = R.N.gi[R.q];
    f32x4 s;
    s[0] = (g.x - gm[0]) * gi[0];
    s[1] = (g.y - gm[1]) * gi[1];
    s[2] = (g.z - gm[2]) * gi[2];
    s[3] = (g.w - gm[3]) * gi[3];
    return s;
}

// W1 x of output block c with both operands split: hi*hi + lo*hi + hi*lo
__device__ __forceinline__ f32x4 mlp_layer1(const MLPView &R, int c, bf16x4 b0, bf16x4 b0l) {
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    const bf16x4 a1 = R.f(NF_A1 + c);
    f32x4 z = mfma16(R.f(NF_A1L + c), b0, zero);
    z = mfma16(a1, b0l, z);
    return mfma16(a1, b0, z);
}

// forward pass of one 16-particle tile: returns y of particle col (all four
// lane groups hold it); keeps activations and SiLU derivatives
__device__ __forceinline__ float mlp_forward(const MLPView &R, bf16x4 b0, bf16x4 b0l, f32x4 (&h1)[4],
                                             f32x4 (&dh1)[4], bf16x4 (&bh1)[4], f32x4 (&h2)[4], f32x4 (&dh2)[4]) {
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < 4; c++) {
        const f32x4 z = mlp_layer1(R, c, b0, b0l), b1 = R.b1(c);
#pragma unroll
        for (int v = 0; v < 4; v++) {
            float h, dh;
            silu(z[v] + b1[v], h, dh);
            h1[c][v] = h;
            dh1[c][v] = dh;
        }
        bh1[c] = pack4(h1[c]);
    }
#pragma unroll
    for (int c = 0; c < 4; c++) {
        f32x4 z = zero;
        const f32x4 b2 = R.b2(c);
#pragma unroll
        for (int kc = 0; kc < 4; kc++) z = mfma16(R.f(NF_A2 + 4 * c + kc), bh1[kc], z);
#pragma unroll
        for (int v = 0; v < 4; v++) {
            float h, dh;
            silu(z[v] + b2[v], h, dh);
            h2[c][v] = h;
            dh2[c][v] = dh;
        }
    }
    float y = 0.f;
#pragma unroll
    for (int c = 0; c < 4; c++) {
        const f32x4 w3 = R.w3(c);
#pragma unroll
        for (int v = 0; v < 4; v++) y = fmaf(w3[v], h2[c][v], y);
    }
    y += __shfl_xor(y, 16, 64);
    y += __shfl_xor(y, 32, 64);
    return y + R.N.b3;
}

// dy/d(standardised descriptor) of particle col, features 4q..4q+3
__device__ __forceinline__ f32x4 mlp_input_grad(const MLPView &R, const f32x4 (&dh1)[4], const f32x4 (&dh2)[4]) {
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    bf16x4 bg2[4], bg1[4], bg1l[4];
#pragma unroll
    for (int c = 0; c < 4; c++) {
        const f32x4 w3 = R.w3(c);
        bg2[c] = pack4(w3[0] * dh2[c][0], w3[1] * dh2[c][1], w3[2] * dh2[c][2], w3[3] * dh2[c][3]);
    }
#pragma unroll
    for (int c = 0; c < 4; c++) {
        f32x4 a = zero;
#pragma unroll
        for (int kc = 0; kc < 4; kc++) a = mfma16(R.f(NF_A2T + 4 * c + kc), bg2[kc], a);
        split4(a[0] * dh1[c][0], a[1] * dh1[c][1], a[2] * dh1[c][2], a[3] * dh1[c][3], bg1[c], bg1l[c]);
    }
    // W1^T g1, both split like the forward first layer
    f32x4 d = zero;
#pragma unroll
    for (int kc = 0; kc < 4; kc++) {
        const bf16x4 a1t = R.f(NF_A1T + kc);
        d = mfma16(R.f(NF_A1TL + kc), bg1[kc], d);
        d = mfma16(a1t, bg1l[kc], d);
        d = mfma16(a1t, bg1[kc], d);
    }
    return d;
}

// E and dE/dG (raw descriptor units) of n rows; one wave per 16-row tile.
// IMG: the rows are the locals of a force evaluation, and a local's dE/dG goes
// to its ghost images too (im.on), in place of a copy pass over the ghosts.
template <bool WANT_D, bool IMG, int NT>
__global__ __launch_bounds__(NT) void k_mlp_eval(const float *__restrict__ p, const float *__restrict__ sc,
                                                  const float *__restrict__ G, int n, float *__restrict__ E,
                                                  float *__restrict__ D, Images im) {
    const int lane = threadIdx.x & 63, q = lane >> 4, col = lane & 15;
    const int wave = blockIdx.x * (NT / 64) + (threadIdx.x >> 6), nw = gridDim.x * (NT / 64);
    const int ntiles = (n + 15) >> 4;
    __shared__ MLPNet N;
    // a tile's rows are loaded a turn ahead, the first before the weights
    float4 g = make_float4(0.f, 0.f, 0.f, 0.f);
    int ni = 0;
    const auto load = [&](int t) __attribute__((always_inline)) {
        const int row = t * 16 + col;
        if (row >= n) return;
        g = *(const float4 *) (G + (size_t) row * MLP_ND + 4 * q);
        if (IMG && im.on) ni = min(im.cnt[row], IMG_MAX);
    };
    load(wave);
    mlp_stage<WANT_D, NT>(N, p, sc);
    for (int t = wave; t < ntiles; t += nw) {
        mlp_keep_in_lds();
        const MLPView R{N, lane, q};
        const int row = t * 16 + col;
        const bool ok = row < n;
        bf16x4 b0, b0l;
        split4(mlp_input(R, g), b0, b0l);
        const int images = ni;
        load(t + nw);
        f32x4 h1[4], dh1[4], h2[4], dh2[4];
        bf16x4 bh1[4];
        const float y = mlp_forward(R, b0, b0l, h1, dh1, bh1, h2, dh2);
        if (ok && q == 0 && E) E[row] = fmaf(R.N.es, y, R.N.em);
        if (WANT_D) {
            const f32x4 d = mlp_input_grad(R, dh1, dh2);
            const float4 gi = R.gi();
            if (ok) {
                float4 o;
                o.x = R.N.es * d[0] * gi.x;
                o.y = R.N.es * d[1] * gi.y;
                o.z = R.N.es * d[2] * gi.z;
                o.w = R.N.es * d[3] * gi.w;
                *(float4 *) (D + (size_t) row * MLP_ND + 4 * q) = o;
                if (IMG && im.on) {
                    for (int k = 0; k < images; k++) {
                        const int gq = im.tab[(size_t) k * im.cap + row].x;
                        *(float4 *) (D + (size_t) (n + gq) * MLP_ND + 4 * q) = o;
                    }
                }
            }
        }
    }
}

// ---------------------------------------------------------------- descriptors and forces

// log2(e) / (2 w^2): exp(-t^2 / (2 w^2)) = exp2(-t^2 * MLP_C)
constexpr float MLP_C = 1.4426950408889634f / (2.0f * MLP_W * MLP_W);
constexpr float MLP_IW2 = 1.0f / (MLP_W * MLP_W);
constexpr float MLP_PIRC = 3.14159265358979323846f / (float) MLP_RC;

struct MLPSegArgs {
    const int *counters;
    const double *X, *Y, *Z;
    const double4 *P;    // (x, y, z, type) of X, Y, Z packed: one 16-byte and one 8-byte gather
    const uint32_t *nl;
    int nl_stride;
    const int *numneighs;
    int ncap;            // list rows: counts are clamped to it
    int pstride;
    const float *D, *E;
    float *G;
    double *fx, *fy, *fz;
    double *partials;
    const float4 *rho;   // MODE 2: dL/dF of every slot (a ghost holds its root's)
    const float *sc;     // MODE 2: standardisation (e_std, g_istd)
    float *U;            // MODE 2: [cap][16] back-projected directions
    // MODE 1 without RED, vv set: the integration of k_vv_post fused behind
    // the force (final_integrate(ts) if vv2, initial_integrate(ts+1) and the
    // next positions and images if vv1)
    int vv, vv2, vv1;
    double dt, hdt;
    const int *flags, *type;
    const double *mass;
    double *vx, *vy, *vz;
    double *Xn, *Yn, *Zn;
    double4 *Pn;         // packed copy of the next positions, or null
    Images im;
    Geom g;
};

// G of the 32 locals of one wave (MODE 0), or their force, energy and
// virial (MODE 1), or (MODE 2) the back-projection of force residuals onto
// the descriptor gradients: with rho_i = dL/dF_i and F_i = -sum_j w_ij .
// (D_i + D_j), w_ij,k = dphi_k(r_ij) (x_i - x_j) / r_ij,
//   dL/dD_a,k = -sum_{j in list(a)} w_aj,k . (rho_a - rho_j),
// written as U_a,k = e_std g_istd,k dL/dD_a,k (the direction the network's
// input gradient is differentiated along).  L lanes per local (2, or 4 for
// small systems): lane L p + h walks entries 4s + L q + h of local p's list
// (one 16-byte group of four per step), the L partial sums are added across
// the lanes at the end (FP32 / FP64 sums in any order: the potential is not
// bit-matched to a reference), so L times as many waves hide the gathers'
// latency.  Pairs at r >= 2.5 and entries past a lane's count are masked.
//
// Bound by vector work (210 operations per pair in MODE 1, 67 us' worth at
// 131072 atoms) and, as each lane gathered its partners' rows by itself, by the
// cache-line look-ups of those gathers (6 per pair in MODE 1, 107 us' worth at
// one a cycle and CU).  So on two lanes per local MODE 1 loads each position
// record with one instruction of the lane pair (x, y on one lane, z on the
// other, swapped by DPP) and each 64-byte row of dE/dG with four lanes, handed
// over through LDS (the chunks of a row are rotated by lane group: no bank
// conflicts on either side): 2 look-ups per pair, the arithmetic unchanged.
// 131072 atoms: MODE 1 89 -> 78 us, MODE 0 42 -> 39.  On four lanes (small
// systems) the hand-over only lengthens a step's chain (16.6 -> 20 us at 2048
// atoms), and in MODE 0 the swap costs more than the look-ups (39 -> 48): both
// gather directly.
template <int MODE, bool RED, int L>
__global__ __launch_bounds__(64) void k_mlp_wave(MLPSegArgs A) {
    constexpr int U = 4 / L;  // entries per lane per step
    constexpr bool ROWS = MODE == 1 && L == 2;  // dE/dG rows loaded by four lanes each
    __shared__ __align__(16) float4 s_d[ROWS ? 256 : 1];
    const int wv = xcd_block(blockIdx.x, gridDim.x);
    const int lane = threadIdx.x & 63, h = lane & (L - 1), odd = lane & 1;
    const int nlocal = A.counters[C_NLOCAL];
    const uint32_t jmax = (uint32_t) max(nlocal + A.counters[C_NGHOST] - 1, 0);
    const char *__restrict__ P = (const char *) A.P;
    const double rc2 = MLP_RC * MLP_RC;
    double pe = 0.0, vir = 0.0;
    const int i0 = wv * (64 / L);
    if (i0 < nlocal) {  // wave-uniform
        const int i = i0 + lane / L;
        const bool live = i < nlocal;
        const int ii = live ? i : i0;
        const int n = live ? min(A.numneighs[ii], A.ncap) : 0;
        const int nmax = wave_max_uniform(n);
        const double xi = A.X[ii], yi = A.Y[ii], zi = A.Z[ii];
        float acc[MLP_ND], di[MLP_ND];
#pragma unroll
        for (int k = 0; k < MLP_ND; k++) acc[k] = 0.f;
        if (MODE == 1) {
            const float4 *dp = (const float4 *) (A.D + (size_t) ii * MLP_ND);
#pragma unroll
            for (int k4 = 0; k4 < 4; k4++) {
                const float4 d = dp[k4];
                di[4 * k4] = d.x; di[4 * k4 + 1] = d.y; di[4 * k4 + 2] = d.z; di[4 * k4 + 3] = d.w;
            }
        }
        const float4 rhoi = MODE == 2 ? A.rho[ii] : make_float4(0.f, 0.f, 0.f, 0.f);
        double f0 = 0.0, f1 = 0.0, f2 = 0.0, w = 0.0;
        const float gb = exp2f(-2.0f * MLP_DMU * MLP_DMU * MLP_C);  // a_{k+1} / a_k
        const uint4 *lp = (const uint4 *) A.nl + ii;
        const int gl = max((n + 3) / 4 - 1, 0);
        const int nst = (nmax + 3) / 4;
        // the lane's chunk of the records the wave loads together: record
        // 16 m + lane / 4, chunk rotated by the record's group of four
        const int rsub = lane >> 2, rot = (lane >> 2) & 3;
        const int chunk_in = (lane & 3) ^ ((rsub >> 2) & 3);
        for (int st = 0; st < nst; st++) {
            // groups past the lane's list re-read its last group; entries past
            // its count read the spare record behind the last slot (zero times the
            // distance to a particle at infinity would be NaN), entries are
            // clamped to the last particle slot
            const uint4 grp = lp[(size_t) min(st, gl) * A.nl_stride];
            uint32_t jq[U];
#pragma unroll
            for (int q = 0; q < U; q++) {
                const int c = L * q + h;
                // (a group holds its entries as 0, 2, 1, 3)
                const uint32_t e = (c & 2) ? ((c & 1) ? grp.w : grp.y) : ((c & 1) ? grp.z : grp.x);
                jq[q] = 4 * st + c < n ? min(e, jmax) : (uint32_t) A.nl_stride;
            }
            struct Ent { double2 a, b; float4 d0, d1, d2, d3, rho; };
            auto gather = [&](uint32_t j, Ent &e) __attribute__((always_inline)) {
                if (!ROWS) {
                    e.a = *(const double2 *) (P + (j << 5));
                    e.b.x = *(const double *) (P + (j << 5) + 16);
                    if (MODE == 1) {
                        const float4 *dp = (const float4 *) (A.D + (size_t) j * MLP_ND);
                        e.d0 = dp[0]; e.d1 = dp[1]; e.d2 = dp[2]; e.d3 = dp[3];
                    }
                    if (MODE == 2) e.rho = A.rho[j];
                    return;
                }
                const uint32_t jp = (uint32_t) __builtin_amdgcn_mov_dpp((int) j, 0xB1, 0xF, 0xF, true);
                const uint32_t je = odd ? jp : j, jo = odd ? j : jp;
                e.a = *(const double2 *) (P + ((je << 5) + (odd ? 16u : 0u)));
                e.b = *(const double2 *) (P + ((jo << 5) + (odd ? 0u : 16u)));
                auto row = [&](int m) {
                    return *((const float4 *) (A.D + (size_t) __shfl((int) j, 16 * m + rsub, 64) * MLP_ND) + chunk_in);
                };
                e.d0 = row(0); e.d1 = row(1); e.d2 = row(2); e.d3 = row(3);
            };
            auto pair = [&](int q, const Ent &e) __attribute__((always_inline)) {
                const double2 xy = ROWS && odd ? e.b : e.a;
                const double zj = ROWS ? pair_swap(odd ? e.a.x : e.b.x) : e.b.x;
                const double dx = xi - xy.x, dy = yi - xy.y, dz = zi - zj;
                double rsq = dx * dx + dy * dy;
                rsq = rsq + dz * dz;
                const bool in = (4 * st + L * q + h < n) && rsq < rc2;
                // masked entries take an in-range stand-in distance, so the
                // Gaussian recurrence below stays finite; 1/r from the
                // hardware reciprocal square root, r = rsq / r
                const float rsqf = (float) rsq;
                const float rinv = in ? __builtin_amdgcn_rsqf(rsqf) : 1.0f / MLP_MU0;
                const float r = in ? rsqf * rinv : MLP_MU0;
                // g_k by recurrence over the uniform centres,
                // g_{k+1} = g_k a_k, a_{k+1} = a_k b, from two directly
                // computed anchors (k = 0 and k = 8): four exponentials per
                // pair instead of sixteen, relative error below 1e-5
                const float t0 = r - MLP_MU0;
                // (arguments in the normal range of exp2, |t| < 1.8: the
                // hardware's exponential as it is)
                auto anchor = [&](int k0, float &g, float &a) {
                    const float t = t0 - (float) k0 * MLP_DMU;
                    g = __builtin_amdgcn_exp2f(-(t * t) * MLP_C);
                    a = __builtin_amdgcn_exp2f((2.0f * t - MLP_DMU) * MLP_DMU * MLP_C);
                };
                float gk, ak;
                if (MODE == 0) {
                    const float fc = in ? 0.5f * (cosf(MLP_PIRC * r) + 1.0f) : 0.0f;
#pragma unroll
                    for (int kk = 0; kk < MLP_ND; kk++) {
                        if (kk % 8 == 0) anchor(kk, gk, ak);
                        acc[kk] = fmaf(gk, fc, acc[kk]);
                        gk *= ak;
                        ak *= gb;
                    }
                } else if (MODE == 2) {
                    // the cutoff's sine and cosine from the hardware units
                    // (argument in turns: pi r / rc = 2 pi (r / 2 rc), r < rc)
                    const float ang = r * (0.5f / (float) MLP_RC);
                    const float sn = __builtin_amdgcn_sinf(ang), cs = __builtin_amdgcn_cosf(ang);
                    const float fc = 0.5f * (cs + 1.0f), dfc = -0.5f * MLP_PIRC * sn;
                    // (x_a - x_j) / r . (rho_a - rho_j), zero for a masked entry
                    float proj = (float) dx * (rhoi.x - e.rho.x) + (float) dy * (rhoi.y - e.rho.y);
                    proj = proj + (float) dz * (rhoi.z - e.rho.z);
                    proj = in ? -proj * rinv : 0.0f;
#pragma unroll
                    for (int kk = 0; kk < MLP_ND; kk++) {
                        if (kk % 8 == 0) anchor(kk, gk, ak);
                        const float t = t0 - (float) kk * MLP_DMU;
                        const float dphi = gk * fmaf(-t * MLP_IW2, fc, dfc);
                        acc[kk] = fmaf(dphi, proj, acc[kk]);
                        gk *= ak;
                        ak *= gb;
                    }
                } else {
                    // this lane's row, from the lanes that loaded its chunks
                    if (ROWS) {
                        s_d[lane] = e.d0; s_d[64 + lane] = e.d1; s_d[128 + lane] = e.d2; s_d[192 + lane] = e.d3;
                        wave_lds_sync();
                    }
                    const float ang = r * (0.5f / (float) MLP_RC);
                    const float sn = __builtin_amdgcn_sinf(ang), cs = __builtin_amdgcn_cosf(ang);
                    const float fc = 0.5f * (cs + 1.0f), dfc = -0.5f * MLP_PIRC * sn;
                    float ci = 0.f, cj = 0.f;
#pragma unroll
                    for (int k4 = 0; k4 < 4; k4++) {
                        const float4 d4 = ROWS ? s_d[4 * lane + (k4 ^ rot)] : k4 == 0 ? e.d0 : k4 == 1 ? e.d1 : k4 == 2 ? e.d2 : e.d3;
                        const float dq[4] = {d4.x, d4.y, d4.z, d4.w};
#pragma unroll
                        for (int v = 0; v < 4; v++) {
                            const int kk = 4 * k4 + v;
                            if (kk % 8 == 0) anchor(kk, gk, ak);
                            const float t = t0 - (float) kk * MLP_DMU;
                            const float dphi = gk * fmaf(-t * MLP_IW2, fc, dfc);
                            ci = fmaf(di[kk], dphi, ci);
                            cj = fmaf(dq[v], dphi, cj);
                            gk *= ak;
                            ak *= gb;
                        }
                    }
                    if (ROWS) wave_lds_sync();
                    const float cc = ci + cj;
                    const double coef = in ? (double) (-cc * rinv) : 0.0;
                    f0 += coef * dx; f1 += coef * dy; f2 += coef * dz;
                    if (RED) w += in ? (double) (-cc * r) : 0.0;
                }
            };
            Ent e0, e1;
            gather(jq[0], e0);
            if (U == 2) gather(jq[U - 1], e1);
            pair(0, e0);
            if (U == 2) pair(U - 1, e1);
        }
        // the L lanes of a local: partial sums added
#pragma unroll
        for (int o = 1; o < L; o <<= 1) {
            if (MODE == 1) {
                f0 += __shfl_xor(f0, o, 64);
                f1 += __shfl_xor(f1, o, 64);
                f2 += __shfl_xor(f2, o, 64);
                if (RED) w += __shfl_xor(w, o, 64);
            } else {
#pragma unroll
                for (int k = 0; k < MLP_ND; k++) acc[k] += __shfl_xor(acc[k], o, 64);
            }
        }
        if (live && h == 0) {
            if (MODE == 0) {
                float4 *gp = (float4 *) (A.G + (size_t) i * MLP_ND);
#pragma unroll
                for (int k4 = 0; k4 < 4; k4++)
                    gp[k4] = make_float4(acc[4 * k4], acc[4 * k4 + 1], acc[4 * k4 + 2], acc[4 * k4 + 3]);
            } else if (MODE == 2) {
                const float es = A.sc[MLP_ESTD];
                float4 *up = (float4 *) (A.U + (size_t) i * MLP_ND);
#pragma unroll
                for (int k4 = 0; k4 < 4; k4++) {
                    const float *gi = A.sc + MLP_GISTD + 4 * k4;
                    up[k4] = make_float4(es * gi[0] * acc[4 * k4], es * gi[1] * acc[4 * k4 + 1],
                                         es * gi[2] * acc[4 * k4 + 2], es * gi[3] * acc[4 * k4 + 3]);
                }
            } else {
                A.fx[i] = f0; A.fy[i] = f1; A.fz[i] = f2;
                if (RED) { pe += (double) A.E[i]; vir += 0.5 * w; }
                if (!RED && A.vv) {  // k_vv_post's update, on the forces just summed
                    const double m = A.mass[i];
                    double v0 = A.vx[i], v1 = A.vy[i], v2 = A.vz[i];
                    double px = A.X[i], py = A.Y[i], pz = A.Z[i];
                    if (!(A.flags[i] & FLAG_FIXED)) {
                        const double hdt = A.hdt, dt = A.dt;
                        if (A.vv2) {
                            double a0 = hdt * f0, a1 = hdt * f1, a2 = hdt * f2;
                            a0 = a0 / m; a1 = a1 / m; a2 = a2 / m;
                            v0 = v0 + a0; v1 = v1 + a1; v2 = v2 + a2;
                        }
                        if (A.vv1) {
                            double a0 = hdt * f0, a1 = hdt * f1, a2 = hdt * f2;
                            a0 = a0 / m; a1 = a1 / m; a2 = a2 / m;
                            v0 = v0 + a0; v1 = v1 + a1; v2 = v2 + a2;
                            px = px + dt * v0; py = py + dt * v1; pz = pz + dt * v2;
                        }
                        A.vx[i] = v0; A.vy[i] = v1; A.vz[i] = v2;
                    }
                    if (A.vv1) {
                        A.Xn[i] = px; A.Yn[i] = py; A.Zn[i] = pz;
                        const double tw = type_w(A.type[i]);
                        if (A.Pn) A.Pn[i] = make_double4(px, py, pz, tw);
                        if (A.im.on)
                            write_images(A.im, i, A.counters[C_NLOCAL], px, py, pz, A.X, A.Y, A.Z, A.Xn, A.Yn, A.Zn,
                                         A.g, A.Pn, tw);
                    }
                }
            }
        }
    }
    if (MODE == 1 && RED) {
        // one partial per wave (energy, virial rows)
        const double a = wave_sum(pe), b = wave_sum(vir);
        if (lane == 0) {
            A.partials[(size_t) A.pstride + wv] = a;
            A.partials[(size_t) 2 * A.pstride + wv] = b;
        }
    }
}

// lanes per local of the list passes: 4 below 32768 locals (a small system
// fills few waves otherwise), 2 above
static int mlp_lanes(const DevState &d) { return d.nlocal < 32768 ? 4 : 2; }
int mlp_waves(const DevState &d) {
    const int per = 64 / mlp_lanes(d);
    return (d.nlocal + per - 1) / per;
}
template <int MODE, bool RED>
static void launch_mlp_wave(hipStream_t s, const DevState &d, const MLPSegArgs &A) {
    if (mlp_lanes(d) == 4) hipLaunchKernelGGL((k_mlp_wave<MODE, RED, 4>), dim3(mlp_waves(d)), dim3(64), 0, s, A);
    else hipLaunchKernelGGL((k_mlp_wave<MODE, RED, 2>), dim3(mlp_waves(d)), dim3(64), 0, s, A);
}

// dE/dG of every ghost = that of the local at the end of its source chain
__global__ __launch_bounds__(256) void k_mlp_ghost_d(const int *__restrict__ counters, const int *__restrict__ sync_src,
                                                     float *__restrict__ D) {
    const int nlocal = counters[C_NLOCAL], ng = counters[C_NGHOST];
    for (int q = blockIdx.x * 256 + threadIdx.x; q < ng; q += gridDim.x * 256) {
        int root = sync_src[q];
        for (int hop = 0; root >= nlocal && hop < 64; hop++) root = sync_src[root - nlocal];
        if (root >= nlocal) root = nlocal + q;  // unresolved chain: leave the slot as it is
        const float4 *s = (const float4 *) (D + (size_t) root * MLP_ND);
        float4 *d = (float4 *) (D + (size_t) (nlocal + q) * MLP_ND);
#pragma unroll
        for (int k4 = 0; k4 < 4; k4++) d[k4] = s[k4];
    }
}

// ---------------------------------------------------------------- training

__device__ __forceinline__ uint64_t splitmix64(uint64_t x) {
    x += 0x9e3779b97f4a7c15ull;
    x = (x ^ (x >> 30)) * 0xbf58476d1ce4e5b9ull;
    x = (x ^ (x >> 27)) * 0x94d049bb133111ebull;
    return x ^ (x >> 31);
}

// What the gradient kernels accumulate over the tiles of one partial: bias
// gradients and output-weight gradient per lane ([4 c + v][lane]; b1, b2, w3),
// then db3 and the squared error.
constexpr int GACC = 50;

// the sums over the 16 particles of a lane group, written to the partial
__device__ __forceinline__ void mlp_write_bias(const float (&acc)[GACC][64], float *__restrict__ out,
                                               float *__restrict__ loss, int wl, int lane) {
    const int q = lane >> 4, col = lane & 15;
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const int k = 4 * wl + v;
        float a = acc[k][lane], b = acc[16 + k][lane], w = acc[32 + k][lane];
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) {
            a += __shfl_xor(a, o, 64); b += __shfl_xor(b, o, 64); w += __shfl_xor(w, o, 64);
        }
        if (col == 0) {
            const int hh = 16 * wl + 4 * q + v;
            out[MLP_B1 + hh] = a; out[MLP_B2 + hh] = b; out[MLP_W3 + hh] = w;
        }
    }
    if (wl == 0) {
        float gb3 = acc[48][lane], lsum = acc[49][lane];
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) { gb3 += __shfl_xor(gb3, o, 64); lsum += __shfl_xor(lsum, o, 64); }
        if (lane == 0) { out[MLP_B3] = gb3; *loss = lsum; }
    }
}

// the partial's weight gradients: wave wl holds rows 16 wl .. 16 wl + 15
__device__ __forceinline__ void mlp_write_weights(const f32x4 (&gW2)[4], const f32x4 &gW1, float *__restrict__ out,
                                                  int wl, int lane) {
    const int q = lane >> 4, col = lane & 15;
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const int row = 16 * wl + 4 * q + v;
#pragma unroll
        for (int c1 = 0; c1 < 4; c1++) out[MLP_W2 + row * MLP_H + 16 * c1 + col] = gW2[c1][v];
        out[MLP_W1 + row * MLP_ND + col] = gW1[v];
    }
}

// Gradient of L = (1/B) sum_b (y_b - (label_b - e_mean) / e_std)^2 over one
// minibatch into nwaves partials, one workgroup each: partial w sums the
// 16-row tiles w, w + nwaves, ... in that order.  The four waves take four
// consecutive tiles of the partial at once -- forward and backward pass of a
// tile are one long chain of MFMAs and exponentials, which bounds the kernel --
// and hand them over transposed in LDS; then each wave accumulates its quarter
// of the weight gradients (K = 16-particle MFMAs) over the four tiles in order,
// and the waves add their lanes' bias terms in turn, so every sum has the order
// of one wave walking the tiles.  Batch 4096: 22.5 us with one wave per
// partial, 12.9 so.
__global__ __launch_bounds__(256) void k_mlp_grad(const float *__restrict__ p, const float *__restrict__ sc,
                                                  MLPTrain t, uint64_t seed, int step) {
    __shared__ MLPNet N;
    __shared__ short s_tile[4][3 * MLP_H * 16 + MLP_ND * 16];
    __shared__ float s_acc[GACC][64];
    const int lane = threadIdx.x & 63, q = lane >> 4, col = lane & 15, wl = threadIdx.x >> 6;
    const int part = blockIdx.x, np = gridDim.x;
    for (int k = threadIdx.x; k < GACC * 64; k += 256) (&s_acc[0][0])[k] = 0.f;
    const int mine = ((t.batch >> 4) - part + np - 1) / np;  // tiles of this partial
    float4 g = make_float4(0.f, 0.f, 0.f, 0.f);
    float lab = 0.f;
    const auto load = [&](int k) __attribute__((always_inline)) {  // row col of the partial's tile k
        if (k >= mine) return;
        const uint64_t j = (uint64_t) ((part + k * np) * 16 + col);
        const uint64_t h = splitmix64(seed ^ ((uint64_t) step << 32) ^ j);
        const int idx = (int) (h % (uint64_t) t.rows);
        g = *(const float4 *) (t.G + (size_t) idx * MLP_ND + 4 * q);
        lab = t.label[idx];
    };
    load(wl);
    mlp_stage<true, 256>(N, p, sc);
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 gW2[4] = {zero, zero, zero, zero}, gW1 = zero;
    const float inv_es = 1.0f / N.es, scale = 2.0f / (float) t.batch;
    for (int t0 = 0; t0 < mine; t0 += 4) {
        mlp_keep_in_lds();
        const MLPView R{N, lane, q};
        const int nt = min(4, mine - t0);
        float a1[4][4], a2[4][4], h3[4][4], e = 0.f, err = 0.f;
        if (wl < nt) {
            short *sD2 = s_tile[wl], *sH1 = sD2 + MLP_H * 16, *sD1 = sH1 + MLP_H * 16, *sG = sD1 + MLP_H * 16;
            bf16x4 b0, b0l;
            split4(mlp_input(R, g), b0, b0l);
#pragma unroll
            for (int v = 0; v < 4; v++) sG[(4 * q + v) * 16 + col] = b0[v];
            f32x4 h1[4], dh1[4], h2[4], dh2[4];
            bf16x4 bh1[4];
            const float y = mlp_forward(R, b0, b0l, h1, dh1, bh1, h2, dh2);
#pragma unroll
            for (int c = 0; c < 4; c++)
#pragma unroll
                for (int v = 0; v < 4; v++) sH1[(16 * c + 4 * q + v) * 16 + col] = bh1[c][v];
            err = y - (lab - N.em) * inv_es;
            load(t0 + 4 + wl);
            e = scale * err;
            bf16x4 bd2[4];
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const f32x4 w3 = R.w3(c);
                f32x4 d2;
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    h3[c][v] = h2[c][v];
                    d2[v] = e * w3[v] * dh2[c][v];
                    a2[c][v] = d2[v];
                }
                bd2[c] = pack4(d2);
#pragma unroll
                for (int v = 0; v < 4; v++) sD2[(16 * c + 4 * q + v) * 16 + col] = bd2[c][v];
            }
#pragma unroll
            for (int c = 0; c < 4; c++) {
                f32x4 a = zero;
#pragma unroll
                for (int kc = 0; kc < 4; kc++) a = mfma16(R.f(NF_A2T + 4 * c + kc), bd2[kc], a);
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const float d1 = a[v] * dh1[c][v];
                    a1[c][v] = d1;
                    sD1[(16 * c + 4 * q + v) * 16 + col] = f2bf(d1);
                }
            }
        }
        for (int u = 0; u < nt; u++) {
            if (u == wl) {
#pragma unroll
                for (int c = 0; c < 4; c++)
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        const int k = 4 * c + v;
                        s_acc[k][lane] += a1[c][v];
                        s_acc[16 + k][lane] += a2[c][v];
                        s_acc[32 + k][lane] = fmaf(e, h3[c][v], s_acc[32 + k][lane]);
                    }
                if (q == 0) {
                    s_acc[48][lane] += e;
                    s_acc[49][lane] = fmaf(err, err, s_acc[49][lane]);
                }
            }
            __syncthreads();
        }
        for (int u = 0; u < nt; u++) {
            const short *sD2 = s_tile[u], *sH1 = sD2 + MLP_H * 16, *sD1 = sH1 + MLP_H * 16, *sG = sD1 + MLP_H * 16;
            const bf16x4 a = *(const bf16x4 *) (sD2 + (16 * wl + col) * 16 + 4 * q);
#pragma unroll
            for (int c1 = 0; c1 < 4; c1++)
                gW2[c1] = mfma16(a, *(const bf16x4 *) (sH1 + (16 * c1 + col) * 16 + 4 * q), gW2[c1]);
            gW1 = mfma16(*(const bf16x4 *) (sD1 + (16 * wl + col) * 16 + 4 * q),
                         *(const bf16x4 *) (sG + col * 16 + 4 * q), gW1);
        }
        __syncthreads();
    }
    float *out = t.partial + (size_t) part * MLP_NP;
    mlp_write_weights(gW2, gW1, out, wl, lane);
    mlp_write_bias(s_acc, out, t.loss + part, wl, lane);
}

// SiLU with its first and second derivatives:
// h = z s, h' = s (1 + z (1 - s)), h'' = s (1 - s) (2 + z (1 - 2 s)), s = sigmoid(z)
__device__ __forceinline__ void silu3(float z, float &h, float &dh, float &ddh) {
    const float sg = __builtin_amdgcn_rcpf(1.0f + __expf(-z));
    h = z * sg;
    dh = sg * fmaf(z, 1.0f - sg, 1.0f);
    ddh = sg * (1.0f - sg) * fmaf(z, 1.0f - 2.0f * sg, 2.0f);
}

// Gradient over the parameters of one configuration's loss (rows [0, n), one
// per local): sum_a [eps_a y_a + (dy_a/ds) . u_a], eps_a = eps_scale *
// (y_a - (E*_a - e_mean) / e_std) and u_a = U row a held fixed.  Per
// 16-particle tile: the forward pass (h1, h2 and both SiLU derivatives), the
// tangent along u (dz1 = W1 u, dh1 = h1' dz1, dz2 = W2 dh1), then reverse mode
// through both:
//   bar dz2 = w3 h2',  bar z2 = w3 (eps h2' + h2'' dz2),
//   bar dz1 = (W2^T bar dz2) h1',  bar z1 = (W2^T bar z2) h1' + (W2^T bar dz2) h1'' dz1,
//   dW2 = bar z2 h1^T + bar dz2 dh1^T,  dW1 = bar z1 s^T + bar dz1 u^T,
//   db1 = bar z1, db2 = bar z2, dw3 = eps h2 + h2' dz2, db3 = eps.
// Layer products and weight gradients are MFMAs in the layout of k_mlp_grad
// (BF16 operands, FP32 accumulation; s and u enter the first layer as hi + lo
// pairs), and the tiles of a partial are shared among the waves of its
// workgroup as there (2048 rows: 18 -> 12.2 us).  Tiles past the end have eps =
// u = 0 and add exact zeros.
__global__ __launch_bounds__(256) void k_mlp_cgrad(const float *__restrict__ p, const float *__restrict__ sc,
                                                   MLPCfgGrad t) {
    __shared__ MLPNet N;
    __shared__ short s_tile[4][6 * MLP_H * 16 + 2 * MLP_ND * 16];
    __shared__ float s_acc[GACC][64];
    const int lane = threadIdx.x & 63, q = lane >> 4, col = lane & 15, wl = threadIdx.x >> 6;
    const int part = blockIdx.x, np = gridDim.x;
    for (int k = threadIdx.x; k < GACC * 64; k += 256) (&s_acc[0][0])[k] = 0.f;
    const int ntiles = (t.n + 15) >> 4;
    const int iters = (ntiles + np - 1) / np;
    float4 g, uu;
    double lab;
    bool ok;
    const auto load = [&](int k) __attribute__((always_inline)) {  // row col of the partial's tile k
        const int row = (part + k * np) * 16 + col;
        ok = k < iters && row < t.n;
        g = uu = make_float4(0.f, 0.f, 0.f, 0.f);
        lab = 0.0;
        if (!ok) return;
        g = *(const float4 *) (t.G + (size_t) row * MLP_ND + 4 * q);
        uu = *(const float4 *) (t.U + (size_t) row * MLP_ND + 4 * q);
        lab = t.label[row];
    };
    load(wl);
    mlp_stage<true, 256>(N, p, sc);
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 gW2[4] = {zero, zero, zero, zero}, gW1 = zero;
    const float inv_es = 1.0f / N.es;
    for (int t0 = 0; t0 < iters; t0 += 4) {
        mlp_keep_in_lds();
        const MLPView R{N, lane, q};
        const int nt = min(4, iters - t0);
        float a1[4][4], a2[4][4], h3[4][4], d3[4][4], x3[4][4], e = 0.f, err = 0.f;
        if (wl < nt) {
            short *sZ2 = s_tile[wl], *sH1 = sZ2 + MLP_H * 16, *sT2 = sH1 + MLP_H * 16, *sTH1 = sT2 + MLP_H * 16;
            short *sZ1 = sTH1 + MLP_H * 16, *sT1 = sZ1 + MLP_H * 16, *sS = sT1 + MLP_H * 16, *sU = sS + MLP_ND * 16;
            bf16x4 b0, b0l, u0, u0l;
            split4(mlp_input(R, g), b0, b0l);
            split4(uu.x, uu.y, uu.z, uu.w, u0, u0l);
#pragma unroll
            for (int v = 0; v < 4; v++) {
                sS[(4 * q + v) * 16 + col] = b0[v];
                sU[(4 * q + v) * 16 + col] = u0[v];
            }
            // forward, keeping h, h' and h'' of both layers
            f32x4 h1[4], d1[4], e1[4], h2[4], d2[4], e2[4];
            bf16x4 bh1[4];
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const f32x4 z = mlp_layer1(R, c, b0, b0l), b1 = R.b1(c);
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    float h, dh, ddh;
                    silu3(z[v] + b1[v], h, dh, ddh);
                    h1[c][v] = h; d1[c][v] = dh; e1[c][v] = ddh;
                }
                bh1[c] = pack4(h1[c]);
            }
#pragma unroll
            for (int c = 0; c < 4; c++) {
                f32x4 z = zero;
                const f32x4 b2 = R.b2(c);
#pragma unroll
                for (int kc = 0; kc < 4; kc++) z = mfma16(R.f(NF_A2 + 4 * c + kc), bh1[kc], z);
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    float h, dh, ddh;
                    silu3(z[v] + b2[v], h, dh, ddh);
                    h2[c][v] = h; d2[c][v] = dh; e2[c][v] = ddh;
                }
            }
            float y = 0.f;
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const f32x4 w3 = R.w3(c);
#pragma unroll
                for (int v = 0; v < 4; v++) y = fmaf(w3[v], h2[c][v], y);
            }
            y += __shfl_xor(y, 16, 64);
            y += __shfl_xor(y, 32, 64);
            y += N.b3;
            err = ok ? y - ((float) lab - N.em) * inv_es : 0.0f;
            load(t0 + 4 + wl);
            e = t.eps_scale * err;
            // tangent along u
            f32x4 t1[4];
            bf16x4 bth1[4];
#pragma unroll
            for (int c = 0; c < 4; c++) {
                t1[c] = mlp_layer1(R, c, u0, u0l);
                bth1[c] = pack4(d1[c][0] * t1[c][0], d1[c][1] * t1[c][1], d1[c][2] * t1[c][2], d1[c][3] * t1[c][3]);
            }
            bf16x4 bz2[4], bt2[4];
#pragma unroll
            for (int c = 0; c < 4; c++) {
                f32x4 t2 = zero;
                const f32x4 w3 = R.w3(c);
#pragma unroll
                for (int kc = 0; kc < 4; kc++) t2 = mfma16(R.f(NF_A2 + 4 * c + kc), bth1[kc], t2);
                f32x4 z2b, t2b;
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const float w = w3[v];
                    h3[c][v] = h2[c][v];
                    d3[c][v] = d2[c][v];
                    x3[c][v] = t2[v];
                    t2b[v] = w * d2[c][v];
                    z2b[v] = w * fmaf(e, d2[c][v], e2[c][v] * t2[v]);
                    a2[c][v] = z2b[v];
                }
                bz2[c] = pack4(z2b);
                bt2[c] = pack4(t2b);
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int f = (16 * c + 4 * q + v) * 16 + col;
                    sZ2[f] = bz2[c][v];
                    sT2[f] = bt2[c][v];
                    sH1[f] = bh1[c][v];
                    sTH1[f] = bth1[c][v];
                }
            }
#pragma unroll
            for (int c = 0; c < 4; c++) {
                f32x4 a = zero, at = zero;
#pragma unroll
                for (int kc = 0; kc < 4; kc++) {
                    const bf16x4 w = R.f(NF_A2T + 4 * c + kc);
                    a = mfma16(w, bz2[kc], a);
                    at = mfma16(w, bt2[kc], at);
                }
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const float z1b = fmaf(at[v] * e1[c][v], t1[c][v], a[v] * d1[c][v]);
                    a1[c][v] = z1b;
                    const int f = (16 * c + 4 * q + v) * 16 + col;
                    sZ1[f] = f2bf(z1b);
                    sT1[f] = f2bf(at[v] * d1[c][v]);
                }
            }
        }
        // the waves in turn; dw3 = eps h2 + h2' dz2
        for (int u = 0; u < nt; u++) {
            if (u == wl) {
#pragma unroll
                for (int c = 0; c < 4; c++)
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        const int k = 4 * c + v;
                        s_acc[k][lane] += a1[c][v];
                        s_acc[16 + k][lane] += a2[c][v];
                        s_acc[32 + k][lane] = fmaf(e, h3[c][v], fmaf(d3[c][v], x3[c][v], s_acc[32 + k][lane]));
                    }
                if (q == 0) {
                    s_acc[48][lane] += e;
                    s_acc[49][lane] = fmaf(err, err, s_acc[49][lane]);
                }
            }
            __syncthreads();
        }
        for (int u = 0; u < nt; u++) {
            const short *sZ2 = s_tile[u], *sH1 = sZ2 + MLP_H * 16, *sT2 = sH1 + MLP_H * 16, *sTH1 = sT2 + MLP_H * 16;
            const short *sZ1 = sTH1 + MLP_H * 16, *sT1 = sZ1 + MLP_H * 16, *sS = sT1 + MLP_H * 16, *sU = sS + MLP_ND * 16;
            const int at_row = (16 * wl + col) * 16 + 4 * q;
            const bf16x4 az = *(const bf16x4 *) (sZ2 + at_row), at = *(const bf16x4 *) (sT2 + at_row);
#pragma unroll
            for (int c1 = 0; c1 < 4; c1++) {
                const int b = (16 * c1 + col) * 16 + 4 * q;
                gW2[c1] = mfma16(az, *(const bf16x4 *) (sH1 + b), gW2[c1]);
                gW2[c1] = mfma16(at, *(const bf16x4 *) (sTH1 + b), gW2[c1]);
            }
            gW1 = mfma16(*(const bf16x4 *) (sZ1 + at_row), *(const bf16x4 *) (sS + col * 16 + 4 * q), gW1);
            gW1 = mfma16(*(const bf16x4 *) (sT1 + at_row), *(const bf16x4 *) (sU + col * 16 + 4 * q), gW1);
        }
        __syncthreads();
    }
    float *out = t.partial + (size_t) part * MLP_NP;
    mlp_write_weights(gW2, gW1, out, wl, lane);
    mlp_write_bias(s_acc, out, t.loss + part, wl, lane);
}

// rho_i = 2 w_force (F_i - F*_i) / sum_j |F*_j|^2 for the locals; the sum is
// taken from k_force_diff's per-block partials (rows 2b + 1)
__global__ __launch_bounds__(256) void k_mlp_rho(const int *__restrict__ counters, const double *__restrict__ fx,
                                                 const double *__restrict__ fy, const double *__restrict__ fz,
                                                 const double *__restrict__ lx, const double *__restrict__ ly,
                                                 const double *__restrict__ lz, const double *__restrict__ partials,
                                                 int nb, double w_force, float4 *__restrict__ rho) {
    __shared__ double s_scale;
    if (threadIdx.x == 0) {
        double den = 0.0;
        for (int b = 0; b < nb; b++) den += partials[2 * b + 1];
        s_scale = den > 0.0 ? 2.0 * w_force / den : 0.0;
    }
    __syncthreads();
    const double sc = s_scale;
    const int n = counters[C_NLOCAL];
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256)
        rho[i] = make_float4((float) (sc * (fx[i] - lx[i])), (float) (sc * (fy[i] - ly[i])),
                             (float) (sc * (fz[i] - lz[i])), 0.0f);
}

// rho of every ghost = that of the local at the end of its source chain
__global__ __launch_bounds__(256) void k_mlp_ghost_rho(const int *__restrict__ counters,
                                                       const int *__restrict__ sync_src, float4 *__restrict__ rho) {
    const int nlocal = counters[C_NLOCAL], ng = counters[C_NGHOST];
    for (int q = blockIdx.x * 256 + threadIdx.x; q < ng; q += gridDim.x * 256) {
        int root = sync_src[q];
        for (int hop = 0; root >= nlocal && hop < 64; hop++) root = sync_src[root - nlocal];
        rho[nlocal + q] = root < nlocal ? rho[root] : make_float4(0.f, 0.f, 0.f, 0.f);
    }
}

// parameter k of the gradient: the partials added in order.  Thirty-two
// loads are in flight before the first is added (64 partials: 16.6 us with one
// load a turn, 4.3 so).
__device__ __forceinline__ float sum_partials(const float *__restrict__ partial, int n, int k) {
    float s = 0.f;
    int w = 0;
    for (; w + 32 <= n; w += 32) {
        float v[32];
#pragma unroll
        for (int u = 0; u < 32; u++) v[u] = partial[(size_t) (w + u) * MLP_NP + k];
#pragma unroll
        for (int u = 0; u < 32; u++) s += v[u];
    }
    for (; w < n; w++) s += partial[(size_t) w * MLP_NP + k];
    return s;
}

// acc += sum over waves of the gradient partials (in wave order); with out,
// the sum itself is also written there
__global__ __launch_bounds__(64) void k_mlp_accum(const float *__restrict__ partial, int nwaves,
                                                   float *__restrict__ acc, float *__restrict__ out) {
    const int k = blockIdx.x * 64 + threadIdx.x;
    if (k >= MLP_NP) return;
    const float s = sum_partials(partial, nwaves, k);
    if (acc) acc[k] += s;
    if (out) out[k] = s;
}

// Adam (beta1 0.9, beta2 0.999, eps 1e-8) on the summed wave partials
__global__ __launch_bounds__(64) void k_mlp_adam(float *__restrict__ p, float *__restrict__ m, float *__restrict__ v,
                                                  const float *__restrict__ partial, const float *__restrict__ loss,
                                                  int nwaves, int batch, float lr, float bc1, float bc2,
                                                  float gscale, float *__restrict__ loss_out) {
    const int k = blockIdx.x * 64 + threadIdx.x;
    if (k < MLP_NP) {
        float gsum = sum_partials(partial, nwaves, k);
        gsum *= gscale;
        const float mm = 0.9f * m[k] + 0.1f * gsum;
        const float vv = 0.999f * v[k] + 0.001f * gsum * gsum;
        m[k] = mm;
        v[k] = vv;
        p[k] -= lr * (mm / bc1) / (sqrtf(vv / bc2) + 1e-8f);
    }
    if (k == 0 && loss_out) {
        float s = 0.f;
#pragma unroll 16
        for (int w = 0; w < nwaves; w++) s += loss[w];
        *loss_out = s / (float) batch;
    }
}

// column moments: per block, 16 descriptor sums, 16 sums of squares, label sum and sum of squares
__global__ __launch_bounds__(256) void k_mlp_moments(const float *__restrict__ G, const float *__restrict__ label,
                                                     int n, double *__restrict__ partials) {
    __shared__ double red[16][34];
    const int col = threadIdx.x & 15, sub = threadIdx.x >> 4;
    double s = 0.0, s2 = 0.0, l = 0.0, l2 = 0.0;
    for (int r = blockIdx.x * 16 + sub; r < n; r += gridDim.x * 16) {
        const double x = G[(size_t) r * MLP_ND + col];
        s += x; s2 += x * x;
        if (col == 0) { const double y = label[r]; l += y; l2 += y * y; }
    }
    red[sub][col] = s;
    red[sub][16 + col] = s2;
    if (col == 0) { red[sub][32] = l; red[sub][33] = l2; }
    __syncthreads();
    if (threadIdx.x < 34) {
        double a = 0.0;
        for (int k = 0; k < 16; k++) a += red[k][threadIdx.x];
        partials[(size_t) blockIdx.x * 34 + threadIdx.x] = a;
    }
}

__global__ __launch_bounds__(256) void k_mlp_sqerr(const float *__restrict__ E, const float *__restrict__ label, int n,
                                                   double *__restrict__ partials) {
    double s = 0.0;
    for (int r = blockIdx.x * 256 + threadIdx.x; r < n; r += gridDim.x * 256) {
        const double d = (double) E[r] - (double) label[r];
        s += d * d;
    }
    __shared__ double red[4];
    const double a = wave_sum(s);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = a;
    __syncthreads();
    if (threadIdx.x == 0) partials[blockIdx.x] = ((red[0] + red[1]) + red[2]) + red[3];
}

__global__ __launch_bounds__(256) void k_mlp_snapshot(const float *__restrict__ G, const double *__restrict__ eatom,
                                                      int nlocal, float *__restrict__ dG, float *__restrict__ dl) {
    for (int i = blockIdx.x * 256 + threadIdx.x; i < nlocal; i += gridDim.x * 256) {
        const float4 *s = (const float4 *) (G + (size_t) i * MLP_ND);
        float4 *d = (float4 *) (dG + (size_t) i * MLP_ND);
#pragma unroll
        for (int k4 = 0; k4 < 4; k4++) d[k4] = s[k4];
        dl[i] = (float) eatom[i];
    }
}

__global__ __launch_bounds__(256) void k_force_diff(const double *__restrict__ ax, const double *__restrict__ ay,
                                                    const double *__restrict__ az, const double *__restrict__ bx,
                                                    const double *__restrict__ by, const double *__restrict__ bz,
                                                    int n, double *__restrict__ partials) {
    double s = 0.0, r = 0.0;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
        const double d0 = ax[i] - bx[i], d1 = ay[i] - by[i], d2 = az[i] - bz[i];
        s += d0 * d0 + d1 * d1 + d2 * d2;
        r += bx[i] * bx[i] + by[i] * by[i] + bz[i] * bz[i];
    }
    __shared__ double red[2][4];
    const double a = wave_sum(s), b = wave_sum(r);
    if ((threadIdx.x & 63) == 0) { red[0][threadIdx.x >> 6] = a; red[1][threadIdx.x >> 6] = b; }
    __syncthreads();
    if (threadIdx.x < 2) {
        const int k = threadIdx.x;
        partials[2 * blockIdx.x + k] = ((red[k][0] + red[k][1]) + red[k][2]) + red[k][3];
    }
}

// ---------------------------------------------------------------- launchers

static MLPSegArgs seg_args(const DevState &d, int cur) {
    MLPSegArgs A{};
    A.counters = d.counters;
    A.X = d.X[cur]; A.Y = d.Y[cur]; A.Z = d.Z[cur];
    A.P = d.P[cur];
    A.nl = d.nl;
    A.nl_stride = d.nl_stride;
    A.numneighs = d.numneighs;
    A.ncap = d.ncap;
    A.pstride = d.pstride;
    return A;
}

void launch_mlp_descriptors(hipStream_t s, const DevState &d, const Geom &g, int cur, float *G, bool pack) {
    if (d.nlocal <= 0) return;
    (void) g;
    if (pack) launch_pack_p(s, d, cur);  // both passes gather packed positions
    MLPSegArgs A = seg_args(d, cur);
    A.G = G;
    launch_mlp_wave<0, false>(s, d, A);
}

// k_mlp_eval by rows: workgroups of 16 waves convert the weights once per CU and
// let four tiles share each SIMD, in at most 256 workgroups (one per CU); few
// rows spread better over workgroups of 4.  Measured, 4 waves | 16: 2048 rows
// 9.6 | 11.1 us; a step at 8400 rows 98.6 | 96.9, at 35152 100.2 | 97.8, at
// 131072 167.5 | 164.1 (the pass itself 23 | 18 us).
template <bool WANT_D, bool IMG, int NT>
static void eval_launch(hipStream_t s, const float *p, const float *sc, const float *G, int n, float *E, float *D,
                        const Images &im) {
    const int ntiles = (n + 15) / 16, per = NT / 64;
    const int grid = std::min((ntiles + per - 1) / per, 256);
    hipLaunchKernelGGL((k_mlp_eval<WANT_D, IMG, NT>), dim3(grid), dim3(NT), 0, s, p, sc, G, n, E, D, im);
}

template <bool WANT_D, bool IMG>
static void eval_any(hipStream_t s, const float *p, const float *sc, const float *G, int n, float *E, float *D,
                     const Images &im) {
    if (n < 8192) eval_launch<WANT_D, IMG, 256>(s, p, sc, G, n, E, D, im);
    else eval_launch<WANT_D, IMG, 1024>(s, p, sc, G, n, E, D, im);
}

void launch_mlp_eval(hipStream_t s, const float *p, const float *sc, const float *G, int n, float *E, float *D) {
    if (n <= 0) return;
    const Images none{};
    if (D) eval_any<true, false>(s, p, sc, G, n, E, D, none);
    else eval_any<false, false>(s, p, sc, G, n, E, D, none);
}

void launch_mlp_forces(hipStream_t s, const DevState &d, const Geom &g, const MLPBind &b, int cur, int reduce,
                       int ghost_grid, const MLPVV *vv, bool pack) {
    if (d.nlocal <= 0) return;
    launch_mlp_descriptors(s, d, g, cur, b.G, pack);
    const Images im = images_of(d, true);
    eval_any<true, true>(s, b.p, b.sc, b.G, d.nlocal, b.E, b.D, im);
    if (!im.on)
        hipLaunchKernelGGL(k_mlp_ghost_d, dim3(std::max(ghost_grid, 1)), dim3(256), 0, s, d.counters, d.sync_src, b.D);
    MLPSegArgs A = seg_args(d, cur);
    A.D = b.D;
    A.E = b.E;
    A.fx = d.fx; A.fy = d.fy; A.fz = d.fz;
    A.partials = d.partials;
    if (vv && !reduce) {
        A.vv = 1;
        A.vv2 = vv->vv2; A.vv1 = vv->vv1;
        A.dt = vv->prm->dt; A.hdt = vv->prm->hdt;
        A.flags = d.flags; A.type = d.type; A.mass = d.mass;
        A.vx = d.vx; A.vy = d.vy; A.vz = d.vz;
        A.Xn = d.X[vv->next]; A.Yn = d.Y[vv->next]; A.Zn = d.Z[vv->next];
        A.im = images_of(d, vv->vv1 && vv->next != cur);
        A.g = g;
        A.Pn = vv->Pn;
    }
    if (reduce) launch_mlp_wave<1, true>(s, d, A);
    else launch_mlp_wave<1, false>(s, d, A);
}

void launch_mlp_grad(hipStream_t s, const float *p, const float *sc, const MLPTrain &t, uint64_t seed, int step) {
    hipLaunchKernelGGL(k_mlp_grad, dim3(t.nwaves), dim3(256), 0, s, p, sc, t, seed, step);
}

void launch_mlp_adam(hipStream_t s, float *p, float *m, float *v, const MLPTrain &t, float lr, int step,
                     float *loss_out) {
    const float bc1 = 1.0f - powf(0.9f, (float) step), bc2 = 1.0f - powf(0.999f, (float) step);
    hipLaunchKernelGGL(k_mlp_adam, dim3((MLP_NP + 63) / 64), dim3(64), 0, s, p, m, v, t.partial, t.loss,
                       t.nwaves, t.batch, lr, bc1, bc2, t.gscale, loss_out);
}

void launch_mlp_config_grad(hipStream_t s, const DevState &d, const Geom &g, const MLPBind &b, int cur,
                            const double *lx, const double *ly, const double *lz, const double *eatom,
                            double w_energy, double w_force, float4 *rho, float *U, double *red, int nb,
                            int ghost_grid, const MLPCfgGrad &t) {
    const int n = d.nlocal;
    if (n <= 0) return;
    // the network's forces (descriptors, E, dE/dG of locals and ghosts) into d.f*
    launch_mlp_forces(s, d, g, b, cur, 0, ghost_grid);
    launch_force_diff(s, d.fx, d.fy, d.fz, lx, ly, lz, n, red, nb);
    hipLaunchKernelGGL(k_mlp_rho, dim3(std::min((n + 255) / 256, 1024)), dim3(256), 0, s, d.counters, d.fx, d.fy,
                       d.fz, lx, ly, lz, red, nb, w_force, rho);
    hipLaunchKernelGGL(k_mlp_ghost_rho, dim3(std::max(ghost_grid, 1)), dim3(256), 0, s, d.counters, d.sync_src,
                       rho);
    MLPSegArgs A = seg_args(d, cur);
    A.rho = rho;
    A.sc = b.sc;
    A.U = U;
    launch_mlp_wave<2, false>(s, d, A);
    MLPCfgGrad tt = t;
    tt.G = b.G;
    tt.label = eatom;
    tt.U = U;
    tt.n = n;
    tt.eps_scale = (float) (2.0 * w_energy / n);
    hipLaunchKernelGGL(k_mlp_cgrad, dim3(tt.nwaves), dim3(256), 0, s, b.p, b.sc, tt);
}

void launch_mlp_accum(hipStream_t s, const float *partial, int nwaves, float *acc, float *out) {
    hipLaunchKernelGGL(k_mlp_accum, dim3((MLP_NP + 63) / 64), dim3(64), 0, s, partial, nwaves, acc, out);
}

void launch_mlp_moments(hipStream_t s, const float *G, const float *label, int n, double *partials, int nblocks) {
    hipLaunchKernelGGL(k_mlp_moments, dim3(nblocks), dim3(256), 0, s, G, label, n, partials);
}

void launch_mlp_sqerr(hipStream_t s, const float *E, const float *label, int n, double *partials, int nblocks) {
    hipLaunchKernelGGL(k_mlp_sqerr, dim3(nblocks), dim3(256), 0, s, E, label, n, partials);
}

void launch_mlp_snapshot(hipStream_t s, const float *G, const double *eatom, int nlocal, float *dst_G,
                         float *dst_label) {
    if (nlocal <= 0) return;
    hipLaunchKernelGGL(k_mlp_snapshot, dim3(std::min((nlocal + 255) / 256, 2048)), dim3(256), 0, s, G, eatom, nlocal,
                       dst_G, dst_label);
}

void launch_force_diff(hipStream_t s, const double *ax, const double *ay, const double *az, const double *bx,
                       const double *by, const double *bz, int n, double *partials, int nblocks) {
    hipLaunchKernelGGL(k_force_diff, dim3(nblocks), dim3(256), 0, s, ax, ay, az, bx, by, bz, n, partials);
}

}  // namespace pk
