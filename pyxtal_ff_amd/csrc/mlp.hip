// Per-element network energies and their gradients with respect to the
// descriptors, for energy + force evaluation (no parameter gradients).
// Mirrors the reference's per-element feed-forward networks
// (pyxtal_ff/models/neuralnetwork.py:80-200: nn.Linear layers with one
// activation each, descriptors scaled by the element's drange,
// neuralnetwork.py:938-1029) evaluated forward, then backward to dE/dx.
// By what fits in LDS: 16-atom tiles on the FP64 matrix cores (mlp_mfma_kernel
// and mlp_mfma4_kernel, scratch and one element's weights within 160 KB);
// else one wavefront per atom with lane n holding neuron n of a layer
// (widths <= 64), the weights of every element in LDS (mlp_lds_kernel) or
// streamed from L2 (mlp_energy_grad_kernel).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <mutex>

#include "pxff_common.h"
#include "so4_dev.h"

namespace pxff {

constexpr int MLP_MAXW = 64;     // hidden / output width limit (one lane per neuron)
constexpr int MLP_MAXL = 8;      // layers per element
constexpr int MLP_MAXIN = 1024;  // descriptor length limit
constexpr int MLP_LSTRIDE = 6;   // ints per layer in the layout
constexpr int MLP_STRIDE = 1 + MLP_LSTRIDE * MLP_MAXL;

__device__ inline void act_fdf(int id, double z, double &a, double &da) {
    switch (id) {
    case 1: {  // Tanh
        const double t = tanh(z);
        a = t;
        da = 1.0 - t * t;
        break;
    }
    case 2: {  // Sigmoid
        const double s = 1.0 / (1.0 + exp(-z));
        a = s;
        da = s * (1.0 - s);
        break;
    }
    case 3:  // ReLU
        // (a NaN stays one, as in torch)
        a = z <= 0.0 ? 0.0 : z;
        da = z <= 0.0 ? 0.0 : 1.0;
        break;
    case 4: {  // Softplus (beta 1, threshold 20, as torch.nn.Softplus)
        if (z > 20.0) {
            a = z;
            da = 1.0;
        } else {
            a = log1p(exp(z));
            da = 1.0 / (1.0 + exp(-z));
        }
        break;
    }
    case 5:  // ELU (alpha 1)
        if (z > 0.0) {
            a = z;
            da = 1.0;
        } else {
            a = expm1(z);
            da = a + 1.0;
        }
        break;
    default:  // Linear
        a = z;
        da = 1.0;
    }
}

// layout per element e (ints, at d_layout[e * MLP_STRIDE]):
//   nlayers, then per layer {nin, nout, act, w_off, b_off, wt_off}: W
//   row-major [nout][nin] as torch.nn.Linear stores it (read by the
//   backward: lanes over inputs, consecutive addresses) and its transpose
//   [nin][nout] (read by the forward: lanes over outputs), offsets into
//   the parameter array.

// Workgroup-wide barrier (one wavefront per workgroup).
struct WgSync {
    __device__ void operator()() const { __syncthreads(); }
};
// The wavefront's own LDS writes are visible to its later reads (LDS
// operations of one wavefront execute in order; the fences keep the
// compiler from moving them).
struct WaveSync {
    __device__ void operator()() const {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
};

// One atom on one wavefront: lane n holds neuron n of a layer; h0 [nin],
// dact / hout [layers][hw] (hw = the widest layer) are the wavefront's LDS scratch.
template <typename Sync>
__device__ inline void mlp_atom(int64_t i, int lane, int nin, int nelem, const int64_t *__restrict__ species,
                                const int *__restrict__ layout, const double *params, const double *__restrict__ dmin,
                                const double *__restrict__ scale, const double *__restrict__ x,
                                double *__restrict__ e_out, double *__restrict__ beta, double *h0, double *dact,
                                double *hout, int hw, Sync sync) {
    const int64_t el64 = species[i];
    if (el64 < 0 || el64 >= nelem) {  // no network for this atom: NaN results
        if (lane == 0) e_out[i] = __builtin_nan("");
        for (int j = lane; j < nin; j += 64) beta[(size_t)i * nin + j] = __builtin_nan("");
        return;  // whole wavefront
    }
    const int el = (int)el64;
    const int *lay = layout + el * MLP_STRIDE;
    const int nl = lay[0];
    const double *xi = x + (size_t)i * nin;
    const double *dm = dmin + (size_t)el * nin, *sc = scale + (size_t)el * nin;
    for (int j = lane; j < nin; j += 64) h0[j] = (xi[j] - dm[j]) * sc[j];
    sync();
    // forward
    const double *hin = h0;
    for (int k = 0; k < nl; k++) {
        const int *L = lay + 1 + MLP_LSTRIDE * k;
        const int ni = L[0], no = L[1], act = L[2];
        const double *WT = params + L[5], *b = params + L[4];
        if (lane < no) {
            // four partial sums: four independent FMA chains
            double z0 = b[lane], z1 = 0.0, z2 = 0.0, z3 = 0.0;
            int j = 0;
            for (; j + 4 <= ni; j += 4) {
                z0 += WT[(size_t)j * no + lane] * hin[j];
                z1 += WT[(size_t)(j + 1) * no + lane] * hin[j + 1];
                z2 += WT[(size_t)(j + 2) * no + lane] * hin[j + 2];
                z3 += WT[(size_t)(j + 3) * no + lane] * hin[j + 3];
            }
            for (; j < ni; j++) z0 += WT[(size_t)j * no + lane] * hin[j];
            const double z = (z0 + z1) + (z2 + z3);
            double a, da;
            act_fdf(act, z, a, da);
            hout[k * hw + lane] = a;
            dact[k * hw + lane] = da;
        }
        sync();
        hin = hout + k * hw;
    }
    if (lane == 0) e_out[i] = hin[0];
    // backward: dact[k] becomes the pre-activation gradient of layer k; for
    // the output layer (one neuron, dE/dE = 1) it already is act'
    for (int k = nl - 1; k >= 1; k--) {
        const int *L = lay + 1 + MLP_LSTRIDE * k;
        const int ni = L[0], no = L[1];
        const double *W = params + L[3];
        // dE/dh_{k-1}[j] = sum_n W[n][j] g_pre[n]; then times act'_{k-1}
        if (lane < ni) {
            const double *gk = dact + k * hw;
            double g0 = 0.0, g1 = 0.0, g2 = 0.0, g3 = 0.0;
            int n = 0;
            for (; n + 4 <= no; n += 4) {
                g0 += W[(size_t)n * ni + lane] * gk[n];
                g1 += W[(size_t)(n + 1) * ni + lane] * gk[n + 1];
                g2 += W[(size_t)(n + 2) * ni + lane] * gk[n + 2];
                g3 += W[(size_t)(n + 3) * ni + lane] * gk[n + 3];
            }
            for (; n < no; n++) g0 += W[(size_t)n * ni + lane] * gk[n];
            dact[(k - 1) * hw + lane] *= (g0 + g1) + (g2 + g3);
        }
        sync();
    }
    {
        const int *L = lay + 1;
        const int ni = L[0], no = L[1];
        const double *W = params + L[3];
        for (int j = lane; j < ni; j += 64) {
            double g0 = 0.0, g1 = 0.0, g2 = 0.0, g3 = 0.0;
            int n = 0;
            for (; n + 4 <= no; n += 4) {
                g0 += W[(size_t)n * ni + j] * dact[n];
                g1 += W[(size_t)(n + 1) * ni + j] * dact[n + 1];
                g2 += W[(size_t)(n + 2) * ni + j] * dact[n + 2];
                g3 += W[(size_t)(n + 3) * ni + j] * dact[n + 3];
            }
            for (; n < no; n++) g0 += W[(size_t)n * ni + j] * dact[n];
            beta[(size_t)i * nin + j] = ((g0 + g1) + (g2 + g3)) * sc[j];
        }
    }
    sync();  // the next atom reuses the scratch
}

// One wavefront (= one workgroup) per atom, weights read from global memory
// (L2).
__global__ __launch_bounds__(64) void mlp_energy_grad_kernel(int64_t natoms, int nin, int nelem,
                                                              const int64_t *__restrict__ species,
                                                              const int *__restrict__ layout,
                                                              const double *__restrict__ params,
                                                              const double *__restrict__ dmin,
                                                              const double *__restrict__ scale,
                                                              const double *__restrict__ x, double *__restrict__ e_out,
                                                              double *__restrict__ beta, int nlm, int hw) {
    extern __shared__ double sm[];
    double *h0 = sm;
    double *dact = h0 + nin;
    double *hout = dact + nlm * hw;
    mlp_atom(blockIdx.x, threadIdx.x, nin, nelem, species, layout, params, dmin, scale, x, e_out, beta, h0, dact, hout,
             hw, WgSync());
}

// Persistent workgroups of MLP_LW wavefronts: the parameters of every
// element network are copied into LDS once per workgroup, then each
// wavefront runs atoms (grid stride) with its own scratch, reading the
// weights from LDS instead of L2.
constexpr int MLP_LW = 4;
__global__ __launch_bounds__(64 * MLP_LW) void mlp_lds_kernel(int64_t natoms, int nin, int nelem,
                                                               const int64_t *__restrict__ species,
                                                               const int *__restrict__ layout,
                                                               const double *__restrict__ params, int nparams,
                                                               const double *__restrict__ dmin,
                                                               const double *__restrict__ scale,
                                                               const double *__restrict__ x,
                                                               double *__restrict__ e_out, double *__restrict__ beta,
                                                               int nlm, int hw) {
    extern __shared__ double sm[];
    double *P = sm;
    // eight loads in flight per thread before their LDS stores
    for (int k0 = threadIdx.x; k0 < nparams; k0 += 8 * blockDim.x) {
        double v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int k = k0 + u * blockDim.x;
            v[u] = k < nparams ? params[k] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (k0 + u * (int)blockDim.x < nparams) P[k0 + u * blockDim.x] = v[u];
    }
    __syncthreads();
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    double *h0 = sm + nparams + (size_t)wv * (nin + 2 * nlm * hw);
    double *dact = h0 + nin;
    double *hout = dact + nlm * hw;
    for (int64_t i = (int64_t)blockIdx.x * MLP_LW + wv; i < natoms; i += (int64_t)gridDim.x * MLP_LW)
        mlp_atom(i, lane, nin, nelem, species, layout, P, dmin, scale, x, e_out, beta, h0, dact, hout, hw,
                 WaveSync());
}

// ---------------------------------------------------------- matrix cores
// 16 atoms per workgroup of eight wavefronts; every layer is a GEMM on the
// FP64 matrix cores (v_mfma_f64_16x16x4_f64: A[i][k] in lane i + 16 k,
// B[k][j] in lane j + 16 k, D[i][j] in lane j + 16 (i % 4), element i / 4).
// Forward, per 16-neuron tile: Z^T = W_k H_{k-1}^T (A = W_k, B = H^T),
// H_k = act(Z + b_k); backward: G_{k-1} = (G_k W_k) * act'_{k-1} (A = G_k,
// B = W_k), dE/dx = (G_0 W_0) * scale.
// Bound by the latency of its chain (a handful of layers, each a few products
// and one activation), not by any rate, so every step is spread over the
// whole workgroup: the wavefronts of a tile split the sum over k (ks parts,
// added through LDS), and then a thread has one (atom, neuron) for the
// activation, whose tanh is the longest link of the chain.  The tile's inputs
// and species are on their way before the element is known, those of the next
// tile before this one is computed; the weights come a row per wavefront,
// eight rows in flight; the layout is one register, an int per lane.
// Four wavefronts with whole tiles and four activations to a lane
// (mlp_mfma4_kernel): 1000 atoms of 30 inputs 16.3 -> 13.3 us, 777 atoms of 55
// inputs with two elements mixed 32.6 -> 23.7, 4096 of 55 18.7 -> 14.1, 12000
// of 147 65 -> 43, 200000 of 55 411 -> 330.
// The element's weights are staged in LDS first, zero-padded, and every
// activation row is zero past its width, so the GEMM steps need no bounds
// tests (the K loops run over multiples of 4).  LDS rows are 2 doubles past
// a multiple of 32: the operand reads whose lanes walk down 16 rows fall in
// distinct banks.  The 16 atoms may belong to different elements: the tile
// runs the network of every element present and keeps each atom's own
// results.
typedef double mlp_d4 __attribute__((ext_vector_type(4)));
constexpr int MLP_TILE = 16, MLP_WV = 8, MLP_T = 64 * MLP_WV;
constexpr int MLP_XC = 3;          // 64-column groups of a tile's inputs held in registers
constexpr int MLP_ZP = 16 * 17;    // doubles of one wavefront's partial tile

__host__ __device__ inline int mlp_r16(int n) { return (n + 15) & ~15; }
__host__ __device__ inline int mlp_r4(int n) { return (n + 3) & ~3; }
__host__ __device__ inline int mlp_row(int n) { return ((n + 31) & ~31) + 2; }  // LDS row stride

// Parts the k sum of a layer with t tiles is split into, with room for zp
// partial tiles: a power of two, t * parts <= min(wavefronts, zp).
__host__ __device__ inline int mlp_parts(int t, int zp) {
    const int m = zp < MLP_WV ? zp : MLP_WV;
    return t >= m ? 1 : (8 * t <= m ? 8 : (4 * t <= m ? 4 : (2 * t <= m ? 2 : 1)));
}

// acc = sum over the steps t = t0, t0 + ts, ... < S of A[lane & 15][4t ..] x
// B[4t ..][col]: a = &A[lane & 15][lane >> 4] (row-major A), b = &B[lane >>
// 4][col], bstep = 4 x the row stride of B.  Two accumulators in turn.
__device__ inline mlp_d4 mlp_gemm_part(int t0, int ts, int S, const double *a, const double *b, int bstep) {
    mlp_d4 c0 = {0.0, 0.0, 0.0, 0.0}, c1 = c0;
    int t = t0;
    for (; t + ts < S; t += 2 * ts) {
        const double a0 = a[4 * t], a1 = a[4 * (t + ts)], b0 = b[t * bstep], b1 = b[(t + ts) * bstep];
        c0 = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b0, c0, 0, 0, 0);
        c1 = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b1, c1, 0, 0, 0);
    }
    if (t < S) c0 = __builtin_amdgcn_mfma_f64_16x16x4f64(a[4 * t], b[t * bstep], c0, 0, 0, 0);
    return c0 + c1;
}

// A call, not inlined: in the loops over tiles, elements and layers the
// constants of the exponentials were otherwise held in registers throughout
// (186 spilled).
__device__ __attribute__((noinline)) double2 mlp_act(int act, double z) {
    double a, da;
    act_fdf(act, z, a, da);
    return make_double2(a, da);
}

// nbuf: activation buffers ([16][HP] each); zpn: partial tiles.
__global__ __launch_bounds__(MLP_T) __attribute__((amdgpu_waves_per_eu(4))) void mlp_mfma_kernel(int64_t natoms, int nin, int nelem,
                                                         const int64_t *__restrict__ species,
                                                         const int *__restrict__ layout,
                                                         const double *__restrict__ params,
                                                         const double *__restrict__ dmin,
                                                         const double *__restrict__ scale,
                                                         const double *__restrict__ x, double *__restrict__ e_out,
                                                         double *__restrict__ beta, int nlm, int hw, int nbuf, int zpn) {
    constexpr int AR = MLP_TILE / MLP_WV, RU = MLP_MAXW / MLP_WV;  // atoms and rows of W per wavefront
    extern __shared__ double sm[];
    __shared__ int s_sp[MLP_TILE];  // element of each atom; -1 no network, -2 past the end
    __shared__ int s_wo[MLP_MAXL];  // offset of layer k's padded W, then its b, in wl
    const int P0 = mlp_row(nin), HP = mlp_row(hw);
    double *h0 = sm;                                     // [16][P0] scaled inputs, zero-padded
    double *hact = h0 + MLP_TILE * P0;                   // [nbuf][16][HP] activations of the hidden layers, in turn
    double *hder = hact + (size_t)nbuf * MLP_TILE * HP;  // [nlm][16][HP] act', then gradients
    double *zp = hder + (size_t)nlm * MLP_TILE * HP;     // [zpn] partial tiles
    double *wl = zp + (size_t)zpn * MLP_ZP;              // W_k [r16(nout)][row(nin)], b_k [r16(nout)]
    const int tid = threadIdx.x, wv = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int ri = lane & 15, kq = lane >> 4;
    const int ta = tid & 15, tn = tid >> 4;  // the thread's atom and neuron in the combining steps
    // tiles [t0, t1) of this workgroup, in order: an element's weights stay
    // staged from one tile to the next (atoms come sorted by element)
    const int64_t ntiles = (natoms + MLP_TILE - 1) / MLP_TILE;
    const int64_t per = (ntiles + gridDim.x - 1) / gridDim.x;
    const int64_t t0 = (int64_t)blockIdx.x * per, t1 = t0 + per < ntiles ? t0 + per : ntiles;
    int staged = -1;  // element whose weights are in wl
    // wavefront w loads the inputs of atoms AR w .. AR w + AR - 1
    double xv[AR * MLP_XC];
    int64_t spv = 0;
    auto fetch = [&](int64_t a0) __attribute__((always_inline)) {
        if (tid < MLP_TILE) spv = a0 + tid < natoms ? species[a0 + tid] : 0;
#pragma unroll
        for (int u = 0; u < AR * MLP_XC; u++) {
            const int64_t a = a0 + AR * wv + u % AR;
            const int c = u / AR * 64 + lane;
            xv[u] = a < natoms && c < nin ? x[(size_t)a * nin + c] : 0.0;
        }
    };
    if (t0 < t1) fetch(t0 * MLP_TILE);
    // an element's layout in one register, an int per lane (MLP_STRIDE < 64)
    const int lay0 = layout[lane < MLP_STRIDE ? lane : 0];
    for (int64_t tl = t0; tl < t1; tl++) {
        const int64_t a0 = tl * MLP_TILE;
        __syncthreads();  // the previous tile is done with s_sp and the scratch
        if (tid < MLP_TILE) {
            int e = -2;
            if (a0 + tid < natoms) e = (spv >= 0 && spv < nelem) ? (int)spv : -1;
            s_sp[tid] = e;
        }
        __syncthreads();
        const int mine = s_sp[ri];
        bool held = true;  // xv has this tile's inputs
        for (int el = 0; el < nelem; el++) {
            if (!__ballot(mine == el)) continue;  // uniform over the workgroup
            const int layv = el == 0 ? lay0 : layout[el * MLP_STRIDE + (lane < MLP_STRIDE ? lane : 0)];
            auto lay = [&](int k, int q) { return __builtin_amdgcn_readlane(layv, 1 + MLP_LSTRIDE * k + q); };
            const int nl = __builtin_amdgcn_readlane(layv, 0);
            const double *dm = dmin + (size_t)el * nin, *sc = scale + (size_t)el * nin;
            double dv[MLP_XC], sv[MLP_XC];
#pragma unroll
            for (int u = 0; u < MLP_XC; u++) {
                const int c = u * 64 + lane;
                dv[u] = c < nin ? dm[c] : 0.0;
                sv[u] = c < nin ? sc[c] : 0.0;
            }
            if (!held) fetch(a0);
            if (el != staged) {  // uniform over the workgroup
                staged = el;
                // 64 columns of a layer at a time
                for (int k = 0, c0 = 0, wo = 0; k < nl;) {
                    const int ni = lay(k, 0), no = lay(k, 1), R = mlp_r16(no), C = mlp_row(ni), K = mlp_r16(ni);
                    const double *W = params + lay(k, 3);
                    const int c = c0 + lane;
                    double v[RU];
#pragma unroll
                    for (int u = 0; u < RU; u++) {
                        const int r = wv + MLP_WV * u;
                        v[u] = r < no && c < ni ? W[r * ni + c] : 0.0;
                    }
#pragma unroll
                    for (int u = 0; u < RU; u++) {
                        const int r = wv + MLP_WV * u;
                        if (r < R && c < K) wl[wo + r * C + c] = v[u];
                    }
                    if (c0 == 0) {
                        if (tid < R) wl[wo + R * C + tid] = tid < no ? params[lay(k, 4) + tid] : 0.0;
                        if (tid == 0) s_wo[k] = wo;
                    }
                    c0 += 64;
                    if (c0 >= K) {
                        wo += R * (C + 1);
                        c0 = 0;
                        k++;
                    }
                }
            }
#pragma unroll
            for (int u = 0; u < AR * MLP_XC; u++) {
                const int t = AR * wv + u % AR, c = u / AR * 64 + lane;
                if (c < P0) h0[t * P0 + c] = c < nin ? (xv[u] - dv[u / AR]) * sv[u / AR] : 0.0;
            }
            for (int c = 64 * MLP_XC + lane; c < P0; c += 64)
                for (int u = 0; u < AR; u++) {
                    const int64_t a = a0 + AR * wv + u;
                    h0[(AR * wv + u) * P0 + c] =
                        a < natoms && c < nin ? (x[(size_t)a * nin + c] - dm[c]) * sc[c] : 0.0;
                }
            held = false;
            __syncthreads();
            // the next tile's inputs, once this one's are no longer needed
            if (tl + 1 < t1 && !__ballot(mine > el)) fetch(a0 + MLP_TILE);
            // forward
            const double *hin = h0;
            int ldi = P0;
            for (int k = 0; k < nl; k++) {
                const int ni = lay(k, 0), no = lay(k, 1), act = lay(k, 2), C = mlp_row(ni), T = mlp_r16(no) >> 4;
                const double *W = wl + s_wo[k], *bias = W + mlp_r16(no) * C;
                double *ho = hact + (size_t)(k % (nbuf > 0 ? nbuf : 1)) * MLP_TILE * HP;
                double *hd = hder + (size_t)k * MLP_TILE * HP;
                const int ks = mlp_parts(T, zpn);
                if (wv < T * ks) {
                    // D[j][i] = sum_k W[j][k] H[i][k]: A rows = neurons of the
                    // tile, B columns = atoms
                    const int ct = wv / ks;
                    const mlp_d4 acc = mlp_gemm_part(wv - ct * ks, ks, mlp_r4(ni) >> 2, W + (ct * 16 + ri) * C + kq,
                                                     hin + ri * ldi + kq, 4);
#pragma unroll
                    for (int r = 0; r < 4; r++) zp[wv * MLP_ZP + (kq + 4 * r) * 17 + ri] = acc[r];
                }
                __syncthreads();
                for (int j = tn; j < 16 * T; j += MLP_T / 16) {
                    const double *z = zp + (j >> 4) * ks * MLP_ZP + (j & 15) * 17 + ta;
                    double v = bias[j];
                    for (int p = 0; p < ks; p++) v += z[p * MLP_ZP];
                    double2 f = mlp_act(act, v);
                    if (j >= no) f = make_double2(0.0, 0.0);  // zero past the layer width
                    if (k < nl - 1)
                        ho[ta * HP + j] = f.x;
                    else if (j == 0 && s_sp[ta] == el)
                        e_out[a0 + ta] = f.x;
                    hd[ta * HP + j] = f.y;
                }
                __syncthreads();
                hin = ho;
                ldi = HP;
            }
            // backward; hder of the output layer (one neuron) already is dE/dz
            for (int k = nl - 1; k >= 1; k--) {
                const int ni = lay(k, 0), no = lay(k, 1), C = mlp_row(ni), T = mlp_r16(ni) >> 4, S = mlp_r4(no) >> 2;
                const double *W = wl + s_wo[k];
                const double *g = hder + (size_t)k * MLP_TILE * HP;
                double *gp = hder + (size_t)(k - 1) * MLP_TILE * HP;
                const int ks = S > 1 ? mlp_parts(T, zpn) : 1;
                if (wv < T * ks) {
                    // B[n][j] = W[n][j]
                    const int ct = wv / ks;
                    const mlp_d4 acc = mlp_gemm_part(wv - ct * ks, ks, S, g + ri * HP + kq, W + kq * C + ct * 16 + ri,
                                                     4 * C);
#pragma unroll
                    for (int r = 0; r < 4; r++) zp[wv * MLP_ZP + ri * 17 + kq + 4 * r] = acc[r];
                }
                __syncthreads();
                for (int j = tn; j < 16 * T; j += MLP_T / 16) {
                    const double *z = zp + (j >> 4) * ks * MLP_ZP + (j & 15) * 17 + ta;
                    double v = 0.0;
                    for (int p = 0; p < ks; p++) v += z[p * MLP_ZP];
                    gp[ta * HP + j] *= v;
                }
                __syncthreads();
            }
            {
                const int S = mlp_r4(lay(0, 1)) >> 2, C = mlp_row(nin);
                const double *W = wl + s_wo[0];
                for (int ct = wv; ct * 16 < nin; ct += MLP_WV) {
                    const int j = ct * 16 + ri;
                    const double sj = j < nin ? sc[j] : 0.0;
                    const mlp_d4 acc = mlp_gemm_part(0, 1, S, hder + ri * HP + kq, W + kq * C + j, 4 * C);
                    if (j < nin) {
#pragma unroll
                        for (int r = 0; r < 4; r++) {
                            const int row = kq + 4 * r;
                            if (s_sp[row] == el) beta[(size_t)(a0 + row) * nin + j] = acc[r] * sj;
                        }
                    }
                }
            }
            __syncthreads();  // the next element reuses the scratch
        }
        if (held && tl + 1 < t1) fetch(a0 + MLP_TILE);  // no atom of the tile has a network
        // atoms without a network: NaN results
        for (int q = tid; q < MLP_TILE * nin; q += MLP_T) {
            const int t = q / nin;
            if (s_sp[t] == -1) beta[(size_t)(a0 + t) * nin + (q - t * nin)] = __builtin_nan("");
        }
        if (tid < MLP_TILE && s_sp[tid] == -1) e_out[a0 + tid] = __builtin_nan("");
    }
}

// The same with four wavefronts to a tile, whole 16-neuron tiles per wavefront
// and four activations to a lane, for many tiles of short inputs and narrow
// layers: its chain through a tile is longer, but three workgroups share a CU
// where the registers of the eight-wavefront kernel leave room for two, and
// the tanh of many tiles are then spread better (rule at mlp_four_waves).
// acc = sum_k A[lane & 15][k] B[k][col], k < K (a multiple of 4):
// a = &A[lane & 15][lane >> 4] (row-major A, k steps of 4 elements),
// b = &B[lane >> 4][col], bstep = 4 x the row stride of B.  Four
// accumulators take the k steps in turn (four independent MFMA chains).
__device__ inline mlp_d4 mlp_gemm_tile(int K, const double *a, const double *b, int bstep) {
    mlp_d4 c0 = {0.0, 0.0, 0.0, 0.0}, c1 = c0, c2 = c0, c3 = c0;
    const int S = K >> 2;
    int t = 0;
    for (; t + 4 <= S; t += 4) {
        const double a0 = a[4 * t], a1 = a[4 * t + 4], a2 = a[4 * t + 8], a3 = a[4 * t + 12];
        const double b0 = b[t * bstep], b1 = b[(t + 1) * bstep], b2 = b[(t + 2) * bstep], b3 = b[(t + 3) * bstep];
        c0 = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b0, c0, 0, 0, 0);
        c1 = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b1, c1, 0, 0, 0);
        c2 = __builtin_amdgcn_mfma_f64_16x16x4f64(a2, b2, c2, 0, 0, 0);
        c3 = __builtin_amdgcn_mfma_f64_16x16x4f64(a3, b3, c3, 0, 0, 0);
    }
    for (; t < S; t++) c0 = __builtin_amdgcn_mfma_f64_16x16x4f64(a[4 * t], b[t * bstep], c0, 0, 0, 0);
    return (c0 + c1) + (c2 + c3);
}

__global__ __launch_bounds__(256) void mlp_mfma4_kernel(int64_t natoms, int nin, int nelem,
                                                        const int64_t *__restrict__ species,
                                                        const int *__restrict__ layout,
                                                        const double *__restrict__ params,
                                                        const double *__restrict__ dmin,
                                                        const double *__restrict__ scale,
                                                        const double *__restrict__ x, double *__restrict__ e_out,
                                                        double *__restrict__ beta, int nlm, int hw) {
    extern __shared__ double sm[];
    __shared__ int s_sp[MLP_TILE];  // element of each atom; -1 no network, -2 past the end
    __shared__ int s_wo[MLP_MAXL];  // offset of layer k's padded W, then its b, in wl
    const int P0 = mlp_row(nin), HP = mlp_row(hw);
    double *h0 = sm;                                 // [16][P0] scaled inputs, zero-padded
    double *hact = h0 + MLP_TILE * P0;               // [nlm][16][HP] activations
    double *hder = hact + (size_t)nlm * MLP_TILE * HP;  // [nlm][16][HP] act', then gradients
    double *wl = hder + (size_t)nlm * MLP_TILE * HP;    // W_k [r16(nout)][row(nin)], b_k [r16(nout)]
    const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63;
    const int ri = lane & 15, kq = lane >> 4;
    // tiles [t0, t1) of this workgroup, in order: an element's weights stay
    // staged from one tile to the next (atoms come sorted by element)
    const int64_t ntiles = (natoms + MLP_TILE - 1) / MLP_TILE;
    const int64_t per = (ntiles + gridDim.x - 1) / gridDim.x;
    const int64_t t0 = (int64_t)blockIdx.x * per, t1 = t0 + per < ntiles ? t0 + per : ntiles;
    int staged = -1;  // element whose weights are in wl
    for (int64_t tl = t0; tl < t1; tl++) {
        const int64_t a0 = tl * MLP_TILE;
        __syncthreads();  // the previous tile is done with s_sp and the scratch
        if (tid < MLP_TILE) {
            const int64_t a = a0 + tid;
            int e = -2;
            if (a < natoms) {
                const int64_t sp = species[a];
                e = (sp >= 0 && sp < nelem) ? (int)sp : -1;
            }
            s_sp[tid] = e;
        }
        __syncthreads();
        for (int el = 0; el < nelem; el++) {
            bool any = false;
            for (int t = 0; t < MLP_TILE; t++) any = any || s_sp[t] == el;
            if (!any) continue;  // uniform over the workgroup
            const int *lay = layout + el * MLP_STRIDE;
            const int nl = lay[0];
            const double *dm = dmin + (size_t)el * nin, *sc = scale + (size_t)el * nin;
            // staging: eight loads in flight per thread before their LDS stores
            for (int q0 = tid; q0 < MLP_TILE * P0; q0 += 256 * 8) {
                double v[8];
#pragma unroll
                for (int u = 0; u < 8; u++) {
                    const int q = q0 + 256 * u;
                    const int t = q / P0, j = q - t * P0;
                    const int64_t a = a0 + t;
                    v[u] = (q < MLP_TILE * P0 && a < natoms && j < nin) ? (x[(size_t)a * nin + j] - dm[j]) * sc[j]
                                                                         : 0.0;
                }
#pragma unroll
                for (int u = 0; u < 8; u++)
                    if (q0 + 256 * u < MLP_TILE * P0) h0[q0 + 256 * u] = v[u];
            }
            if (el != staged) {  // uniform over the workgroup
                staged = el;
                int wo = 0;
                for (int k = 0; k < nl; k++) {
                    const int *L = lay + 1 + MLP_LSTRIDE * k;
                    const int ni = L[0], no = L[1], R = mlp_r16(no), C = mlp_row(ni);
                    const double *W = params + L[3], *bias = params + L[4];
                    for (int q0 = tid; q0 < R * C + R; q0 += 256 * 8) {
                        double v[8];
#pragma unroll
                        for (int u = 0; u < 8; u++) {
                            const int q = q0 + 256 * u;
                            v[u] = 0.0;
                            if (q < R * C) {
                                const int r = q / C, c = q - r * C;
                                if (r < no && c < ni) v[u] = W[r * ni + c];
                            } else if (q - R * C < no) {
                                v[u] = bias[q - R * C];
                            }
                        }
#pragma unroll
                        for (int u = 0; u < 8; u++)
                            if (q0 + 256 * u < R * C + R) wl[wo + q0 + 256 * u] = v[u];
                    }
                    if (tid == 0) s_wo[k] = wo;
                    wo += R * C + R;
                }
            }
            __syncthreads();
            // forward
            const double *hin = h0;
            int ldi = P0;
            for (int k = 0; k < nl; k++) {
                const int *L = lay + 1 + MLP_LSTRIDE * k;
                const int ni = L[0], no = L[1], act = L[2], C = mlp_row(ni);
                const double *W = wl + s_wo[k], *bias = W + mlp_r16(no) * C;
                double *ho = hact + (size_t)k * MLP_TILE * HP, *hd = hder + (size_t)k * MLP_TILE * HP;
                for (int ct = wv; ct * 16 < no; ct += 4) {
                    // D[j][i] = sum_k W[j][k] H[i][k]: A rows = neurons of the
                    // tile, B columns = atoms
                    const mlp_d4 acc = mlp_gemm_tile(mlp_r4(ni), W + (ct * 16 + ri) * C + kq, hin + ri * ldi + kq, 4);
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const int j = ct * 16 + kq + 4 * r;  // neuron; the lane's atom is ri
                        double av = 0.0, da = 0.0;          // zero past the layer width
                        if (j < no) act_fdf(act, acc[r] + bias[j], av, da);
                        ho[ri * HP + j] = av;
                        hd[ri * HP + j] = da;
                    }
                }
                __syncthreads();
                hin = ho;
                ldi = HP;
            }
            if (tid < MLP_TILE && s_sp[tid] == el) e_out[a0 + tid] = hin[tid * HP];
            // backward; hder of the output layer (one neuron) already is dE/dz
            for (int k = nl - 1; k >= 1; k--) {
                const int *L = lay + 1 + MLP_LSTRIDE * k;
                const int ni = L[0], no = L[1], C = mlp_row(ni);
                const double *W = wl + s_wo[k];
                const double *g = hder + (size_t)k * MLP_TILE * HP;
                double *gp = hder + (size_t)(k - 1) * MLP_TILE * HP;
                for (int ct = wv; ct * 16 < ni; ct += 4) {
                    const int j = ct * 16 + ri;
                    // B[n][j] = W[n][j]
                    const mlp_d4 acc = mlp_gemm_tile(mlp_r4(no), g + ri * HP + kq, W + kq * C + j, 4 * C);
#pragma unroll
                    for (int r = 0; r < 4; r++) gp[(kq + 4 * r) * HP + j] *= acc[r];
                }
                __syncthreads();
            }
            {
                const int *L = lay + 1;
                const int no = L[1], C = mlp_row(nin);
                const double *W = wl + s_wo[0];
                for (int ct = wv; ct * 16 < nin; ct += 4) {
                    const int j = ct * 16 + ri;
                    const mlp_d4 acc = mlp_gemm_tile(mlp_r4(no), hder + ri * HP + kq, W + kq * C + j, 4 * C);
                    if (j < nin) {
                        const double sj = sc[j];
#pragma unroll
                        for (int r = 0; r < 4; r++) {
                            const int row = kq + 4 * r;
                            if (s_sp[row] == el) beta[(size_t)(a0 + row) * nin + j] = acc[r] * sj;
                        }
                    }
                }
            }
            __syncthreads();  // the next element reuses the scratch
        }
        // atoms without a network: NaN results
        for (int q = tid; q < MLP_TILE * nin; q += 256) {
            const int t = q / nin;
            if (s_sp[t] == -1) beta[(size_t)(a0 + t) * nin + (q - t * nin)] = __builtin_nan("");
        }
        if (tid < MLP_TILE && s_sp[tid] == -1) e_out[a0 + tid] = __builtin_nan("");
    }
}

// One element's parameters from their own tensors into the packed arrays
// (layout row, W, b, W^T, dmin, scale): one launch instead of a transpose per
// layer, a concatenation and a copy of the layout, so that a call can take the
// parameters as they are at that moment (3 us for two hidden layers of 30).
struct MlpPack {
    int lay[MLP_STRIDE];
    const double *w[MLP_MAXL], *b[MLP_MAXL], *dmin, *scale;
};

__global__ __launch_bounds__(256) void mlp_pack_kernel(MlpPack p, int nin, int *__restrict__ layout,
                                                       double *__restrict__ params, double *__restrict__ dmin,
                                                       double *__restrict__ scale) {
    const int t0 = blockIdx.x * blockDim.x + threadIdx.x, nt = gridDim.x * blockDim.x;
    if (t0 < MLP_STRIDE) layout[t0] = p.lay[t0];
    for (int k = t0; k < nin; k += nt) {
        dmin[k] = p.dmin[k];
        scale[k] = p.scale[k];
    }
    for (int l = 0; l < p.lay[0]; l++) {
        const int *L = p.lay + 1 + MLP_LSTRIDE * l;
        const int ni = L[0], no = L[1];
        for (int k = t0; k < ni * no; k += nt) {
            const double v = p.w[l][k];
            const int r = k / ni, c = k - r * ni;
            params[L[3] + k] = v;
            params[L[5] + c * no + r] = v;
        }
        for (int k = t0; k < no; k += nt) params[L[4] + k] = p.b[l][k];
    }
}

static int mlp_check_layout(int nin, int nelem, const int *h_layout) {
    PXFF_REQUIRE(nin > 0 && nin <= MLP_MAXIN, "descriptor length must be in 1..1024");
    PXFF_REQUIRE(nelem > 0 && h_layout != nullptr, "need at least one element network");
    for (int e = 0; e < nelem; e++) {
        const int *lay = h_layout + e * MLP_STRIDE;
        const int nl = lay[0];
        PXFF_REQUIRE(nl >= 1 && nl <= MLP_MAXL, "1..8 layers per element network");
        int prev = nin;
        for (int k = 0; k < nl; k++) {
            const int *L = lay + 1 + MLP_LSTRIDE * k;
            PXFF_REQUIRE(L[0] == prev, "layer input width does not match the previous layer");
            PXFF_REQUIRE(L[1] >= 1 && L[1] <= MLP_MAXW, "layer widths must be in 1..64");
            PXFF_REQUIRE(L[2] >= 0 && L[2] <= 5, "unknown activation id");
            prev = L[1];
        }
        PXFF_REQUIRE(prev == 1, "the last layer must have one output (the atomic energy)");
    }
    return 0;
}

// Dynamic LDS of the matrix-core kernels: what a CU has, less their static LDS.
constexpr size_t MLP_LDS_MAX = 160 * 1024 - 1024;

// Workgroups of lds bytes that a CU's LDS keeps resident, at most `most`.
static int64_t mlp_resident(size_t lds, int64_t most) {
    return std::max<int64_t>(1, std::min<int64_t>(most, (int64_t)(160 * 1024) / (int64_t)(lds + 1024)));
}

// Raise a kernel's dynamic LDS limit to lds; set is the limit so far.  Under a
// lock, so that concurrent callers never lower it below what another relies on.
static int mlp_raise_lds(const void *kernel, int lds, std::atomic<int> &set) {
    static std::mutex mu;
    std::lock_guard<std::mutex> lock(mu);
    if (lds > set.load(std::memory_order_relaxed)) {
        PXFF_HIP_CHECK(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds));
        set.store(lds, std::memory_order_relaxed);
    }
    return 0;
}

// Four wavefronts to a tile (mlp_mfma4_kernel, lds4 bytes) or eight
// (mlp_mfma_kernel, lds8 bytes; at most two of its workgroups fit the
// registers of a CU): by the rounds that the tiles take, a round of the four
// being 1 + (LDS row of the inputs) / 150 of one of the eight (1.2 to 32
// inputs, 1.4 to 64, 1.7 to 96; past three workgroups per CU more of the four
// only slow each other).  Over 1 to 3 layers of 16 to 64, 14 to 91 inputs and 2000 to
// 200000 atoms the choice is at most 5 % slower than the better of the two.
// Where one of them does not fit, the other.  Measured, us, eight / four, two
// elements, layers of 30, 30: 30 inputs, 2000 atoms 23 / 29, 8192 23 / 29,
// 8300 32 / 29, 12000 32 / 26, 16000 39 / 46, 20000 47 / 41, 60000 104 / 90,
// 136000 208 / 201, 200000 307 / 285; with the elements mixed 12000 61 / 44;
// 91 inputs, 8300 38 / 42, 16000 64 / 60, 32000 114 / 104.  Layers of 16, 16
// and 30 inputs, 12000 28 / 20, 200000 259 / 223.
static bool mlp_four_waves(int64_t ntiles, int nin, size_t lds8, size_t lds4) {
    if (lds4 > MLP_LDS_MAX || lds8 > MLP_LDS_MAX) return lds4 <= MLP_LDS_MAX;
    const int64_t n4 = num_cus() * mlp_resident(lds4, 3), n8 = num_cus() * mlp_resident(lds8, 2);
    return (ntiles + n4 - 1) / n4 * (150 + mlp_row(nin)) <= (ntiles + n8 - 1) / n8 * 150;
}

}  // namespace pxff

using namespace pxff;

extern "C" int pxff_mlp_pack(int nin, int nelem, const int *h_layout, const double *const *h_tensors, int *d_layout,
                             double *d_params, double *d_dmin, double *d_scale, void *stream) {
    const int rc = mlp_check_layout(nin, nelem, h_layout);
    if (rc) return rc;
    PXFF_REQUIRE(h_tensors != nullptr, "null tensor table");
    for (int e = 0; e < nelem; e++) {
        const double *const *t = h_tensors + (size_t)e * (2 + 2 * MLP_MAXL);
        MlpPack p{};
        std::copy(h_layout + e * MLP_STRIDE, h_layout + (e + 1) * MLP_STRIDE, p.lay);
        p.dmin = t[0];
        p.scale = t[1];
        int most = nin;
        for (int l = 0; l < p.lay[0]; l++) {
            p.w[l] = t[2 + 2 * l];
            p.b[l] = t[3 + 2 * l];
            most = std::max(most, p.lay[1 + MLP_LSTRIDE * l] * p.lay[2 + MLP_LSTRIDE * l]);
        }
        mlp_pack_kernel<<<std::min(64, div_up(most, 256)), 256, 0, (hipStream_t)stream>>>(
            p, nin, d_layout + e * MLP_STRIDE, d_params, d_dmin + (size_t)e * nin, d_scale + (size_t)e * nin);
        PXFF_LAUNCH_CHECK();
    }
    return 0;
}

extern "C" int pxff_mlp_energy_grad(int64_t natoms, int nin, int nelem, const int64_t *d_species,
                                    const int *h_layout, const int *d_layout, const double *d_params,
                                    const double *d_dmin, const double *d_scale, const double *d_x, double *d_e,
                                    double *d_beta, void *stream) {
    const int rc = mlp_check_layout(nin, nelem, h_layout);
    if (rc) return rc;
    if (natoms <= 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    // parameter array length: the furthest end of any W, b or W^T
    int64_t nparams = 0;
    for (int e = 0; e < nelem; e++) {
        const int *lay = h_layout + e * MLP_STRIDE;
        for (int k = 0; k < lay[0]; k++) {
            const int *L = lay + 1 + MLP_LSTRIDE * k;
            const int64_t nw = (int64_t)L[0] * L[1];
            nparams = std::max({nparams, L[3] + nw, (int64_t)L[4] + L[1], L[5] + nw});
        }
    }
    // scratch per wavefront: the scaled input, then activations and their
    // derivatives of every layer at a stride of the widest layer
    int nlm = 1, hw = 1;
    for (int e = 0; e < nelem; e++) {
        const int *lay = h_layout + e * MLP_STRIDE;
        nlm = std::max(nlm, lay[0]);
        for (int k = 0; k < lay[0]; k++) hw = std::max(hw, lay[1 + MLP_LSTRIDE * k + 1]);
    }
    const size_t scratch = sizeof(double) * ((size_t)nin + 2 * (size_t)nlm * hw);
    // matrix cores: 16 atoms per workgroup, their scratch and one element's
    // zero-padded weights and biases within the 160 KB of a CU
    size_t wmax = 0;
    for (int e = 0; e < nelem; e++) {
        const int *lay = h_layout + e * MLP_STRIDE;
        size_t w = 0;
        for (int k = 0; k < lay[0]; k++) {
            const int *L = lay + 1 + MLP_LSTRIDE * k;
            w += (size_t)mlp_r16(L[1]) * mlp_row(L[0]) + mlp_r16(L[1]);
        }
        wmax = std::max(wmax, w);
    }
    // partial tiles: one per wavefront, or as many as the widest layer has
    // tiles where that decides whether it all fits
    const int nbuf = std::min(2, nlm - 1);
    auto lds_of = [&](int zpn) {
        return sizeof(double) * (MLP_TILE * ((size_t)mlp_row(nin) + ((size_t)nbuf + nlm) * mlp_row(hw)) +
                                 (size_t)zpn * MLP_ZP + wmax);
    };
    int zpn = MLP_WV;
    if (lds_of(zpn) > MLP_LDS_MAX) zpn = mlp_r16(hw) / 16;
    const size_t ldsm = lds_of(zpn);
    const size_t lds4 =
        sizeof(double) * (MLP_TILE * ((size_t)mlp_row(nin) + 2 * (size_t)nlm * mlp_row(hw)) + wmax);
    const int64_t ntiles = div_up(natoms, MLP_TILE);
    if (mlp_four_waves(ntiles, nin, ldsm, lds4)) {
        static std::atomic<int> dyn_max{65536};
        int rc4 = mlp_raise_lds((const void *)mlp_mfma4_kernel, (int)lds4, dyn_max);
        if (rc4) return rc4;
        // persistent: as many workgroups as the LDS keeps resident (at most
        // 8 per CU), each over a contiguous range of 16-atom tiles
        const int64_t nwg = std::min<int64_t>(ntiles, (int64_t)num_cus() * mlp_resident(lds4, 8));
        mlp_mfma4_kernel<<<(unsigned)nwg, 256, lds4, s>>>(natoms, nin, nelem, d_species, d_layout, d_params, d_dmin,
                                                          d_scale, d_x, d_e, d_beta, nlm, hw);
        PXFF_LAUNCH_CHECK();
        return 0;
    }
    // above 64 KB (long descriptors, e.g. SO3 6/6: 147 inputs) one workgroup
    // per CU; the kernel's static LDS (a few hundred bytes) comes on top
    if (ldsm <= MLP_LDS_MAX) {
        static std::atomic<int> dyn_max{65536};
        int rc8 = mlp_raise_lds((const void *)mlp_mfma_kernel, (int)ldsm, dyn_max);
        if (rc8) return rc8;
        // persistent: as many workgroups as the LDS keeps resident (at most
        // 4 per CU, two by their registers), each over a contiguous range of 16-atom tiles
        const int64_t nwg = std::min<int64_t>(ntiles, (int64_t)num_cus() * mlp_resident(ldsm, 4));
        mlp_mfma_kernel<<<(unsigned)nwg, MLP_T, ldsm, s>>>(
            natoms, nin, nelem, d_species, d_layout, d_params, d_dmin, d_scale, d_x, d_e, d_beta, nlm, hw, nbuf, zpn);
        PXFF_LAUNCH_CHECK();
        return 0;
    }
    const size_t ldsp = sizeof(double) * (size_t)nparams + MLP_LW * scratch;
    if (ldsp <= 160 * 1024) {  // the weights fit in LDS next to the scratch
        static std::atomic<int> attr_set{0};  // the limit is one value: setting it twice is harmless
        if (ldsp > 65536 && !attr_set.load(std::memory_order_relaxed)) {
            PXFF_HIP_CHECK(hipFuncSetAttribute((const void *)mlp_lds_kernel,
                                               hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
            attr_set.store(1, std::memory_order_relaxed);
        }
        // as many resident workgroups as the LDS holds (at most 4 per CU)
        const int64_t per_cu = std::max<int64_t>(1, std::min<int64_t>(4, (int64_t)(160 * 1024) / (int64_t)ldsp));
        const int64_t nwg = std::min<int64_t>((natoms + MLP_LW - 1) / MLP_LW, (int64_t)num_cus() * per_cu);
        mlp_lds_kernel<<<(unsigned)nwg, 64 * MLP_LW, ldsp, s>>>(natoms, nin, nelem, d_species, d_layout, d_params,
                                                               (int)nparams, d_dmin, d_scale, d_x, d_e, d_beta, nlm,
                                                               hw);
        PXFF_LAUNCH_CHECK();
        return 0;
    }
    const size_t lds = scratch;
    if (lds > 65536)
        PXFF_HIP_CHECK(hipFuncSetAttribute((const void *)mlp_energy_grad_kernel,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    PXFF_REQUIRE(natoms <= 0x7fffffff, "too many atoms for one launch");
    mlp_energy_grad_kernel<<<(unsigned)natoms, 64, lds, s>>>(natoms, nin, nelem, d_species, d_layout, d_params, d_dmin,
                                                               d_scale, d_x, d_e, d_beta, nlm, hw);
    PXFF_LAUNCH_CHECK();
    return 0;
}
