// Energy-training inner loop on the device: the training part of NNPTE::error
// (src/nnp/nnpte.cpp:869-927) with Cost::grad (src/ml/nn.cpp:1554-1589), for a training set
// whose descriptors are computed once on the GPU (NNP::symm, nnpte.cpp:1976-1977).
//
// Per call (parameter vector x, batch of structures):
//   1. forward pass of every batch atom (per-species 16-atom tiles, FP64 MFMA as the network
//      kernels): out_i = outb + outw a_L (no type energy, as the reference's training energy);
//   2. per structure b: E_b = sum_i out_i (fixed-order tree), dE_b = (E_b - E_ref) / N_b, the loss
//      and dcdo_b = dC/dE_b / N_b of the loss function (MSE, MAE, HUBER, ASINH);
//   3. forward again, then backward per tile: dcdz_L = dcdo outw .* dadz_L, dcdz_{l-1} =
//      (W_l^T dcdz_l) .* dadz_{l-1}; the tile's gradient (bias: sum over its 16 atoms of dcdz_l;
//      weights: dcdz_l^T a_{l-1} as 16 x 16 MFMA tiles with K = 16 atoms) goes to its own row of
//      a partial buffer in the reference's parameter order (operator>>, nn.cpp:797-831: every
//      layer's biases, then every weight matrix column-major);
//   4. the partial rows of a species are summed in a fixed order: groups of consecutive tiles in
//      tile order, then the groups in order.
// Force training (error_force) adds beta/2 |(F_i - F_ref,i) / N|^2 per atom, the forces being the
// model's force kernels applied to the networks' dout/dG at x; its gradient runs the force pass
// backwards: force residuals, descriptor tangents (k_symm_jvp) and a tangent forward/backward
// network pass per tile (k_train_force_tile).
// Every sum has a fixed order, so results do not depend on timing; they match the CPU
// restatement to rounding (different summation order).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <stdexcept>
#include <vector>

#include "../../include/nnp_capi.h"
#include "basis.hpp"
#include "engine.hpp"
#include "netmm.hpp"

namespace atomnn {

hipError_t launch_symm_jvp(int shape, int ns, const DevPlan* plan, const double* rfe, const double* rfr,
                           const int* atom_type, const DevStruc* S, const int* atom_struc, int ntot, const int* cnt,
                           const int* nbr_j, const int* meta, const double4* r, int maxp, int lmaxp, const double* gF,
                           int all_images, double* V, int ldg, int use_mom, int ntypes, hipStream_t st);

// Per-species network for training.  W_l (padded, row-major wpad_l x in_pad_l) and b_l (padded)
// live in the training parameter buffer; inpw / inpb stay in the model's weight buffer.
struct TrainNet {
    int L, nin, nin_pad, act;
    int nodes[kMaxLayers], wpad[kMaxLayers];
    int64_t woff[kMaxLayers], boff[kMaxLayers];  // into the training parameter buffer
    int rb[kMaxLayers], rw[kMaxLayers];          // offsets of b_l and w_l in the species' parameter vector
    int nparams;
    int64_t inpw_off, inpb_off;  // into the model's weight buffer
    double outw, outb;
};
struct TrainPlan {
    int T;
    TrainNet net[kMaxSpecies];
};
// Species ranges of a batch: tiles, species-sorted batch atoms, partial-buffer rows.
struct TrainTiles {
    int tile_start[kMaxSpecies + 1];
    int atom_start[kMaxSpecies + 1];
    int64_t pbase[kMaxSpecies + 1];  // first partial element of the species' first tile
};

constexpr int kTrainWaves = 4;
constexpr int kTrainThreads = kTrainWaves * kWave;

__device__ __forceinline__ int train_species(const TrainTiles& tt, int ntypes, int tile) {
    int s = 0;
    while (s + 1 < ntypes && tile >= tt.tile_start[s + 1]) ++s;
    return s;
}

// Hidden-layer activation and its derivatives.  GEN = false: tanh hidden layers only (the common
// case; the general switch over every activation costs the kernels about 50 VGPRs).
template <bool GEN>
__device__ __forceinline__ void train_act(int act, double z, double& a, double& d) {
    if constexpr (GEN) {
        act_eval<double>(act, z, a, d);
    } else if (act == NEU_LINEAR) {
        a = z;
        d = 1.0;
    } else {
        a = tanh_m1(z);
        d = 1.0 - a * a;
    }
}
template <bool GEN>
__device__ __forceinline__ double train_act_d2(int act, double z, double a) {
    if constexpr (GEN) return act_d2(act, z);
    return act == NEU_LINEAR ? 0.0 : -2.0 * a * (1.0 - a * a);
}

// Sum over the 16 lanes of a DPP row, on every lane.
__device__ __forceinline__ double row16_sum(double x) {
    auto ror = [](double y, auto ctrl) {
        const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(y), ctrl.value, 0xf, 0xf, false);
        const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(y), ctrl.value, 0xf, 0xf, false);
        return __hiloint2double(hi, lo);
    };
    x += ror(x, std::integral_constant<int, 0x128>{});
    x += ror(x, std::integral_constant<int, 0x124>{});
    x += ror(x, std::integral_constant<int, 0x122>{});
    return x + ror(x, std::integral_constant<int, 0x121>{});
}
// The output unit's sum over 16 of its inputs, one a lane of a DPP row.  Every kernel adds the inputs in this order, 16 at a
// time, and forms the output by train_out, so that a call gives the same errors with and without the gradient, whichever
// kernel takes the tiles.
__device__ __forceinline__ double train_unit_part(double w, double a) {
#pragma clang fp contract(off)
    return row16_sum(w * a);
}
__device__ __forceinline__ double train_out(double outb, double outw, double z) { return fma(z, outw, outb); }

// LDS: ins [16][nin_pad], then per layer A_l [16][wpad_l] and D_l [16][wpad_l] (dadz; dcdz in the
// backward pass, in place).
static size_t train_lds_bytes(const TrainNet& n) {
    size_t e = 16 * (size_t)n.nin_pad;
    for (int l = 0; l < n.L; ++l) e += 2 * 16 * (size_t)n.wpad[l];
    return 8 * e;
}

// MODE 0: forward, out[slot] = outb + outw a_L.  MODE 1: forward and backward, the tile's
// gradient row into `partial`.  MODE 2: forward and the input gradient (fpbp + DODZ::grad,
// nn.cpp:1191-1233, 1620-1628): out[slot] and Y[slot] = dout/dG = inpw .* (w_0^T dodz_0).
// MODE 3: out[slot] and the gradient row of the outputs (seed outw instead of dcdo outw), for
// tiles whose atoms belong to one structure: the reduction then weights the row by dcdo.
// Rows beyond the species' atoms or with batom < 0 (padding) carry nothing.
template <int MODE, bool GEN>
__global__ __launch_bounds__(kTrainThreads) void k_train_tile(
    const TrainPlan* __restrict__ tp, const double* __restrict__ Wm, const double* __restrict__ par, TrainTiles tt,
    int tile0, const int* __restrict__ batom, const int* __restrict__ bslot, const int* __restrict__ bstruct,
    const double* __restrict__ G, int ldg, double* __restrict__ out, const double* __restrict__ dcdo,
    double* __restrict__ partial, double* __restrict__ Y) {
    extern __shared__ __align__(16) double tsh[];
    const int tile = tile0 + blockIdx.x;
    const int s = train_species(tt, tp->T, tile);
    const TrainNet& N = tp->net[s];
    const int a0 = tt.atom_start[s], M = tt.atom_start[s + 1] - a0;
    const int r0 = (tile - tt.tile_start[s]) * 16;
    const int tid = threadIdx.x, wv = tid / kWave, lane = tid % kWave, li = lane & 15, lk = lane >> 4;
    double* ins = tsh;
    double* A[kMaxLayers];
    double* D[kMaxLayers];
    {
        double* p = ins + 16 * N.nin_pad;
        for (int l = 0; l < N.L; ++l) {
            A[l] = p;
            D[l] = p + 16 * N.wpad[l];
            p += 32 * N.wpad[l];
        }
    }
    for (int idx = tid; idx < 16 * N.nin_pad; idx += kTrainThreads) {
        const int r = idx / N.nin_pad, k = idx % N.nin_pad;
        double v = 0.0;
        const int src = r0 + r < M ? batom[a0 + r0 + r] : -1;  // -1: padding row
        if (src >= 0 && k < N.nin) v = Wm[N.inpw_off + k] * (G[(int64_t)src * ldg + k] + Wm[N.inpb_off + k]);
        ins[r * N.nin_pad + k] = v;
    }
    __syncthreads();
    for (int l = 0; l < N.L; ++l) {
        const double* prev = l == 0 ? ins : A[l - 1];
        const int in_pad = l == 0 ? N.nin_pad : N.wpad[l - 1], wp = N.wpad[l];
        if (l == N.L - 1) {  // linear, one unit: four rows a wavefront
            static_assert(kTrainWaves * 4 == 16, "a tile's 16 rows");
            const int row = 4 * wv + lk;
            double e = 0.0;
            for (int n = 0; n < in_pad; n += 16) e += train_unit_part(par[N.woff[l] + n + li], prev[row * in_pad + n + li]);
            for (int n = li; n < wp; n += 16) {
                A[l][row * wp + n] = n == 0 ? par[N.boff[l]] + e : 0.0;
                D[l][row * wp + n] = 1.0;
            }
            __syncthreads();
            break;
        }
        for (int jt = wv; jt < wp / 16; jt += kTrainWaves) {
            const d4_t acc = tile_mm_f64<true>(prev, in_pad, par + N.woff[l], in_pad, in_pad, jt, li, lk);
            const int col = jt * 16 + li;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int row = 4 * v + lk;
                double av, dv;
                train_act<GEN>(N.act, acc[v] + par[N.boff[l] + col], av, dv);
                A[l][row * wp + col] = av;
                D[l][row * wp + col] = dv;
            }
        }
        __syncthreads();
    }
    const int L = N.L;
    if constexpr (MODE != 1) {
        if (tid < 16 && r0 + tid < M && batom[a0 + r0 + tid] >= 0)
            out[bslot[a0 + r0 + tid]] = train_out(N.outb, N.outw, A[L - 1][tid * N.wpad[L - 1]]);
    }
    if constexpr (MODE == 0) {
        return;
    } else if constexpr (MODE == 2) {
        // dodz_L = outw .* dadz_L (unit 0), dodz_{l-1} = (w_l^T dodz_l) .* dadz_{l-1}
        {
            const int wp = N.wpad[L - 1];
            for (int idx = tid; idx < 16 * wp; idx += kTrainThreads) D[L - 1][idx] *= (idx % wp == 0) ? N.outw : 0.0;
        }
        __syncthreads();
        for (int l = L - 1; l > 0; --l) {
            const int wp = N.wpad[l], wq = N.wpad[l - 1];
            for (int jt = wv; jt < wq / 16; jt += kTrainWaves) {
                const d4_t acc = tile_mm_f64<false>(D[l], wp, par + N.woff[l], wq, wp, jt, li, lk);
#pragma unroll
                for (int v = 0; v < 4; ++v) D[l - 1][(4 * v + lk) * wq + jt * 16 + li] *= acc[v];
            }
            __syncthreads();
        }
        const int wp = N.wpad[0];
        for (int jt = wv; jt < N.nin_pad / 16; jt += kTrainWaves) {
            const d4_t acc = tile_mm_f64<false>(D[0], wp, par + N.woff[0], N.nin_pad, wp, jt, li, lk);
            const int col = jt * 16 + li;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int row = 4 * v + lk;
                if (r0 + row < M && col < N.nin && batom[a0 + r0 + row] >= 0)
                    Y[(int64_t)bslot[a0 + r0 + row] * ldg + col] = acc[v] * Wm[N.inpw_off + col];
            }
        }
    } else {
        // dcdz_L = dcdo outw .* dadz_L (single output unit; padded units and rows carry zero)
        {
            const int wp = N.wpad[L - 1];
            for (int idx = tid; idx < 16 * wp; idx += kTrainThreads) {
                const int r = idx / wp, n = idx % wp;
                const bool real = r0 + r < M && n < N.nodes[L - 1] && batom[a0 + r0 + r] >= 0;
                const double c = real ? (MODE == 3 ? N.outw : dcdo[bstruct[a0 + r0 + r]] * N.outw) : 0.0;
                D[L - 1][idx] *= c;
            }
        }
        __syncthreads();
        double* prow = partial + tt.pbase[s] + (int64_t)(tile - tt.tile_start[s]) * N.nparams;
        for (int l = L - 1; l >= 0; --l) {
            const double* prev = l == 0 ? ins : A[l - 1];
            const int wp = N.wpad[l], in_pad = l == 0 ? N.nin_pad : N.wpad[l - 1];
            const int in_real = l == 0 ? N.nin : N.nodes[l - 1], no = N.nodes[l];
            const double* dz = D[l];  // dcdz_l [16][wp]
            // bias gradient: sum over the tile's 16 atoms
            for (int n = tid; n < no; n += kTrainThreads) {
                double g = 0.0;
#pragma unroll
                for (int r = 0; r < 16; ++r) g += dz[r * wp + n];
                prow[N.rb[l] + n] = g;
            }
            // weight gradient dcdz_l^T a_{l-1}: tiles (nt, mt) of 16 x 16, K = the 16 atoms
            const int ntn = wp / 16, ntm = in_pad / 16;
            for (int t = wv; t < ntn * ntm; t += kTrainWaves) {
                const int nt = t / ntm, mt = t % ntm;
                d4_t acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int r = 4 * q + lk;
                    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(dz[r * wp + nt * 16 + li], prev[r * in_pad + mt * 16 + li],
                                                               acc, 0, 0, 0);
                }
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int n = nt * 16 + 4 * v + lk, m = mt * 16 + li;
                    if (n < no && m < in_real) prow[N.rw[l] + m * no + n] = acc[v];
                }
            }
            // dcdz_{l-1} = (W_l^T dcdz_l) .* dadz_{l-1}, in place over dadz_{l-1}
            if (l > 0) {
                const int wq = N.wpad[l - 1];
                for (int jt = wv; jt < wq / 16; jt += kTrainWaves) {
                    const d4_t acc = tile_mm_f64<false>(dz, wp, par + N.woff[l], wq, wp, jt, li, lk);
                    const int col = jt * 16 + li;
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const int row = 4 * v + lk;
                        D[l - 1][row * wq + col] *= acc[v];
                    }
                }
            }
            __syncthreads();
        }
    }
}

// ------------------------------------------------------------------ gradient rows of groups of tiles
// Forward and backward pass of consecutive 16-atom tiles of one species, one gradient row for all of them, for
// networks of H = 1 or 2 tanh layers of at most U = 32 or 64 units and at most 16 NI <= 128 inputs (train_group_shape).
// Two teams of U / 16 wavefronts take the tiles in turn; each wavefront owns one 16-column tile of every hidden layer
// and keeps, for all its tiles, layer 0's weights in registers as MFMA operands (layer 1's in LDS, where both
// directions and teams read them) and its part of the weight gradient as MFMA accumulators: dz^T a of a tile is K = 16
// more steps of the same product.  dz of a wavefront's own columns is already the B operand of its gradient products,
// so LDS holds, besides, only what crosses wavefronts: inputs, a_0, dz_1.  At the end the second team's sums are added
// to the first's, through LDS, and the block writes one row.
//   ROWSEED false: rows of one structure, seed outw (the reduction weights the row by the structure's dcdo)
//   ROWSEED true: seed dcdo[structure] outw per row
// k_train_tile reads the weights from L2 for every tile, its LDS rows start in one bank, and it writes a row of every
// parameter per tile, in 8-byte pieces 512 bytes apart: 155 us on 32768 atoms (16 structures, 3 species, 84-64-64-1;
// 2080 tiles) and 30 us more to add its rows; here 68 and 6 us.  Of the 68, 45 are the tiles (10 on each CU; their 96
// products of 64 cycles per wavefront are 25 us, the rest the tanh, staging and barriers between them), 10 the
// plan's, the atoms' and the weights' loads at the start, 5 the row at the end.  Measured: one team with a block or two on
// a CU 70 and 68 us, with the library's expm1 and quotient in tanh 82.
// Registers: U = 64 leaves a wavefront 256, which H = 2 with more than 96 inputs does not fit; those networks keep
// k_train_tile, as do other depths, activations and widths.
template <int NI>
__host__ __device__ constexpr int tg_ldi() {
    return 16 * NI + 4;  // LDS rows: the 16 rows of a K-step start in different banks
}
template <int H, int NI, int U>
__host__ __device__ constexpr int tg_team_elems() {  // of one team: inputs (two buffers), a_0, dz_1, energies, seeds
    return 2 * 16 * tg_ldi<NI>() + (H - 1) * 2 * 16 * (U + 4) + U + 2 * 16;
}
template <int H, int NI, int U>
__host__ __device__ constexpr int tg_lds_elems() {
    constexpr int run = (H - 1) * U * (U + 4) + 2 * 16 * NI + 2 * tg_team_elems<H, NI, U>();
    constexpr int sum = (4 * (NI + (H - 1) * U / 16) + 4) * 4 * U;  // the second team's accumulators at the end
    return run > sum ? run : sum;
}

template <int H, int NI, int U, bool ROWSEED>
__global__ __launch_bounds__(8 * U, U / 32) void k_train_group(
    const TrainPlan* __restrict__ tp, const double* __restrict__ Wm, const double* __restrict__ par, TrainTiles tt,
    TrainTiles tr, const int* __restrict__ gtile, const int* __restrict__ batom, const int* __restrict__ bslot,
    const int* __restrict__ bstruct, const double* __restrict__ G, int ldg, double* __restrict__ out,
    const double* __restrict__ dcdo, double* __restrict__ partial) {
    extern __shared__ __align__(16) double tsh[];
    constexpr int kThreads = 4 * U, ldi = tg_ldi<NI>(), ldu = U + 4, KI = 4 * NI, KH = U / 4, MH = U / 16;
    constexpr int kPer = kThreads / 16, NV = 16 * NI / kPer;  // threads and inputs of a row in the staging
    const int g = blockIdx.x;
    const int s = train_species(tr, tp->T, g);
    const TrainNet& N = tp->net[s];
    const int nin = N.nin, nin_pad = N.nin_pad, n0 = N.nodes[0], n1 = N.nodes[H - 1];
    const double outw = N.outw, outb = N.outb;
    const int a0 = tt.atom_start[s], M = tt.atom_start[s + 1] - a0, ts0 = tt.tile_start[s];
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = __lane_id();
    const int team = wid / (U / 16), wv = wid - team * (U / 16), tid = wv * kWave + lane, li = lane & 15, lk = lane >> 4;
    double* W1 = tsh;                                       // [U][ldu] (H = 2): layer 1's weights, zero padded
    double* sinw = W1 + (H - 1) * U * ldu;                  // [2][16 NI] inpw, inpb
    double* ins = sinw + 2 * 16 * NI + team * tg_team_elems<H, NI, U>();  // [2][16][ldi]
    double* A0 = ins + 2 * 16 * ldi;                        // [16][ldu] (H = 2)
    double* Z1 = A0 + (H - 1) * 16 * ldu;                   // [16][ldu] (H = 2)
    double* ep = Z1 + (H - 1) * 16 * ldu;                   // [U / 16][16] energies of each wavefront's columns
    double* seed = ep + U;                                  // [2][16]
    const int w0 = N.wpad[0], w1 = H == 2 ? N.wpad[1] : w0;  // padded hidden widths (the last one: w1)
    const int col = wv * 16 + li;
    const bool on0 = col < w0, on1 = col < w1;  // units past a layer's width carry zeros (tanh 0 = 0)
    const int t0 = gtile[g], t1 = gtile[g + 1];
    // Staging of a tile's scaled inputs, kPer threads a row: the row's atom two of the team's tiles ahead, its
    // descriptors loaded a tile ahead (in flight over that tile's products), written to the other buffer before the
    // next tile.
    const int sr = tid / kPer, sk0 = tid - sr * kPer;
    auto atom_of = [&](int t) {
        const int row = (t - ts0) * 16 + sr;
        return t < t1 && row < M ? batom[a0 + row] : -1;  // -1: padding row
    };
    double sv[NV];
    auto load = [&](int src) {
        const double* gr = G + (int64_t)max(src, 0) * ldg;
        int sk = sk0;
        asm volatile("" : "+v"(sk));  // (addresses computed each time: kept over the loop they would spill)
#pragma unroll
        for (int j = 0; j < NV; ++j) sv[j] = gr[min(sk + kPer * j, nin - 1)];
    };
    auto stage = [&](int t, int b, int src) {
        int sk = sk0;
        asm volatile("" : "+v"(sk));
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            const int k = sk + kPer * j;
            ins[(b * 16 + sr) * ldi + k] = src >= 0 ? sinw[k] * (sv[j] + sinw[16 * NI + k]) : 0.0;
        }
        if (sk == 0)
            seed[b * 16 + sr] = src < 0 ? 0.0
                                        : (ROWSEED ? dcdo[bstruct[a0 + (t - ts0) * 16 + sr]] * outw : outw);
    };
    int src = atom_of(t0 + team), next = atom_of(t0 + team + 2);
    load(src);
    {
        const double *iw = Wm + N.inpw_off, *ib = Wm + N.inpb_off;
        for (int k = threadIdx.x; k < 16 * NI; k += 2 * kThreads) {
            sinw[k] = k < nin ? iw[k] : 0.0;
            sinw[16 * NI + k] = k < nin ? ib[k] : 0.0;
        }
    }
    // weights: layer 0's forward operands of this wavefront's columns in registers, layer 1 in LDS for both directions
    // (loads at clamped addresses, so that all are in flight together)
    double f0[KI];
    {
        const double* w = par + N.woff[0] + (int64_t)(on0 ? col : 0) * nin_pad;
#pragma unroll
        for (int q = 0; q < KI; ++q) f0[q] = w[min(4 * q + lk, nin_pad - 1)];
    }
    if constexpr (H == 2) {  // each team half of the K-steps
        const double* w = par + N.woff[1] + (int64_t)(on1 ? col : 0) * w0;
        double f1[KH / 2];
#pragma unroll
        for (int q = 0; q < KH / 2; ++q) f1[q] = w[min(4 * (2 * q + team) + lk, w0 - 1)];
#pragma unroll
        for (int q = 0; q < KH / 2; ++q) {
            const int k = 4 * (2 * q + team) + lk;
            W1[col * ldu + k] = on1 && k < w0 ? f1[q] : 0.0;
        }
    }
#pragma unroll
    for (int q = 0; q < KI; ++q) f0[q] = on0 && 4 * q + lk < nin_pad ? f0[q] : 0.0;
    const double bias0 = on0 ? par[N.boff[0] + col] : 0.0, bias1 = H == 2 && on1 ? par[N.boff[1] + col] : 0.0;
    const double wo = on1 ? par[N.woff[H] + col] : 0.0, bo = par[N.boff[H]];
    d4_t g0[NI], g1[H == 2 ? MH : 1];
#pragma unroll
    for (int m = 0; m < NI; ++m) g0[m] = d4_t{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int m = 0; m < (H == 2 ? MH : 1); ++m) g1[m] = d4_t{0.0, 0.0, 0.0, 0.0};
    double gb0 = 0.0, gb1 = 0.0, gwo = 0.0, gbo = 0.0;
    __syncthreads();
    stage(t0 + team, 0, src);
    __syncthreads();
    const int nt = (t1 - t0 + 1) / 2;  // tiles of a team; with an odd count the second team's last one is all padding
    for (int i = 0; i < nt; ++i) {
        const int t = t0 + team + 2 * i, b = i & 1;
        const double* in = ins + b * 16 * ldi;
        src = next;
        next = atom_of(t + 4);
        load(src);
        int slot = -1;  // where the energy of row `lane` goes
        if (!ROWSEED && wv == team && lane < 16 && t < t1) {
            const int row = (t - ts0) * 16 + lane, at = a0 + min(row, M - 1);
            const int q = bslot[at];
            slot = row < M && batom[at] >= 0 ? q : -1;
        }
        double av[4], d0[4], d1[4], z[4];
        // layer 0
        {
            d4_t acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int q = 0; q < KI; ++q)
                acc = __builtin_amdgcn_mfma_f64_16x16x4f64(in[li * ldi + 4 * q + lk], f0[q], acc, 0, 0, 0);
#pragma unroll
            for (int v = 0; v < 4; ++v) z[v] = acc[v] + bias0;
#pragma unroll
            for (int v = 0; v < 4; ++v) train_act<false>(NEU_TANH, z[v], av[v], d0[v]);
        }
        if constexpr (H == 2) {
#pragma unroll
            for (int v = 0; v < 4; ++v) A0[(4 * v + lk) * ldu + col] = av[v];
            double w[KH / 4];  // a quarter of the weights, read ahead of the barrier
#pragma unroll
            for (int q = 0; q < KH / 4; ++q) w[q] = W1[col * ldu + 4 * q + lk];
            __syncthreads();
            d4_t acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int q = 0; q < KH; ++q)
                acc = __builtin_amdgcn_mfma_f64_16x16x4f64(A0[li * ldu + 4 * q + lk],
                                                           q < KH / 4 ? w[q] : W1[col * ldu + 4 * q + lk], acc, 0, 0, 0);
#pragma unroll
            for (int v = 0; v < 4; ++v) z[v] = acc[v] + bias1;
#pragma unroll
            for (int v = 0; v < 4; ++v) train_act<false>(NEU_TANH, z[v], av[v], d1[v]);
        } else {
#pragma unroll
            for (int v = 0; v < 4; ++v) d1[v] = d0[v];
        }
        // output layer (linear, one unit): energy terms, its gradient, and the first backward step
        double dz[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const double sd = seed[b * 16 + 4 * v + lk];
            const double e = train_unit_part(wo, av[v]);
            if (li == 0) ep[wv * 16 + 4 * v + lk] = e;
            gwo += sd * av[v];
            dz[v] = sd * wo * d1[v];
            gb1 += dz[v];
            if constexpr (H == 2) Z1[(4 * v + lk) * ldu + col] = dz[v];
        }
        stage(t + 2, b ^ 1, src);
        __syncthreads();
        gbo += seed[b * 16 + li];
        if (wv == team && lane < 16) {  // outputs (the teams' on different SIMDs)
            double e = 0.0;
#pragma unroll
            for (int n = 0; n < MH; ++n) e += ep[n * 16 + lane];
            if (slot >= 0) out[slot] = train_out(outb, outw, bo + e);
        }
        if constexpr (H == 2) {
            // layer 1's weight gradient a_0^T dz_1 (rows: layer-0 units), and dz_0 = (dz_1 W_1) .* d_0
#pragma unroll
            for (int m = 0; m < MH; ++m)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    g1[m] = __builtin_amdgcn_mfma_f64_16x16x4f64(A0[(4 * q + lk) * ldu + 16 * m + li], dz[q], g1[m], 0, 0, 0);
            d4_t acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int q = 0; q < KH; ++q)
                acc = __builtin_amdgcn_mfma_f64_16x16x4f64(Z1[li * ldu + 4 * q + lk], W1[(4 * q + lk) * ldu + col], acc, 0, 0, 0);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                dz[v] = acc[v] * d0[v];
                gb0 += dz[v];
            }
        }
        // layer 0's weight gradient ins^T dz_0 (rows: inputs)
#pragma unroll
        for (int m = 0; m < NI; ++m)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                g0[m] = __builtin_amdgcn_mfma_f64_16x16x4f64(in[(4 * q + lk) * ldi + 16 * m + li], dz[q], g0[m], 0, 0, 0);
        __syncthreads();  // the next tile overwrites A0, Z1, ep, and this buffer one tile later
    }
    // the second team's sums added to the first's
    auto each = [&](auto f) {
        int q = 0;
#pragma unroll
        for (int m = 0; m < NI; ++m)
#pragma unroll
            for (int v = 0; v < 4; ++v) g0[m][v] = f(g0[m][v], q++);
        if constexpr (H == 2) {
#pragma unroll
            for (int m = 0; m < MH; ++m)
#pragma unroll
                for (int v = 0; v < 4; ++v) g1[m][v] = f(g1[m][v], q++);
            gb0 = f(gb0, q++);
        }
        gb1 = f(gb1, q++);
        gwo = f(gwo, q++);
        gbo = f(gbo, q++);
    };
    if (team == 1) each([&](double x, int q) { return tsh[q * kThreads + tid] = x; });
    __syncthreads();
    if (team == 1) return;
    each([&](double x, int q) { return x + tsh[q * kThreads + tid]; });
    // the row, in the reference's parameter order
    double* prow = partial + tr.pbase[s] + (int64_t)(g - tr.tile_start[s]) * N.nparams;
    auto quarters = [](double v) {
        v += __shfl_xor(v, 16);
        return v + __shfl_xor(v, 32);
    };
    gwo = quarters(gwo);
    gb1 = quarters(gb1);
    if constexpr (H == 2) {
        gb0 = quarters(gb0);
        if (lk == 0 && col < n0) prow[N.rb[0] + col] = gb0;
        if (lk == 0 && col < n1) prow[N.rb[1] + col] = gb1;
        if (lk == 0 && col < n1) prow[N.rw[2] + col] = gwo;
        double* pw = prow + N.rw[1] + lk * n1 + col;
#pragma unroll
        for (int m = 0; m < MH; ++m)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                if (16 * m + 4 * v + lk < n0 && col < n1) pw[(16 * m + 4 * v) * n1] = g1[m][v];
    } else {
        if (lk == 0 && col < n0) prow[N.rb[0] + col] = gb1;
        if (lk == 0 && col < n0) prow[N.rw[1] + col] = gwo;
    }
    double* pw = prow + N.rw[0] + lk * n0 + col;
#pragma unroll
    for (int m = 0; m < NI; ++m)
#pragma unroll
        for (int v = 0; v < 4; ++v)
            if (16 * m + 4 * v + lk < nin && col < n0) pw[(16 * m + 4 * v) * n0] = g0[m][v];
    if (wv == 0) {  // the output bias: the sum of the seeds (one a row, on every 16 lanes)
        gbo = row16_sum(gbo);
        if (lane == 0) prow[N.rb[H]] = gbo;
    }
}

// Hidden layers (1 or 2), inputs in units of 16 (4, 5, 6 or 8) and units (32 or 64) of k_train_group for a model; false
// where it does not apply.
struct GroupShape {
    int h, ni, u;
};
static bool train_group_shape(const TrainPlan& p, GroupShape& r) {
    r.h = p.net[0].L - 1;
    int in = 0, w = 0;
    if (r.h < 1 || r.h > 2) return false;
    for (int t = 0; t < p.T; ++t) {
        const TrainNet& n = p.net[t];
        if (n.L - 1 != r.h || n.act != NEU_TANH) return false;
        for (int l = 0; l < r.h; ++l) w = std::max(w, n.wpad[l]);
        in = std::max(in, n.nin_pad / 16);
    }
    if (in > (r.h == 2 && w > 32 ? 6 : 8) || w > 64) return false;
    r.ni = in <= 4 ? 4 : (in <= 6 ? in : 8);
    r.u = w <= 32 ? 32 : 64;
    return true;
}

struct GroupArgs {
    int ngroups;
    const TrainPlan* tp;
    const double *Wm, *par;
    TrainTiles tt, tr;
    const int *gtile, *batom, *bslot, *bstruct;
    const double* G;
    int ldg;
    double* out;
    const double* dcdo;
    double* partial;
};
template <int H, int NI, int U, bool RS>
static hipError_t launch_group_t(const GroupArgs& a, hipStream_t st) {
    const size_t lds = 8 * (size_t)tg_lds_elems<H, NI, U>();
    if (lds > 65536) {
        const hipError_t e = hipFuncSetAttribute((const void*)k_train_group<H, NI, U, RS>,
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL((k_train_group<H, NI, U, RS>), dim3(a.ngroups), dim3(8 * U), lds, st, a.tp, a.Wm, a.par, a.tt, a.tr,
                       a.gtile, a.batom, a.bslot, a.bstruct, a.G, a.ldg, a.out, a.dcdo, a.partial);
    return hipGetLastError();
}
template <int H, int U, bool RS>
static hipError_t launch_group_n(int ni, const GroupArgs& a, hipStream_t st) {
    if (ni == 4) return launch_group_t<H, 4, U, RS>(a, st);
    if (ni == 5) return launch_group_t<H, 5, U, RS>(a, st);
    if (ni == 8) {
        if constexpr (H == 1 || U == 32) return launch_group_t<H, 8, U, RS>(a, st);
        return hipErrorInvalidValue;
    }
    return launch_group_t<H, 6, U, RS>(a, st);
}
template <bool RS>
static hipError_t launch_group(const GroupShape& p, const GroupArgs& a, hipStream_t st) {
    if (p.h == 1) return p.u == 32 ? launch_group_n<1, 32, RS>(p.ni, a, st) : launch_group_n<1, 64, RS>(p.ni, a, st);
    return p.u == 32 ? launch_group_n<2, 32, RS>(p.ni, a, st) : launch_group_n<2, 64, RS>(p.ni, a, st);
}

// Force training, one 16-atom tile: the gradient of dcdo out + (dout/dG . V) with respect to the
// parameters (the energy term, and the term through which the forces depend on the network:
// V = dL/d(dout/dG) from the descriptor tangents).  dout/dG . V is the network's tangent output
// for the input tangent inpw .* V, so:
//   forward:  z_l = w_l a_(l-1) + b_l,  a_l = act(z_l),  zt_l = w_l t_(l-1),  t_l = act'(z_l) zt_l
//   reverse:  pz_l = p_l .* act'_l,  qz_l = q_l .* act'_l + p_l .* act''_l .* zt_l,
//             grad b_l = sum qz_l,  grad w_l = pz_l^T t_(l-1) + qz_l^T a_(l-1)  (K = the 16 atoms),
//             p_(l-1) = w_l^T pz_l,  q_(l-1) = w_l^T qz_l,  p_L = outw,  q_L = dcdo outw
// (D2ODZDI::grad, nn.cpp:1799-1890, contracted with V; Cost::grad, nn.cpp:1554-1589).
// LDS: ins and tin [16][nin_pad], then per layer A (a), D (act', then pz), T (t) and H (act'' zt,
// then qz), each [16][wpad_l].
static size_t train_force_lds_bytes(const TrainNet& n) {
    size_t e = 2 * 16 * (size_t)n.nin_pad;
    for (int l = 0; l < n.L; ++l) e += 4 * 16 * (size_t)n.wpad[l];
    return 8 * e;
}

template <bool GEN>
__global__ __launch_bounds__(kTrainThreads) void k_train_force_tile(
    const TrainPlan* __restrict__ tp, const double* __restrict__ Wm, const double* __restrict__ par, TrainTiles tt,
    int tile0, const int* __restrict__ batom, const int* __restrict__ bstruct, const double* __restrict__ G,
    const double* __restrict__ V, int ldg, const double* __restrict__ dcdo, double* __restrict__ partial) {
    extern __shared__ __align__(16) double tsh[];
    const int tile = tile0 + blockIdx.x;
    const int s = train_species(tt, tp->T, tile);
    const TrainNet& N = tp->net[s];
    const int a0 = tt.atom_start[s], M = tt.atom_start[s + 1] - a0;
    const int r0 = (tile - tt.tile_start[s]) * 16;
    const int tid = threadIdx.x, wv = tid / kWave, lane = tid % kWave, li = lane & 15, lk = lane >> 4;
    const int L = N.L;
    double* ins = tsh;
    double* tin = ins + 16 * N.nin_pad;
    double *A[kMaxLayers], *D[kMaxLayers], *T[kMaxLayers], *H[kMaxLayers];
    {
        double* p = tin + 16 * N.nin_pad;
        for (int l = 0; l < L; ++l) {
            const int sz = 16 * N.wpad[l];
            A[l] = p;
            D[l] = p + sz;
            T[l] = p + 2 * sz;
            H[l] = p + 3 * sz;
            p += 4 * sz;
        }
    }
    for (int idx = tid; idx < 16 * N.nin_pad; idx += kTrainThreads) {
        const int r = idx / N.nin_pad, k = idx % N.nin_pad;
        double v = 0.0, t = 0.0;
        if (r0 + r < M && k < N.nin) {
            const int64_t src = (int64_t)batom[a0 + r0 + r] * ldg + k;
            const double w = Wm[N.inpw_off + k];
            v = w * (G[src] + Wm[N.inpb_off + k]);
            t = w * V[src];
        }
        ins[idx] = v;
        tin[idx] = t;
    }
    __syncthreads();
    for (int l = 0; l < L; ++l) {
        const double* prev = l == 0 ? ins : A[l - 1];
        const double* tprev = l == 0 ? tin : T[l - 1];
        const int in_pad = l == 0 ? N.nin_pad : N.wpad[l - 1], wp = N.wpad[l];
        const bool last = l == L - 1;
        const int act = last ? NEU_LINEAR : N.act;
        for (int jt = wv; jt < wp / 16; jt += kTrainWaves) {
            const d4_t az = tile_mm_f64<true>(prev, in_pad, par + N.woff[l], in_pad, in_pad, jt, li, lk);
            const d4_t at = tile_mm_f64<true>(tprev, in_pad, par + N.woff[l], in_pad, in_pad, jt, li, lk);
            const int col = jt * 16 + li;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int idx = (4 * v + lk) * wp + col;
                const double z = az[v] + par[N.boff[l] + col];
                double av, dv;
                train_act<GEN>(act, z, av, dv);
                const double d2 = last ? 0.0 : train_act_d2<GEN>(act, z, av);
                A[l][idx] = av;
                D[l][idx] = dv;
                T[l][idx] = dv * at[v];
                H[l][idx] = d2 * at[v];
            }
        }
        __syncthreads();
    }
    // seeds on the output unit of real rows: p = outw, q = dcdo outw
    {
        const int wp = N.wpad[L - 1];
        for (int idx = tid; idx < 16 * wp; idx += kTrainThreads) {
            const int r = idx / wp, n = idx % wp;
            const double p = (r0 + r < M && n == 0) ? N.outw : 0.0;
            const double q = p != 0.0 ? p * dcdo[bstruct[a0 + r0 + r]] : 0.0;
            const double dv = D[L - 1][idx], hv = H[L - 1][idx];
            D[L - 1][idx] = p * dv;
            H[L - 1][idx] = q * dv + p * hv;
        }
    }
    __syncthreads();
    double* prow = partial + tt.pbase[s] + (int64_t)(tile - tt.tile_start[s]) * N.nparams;
    for (int l = L - 1; l >= 0; --l) {
        const double* aprev = l == 0 ? ins : A[l - 1];
        const double* tprev = l == 0 ? tin : T[l - 1];
        const int wp = N.wpad[l], in_pad = l == 0 ? N.nin_pad : N.wpad[l - 1];
        const int in_real = l == 0 ? N.nin : N.nodes[l - 1], no = N.nodes[l];
        const double* pz = D[l];
        const double* qz = H[l];
        for (int n = tid; n < no; n += kTrainThreads) {
            double g = 0.0;
#pragma unroll
            for (int r = 0; r < 16; ++r) g += qz[r * wp + n];
            prow[N.rb[l] + n] = g;
        }
        const int ntn = wp / 16, ntm = in_pad / 16;
        for (int t = wv; t < ntn * ntm; t += kTrainWaves) {
            const int nt = t / ntm, mt = t % ntm;
            d4_t acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int r = 4 * q + lk;
                acc = __builtin_amdgcn_mfma_f64_16x16x4f64(pz[r * wp + nt * 16 + li], tprev[r * in_pad + mt * 16 + li], acc,
                                                           0, 0, 0);
                acc = __builtin_amdgcn_mfma_f64_16x16x4f64(qz[r * wp + nt * 16 + li], aprev[r * in_pad + mt * 16 + li], acc,
                                                           0, 0, 0);
            }
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int n = nt * 16 + 4 * v + lk, m = mt * 16 + li;
                if (n < no && m < in_real) prow[N.rw[l] + m * no + n] = acc[v];
            }
        }
        if (l > 0) {
            const int wq = N.wpad[l - 1];
            for (int jt = wv; jt < wq / 16; jt += kTrainWaves) {
                const d4_t pm = tile_mm_f64<false>(pz, wp, par + N.woff[l], wq, wp, jt, li, lk);
                const d4_t qm = tile_mm_f64<false>(qz, wp, par + N.woff[l], wq, wp, jt, li, lk);
                const int col = jt * 16 + li;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int idx = (4 * v + lk) * wq + col;
                    const double dv = D[l - 1][idx], hv = H[l - 1][idx];
                    D[l - 1][idx] = pm[v] * dv;
                    H[l - 1][idx] = qm[v] * dv + pm[v] * hv;
                }
            }
        }
        __syncthreads();
    }
}

// Force residuals of one batch structure b (atoms [bstart[b], bstart[b+1]) of the workspace,
// reference forces from training atom fstart[b]): fdiff = (F - F_ref) / N, gF = beta fdiff / N
// (dL/dF of beta/2 |fdiff|^2), f2[b] = sum |fdiff|^2 (fixed-order tree; nnptef.cpp:1163-1166).
__global__ __launch_bounds__(256) void k_train_fresid(const double* __restrict__ F, const double* __restrict__ fref,
                                                      const int* __restrict__ bstart, const int64_t* __restrict__ fstart,
                                                      double beta, double* __restrict__ gF, double* __restrict__ f2) {
    __shared__ double part[256];
    const int b = blockIdx.x, t = threadIdx.x;
    const int o0 = bstart[b], n = bstart[b + 1] - o0;
    const double norm = 1.0 / n;
    double acc = 0.0;
    for (int i = t; i < n; i += 256) {
        const int64_t a = o0 + i, g = fstart[b] + i;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const double fd = (F[3 * a + c] - fref[3 * g + c]) * norm;
            gF[3 * a + c] = beta * norm * fd;
            acc += fd * fd;
        }
    }
    part[t] = acc;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (t < o) part[t] += part[t + o];
        __syncthreads();
    }
    if (t == 0) f2[b] = part[0];
}

// Per batch structure: E = sum of its atoms' outputs (fixed-order tree), dE = (E - E_ref) / N,
// the loss and dcdo (nnpte.cpp:876-916).
__global__ __launch_bounds__(256) void k_train_struct(const double* __restrict__ out, const int* __restrict__ bstart,
                                                      const double* __restrict__ eref_b, int loss, double delta,
                                                      double* __restrict__ dcdo, double* __restrict__ lossv,
                                                      double* __restrict__ dE2) {
    __shared__ double part[256];
    const int b = blockIdx.x, t = threadIdx.x;
    const int o0 = bstart[b], n = bstart[b + 1] - o0, chunk = (n + 255) / 256;
    double acc = 0.0;
    for (int i = o0 + t * chunk; i < o0 + min(n, (t + 1) * chunk); ++i) acc += out[i];
    part[t] = acc;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (t < o) part[t] += part[t + o];
        __syncthreads();
    }
    if (t == 0) {
        const double norm = 1.0 / n;
        const double dE = (part[0] - eref_b[b]) * norm;
        double c = norm, L = 0.0;
        const double deltai = 1.0 / delta, delta2 = delta * delta;
        if (loss == NNP_LOSS_MSE) {
            L = 0.5 * dE * dE;
            c *= dE;
        } else if (loss == NNP_LOSS_MAE) {
            L = fabs(dE);
            c *= (double)((0.0 < dE) - (dE < 0.0));
        } else if (loss == NNP_LOSS_HUBER) {
            const double arg = dE * deltai, sq = sqrt(1.0 + arg * arg);
            L = delta2 * (sq - 1.0);
            c *= dE / sq;
        } else {
            const double arg = dE * deltai, sq = sqrt(1.0 + arg * arg), lg = log(arg + sq);
            L = delta2 * (1.0 - sq + arg * lg);
            c *= lg * delta;
        }
        dcdo[b] = c;
        lossv[b] = L;
        dE2[b] = dE * dE;
    }
}

// Network parameters from the reference's order (x, page-locked host memory read in place: one launch in place of a
// transposition on the host and a copy) to the training buffer, whose padding stays zero.
__global__ __launch_bounds__(256) void k_train_params(const TrainPlan* __restrict__ tp, const int64_t* __restrict__ goff,
                                                      const double* __restrict__ x, double* __restrict__ par) {
    const TrainNet& N = tp->net[blockIdx.y];
    const int p = blockIdx.x * 256 + threadIdx.x;
    if (p >= N.nparams) return;
    const double v = x[goff[blockIdx.y] + p];
    for (int l = 0; l < N.L; ++l) {
        const int nodes = N.nodes[l], in_real = l == 0 ? N.nin : N.nodes[l - 1], in_pad = l == 0 ? N.nin_pad : N.wpad[l - 1];
        const int b = p - N.rb[l], w = p - N.rw[l];
        if (b >= 0 && b < nodes) par[N.boff[l] + b] = v;
        if (w >= 0 && w < in_real * nodes) par[N.woff[l] + (int64_t)(w % nodes) * in_pad + w / nodes] = v;
    }
}

// Gradient rows summed in two fixed-order levels (all rows of a level in parallel):
// level 1: groups of kReduceGroup consecutive tiles of a species, each summed in tile order into
// grp[s][g][p]; level 2: grad[goff_s + p] (+)= the groups in order.
constexpr int kReduceGroup = 32;
__global__ __launch_bounds__(256) void k_train_reduce1(const TrainPlan* __restrict__ tp, TrainTiles tt, int tile0,
                                                       int tile1, const double* __restrict__ partial, int gmax,
                                                       int64_t gstride, double* __restrict__ grp,
                                                       const int* __restrict__ tstruct, const double* __restrict__ dcdo) {
    const int s = blockIdx.z, g = blockIdx.y;
    const TrainNet& N = tp->net[s];
    const int p = blockIdx.x * 256 + threadIdx.x;
    if (p >= N.nparams || g >= gmax) return;
    const int t0 = max(tile0, tt.tile_start[s]), t1 = min(tile1, tt.tile_start[s + 1]);
    const int a = t0 + g * kReduceGroup, b = min(t1, a + kReduceGroup);
    double acc = 0.0;
    if (tstruct) {  // rows of single-structure tiles, weighted by their structure's dcdo
#pragma unroll 8
        for (int t = a; t < b; ++t)
            acc += dcdo[tstruct[t]] * partial[tt.pbase[s] + (int64_t)(t - tt.tile_start[s]) * N.nparams + p];
    } else {
#pragma unroll 8
        for (int t = a; t < b; ++t) acc += partial[tt.pbase[s] + (int64_t)(t - tt.tile_start[s]) * N.nparams + p];
    }
    grp[(int64_t)s * gstride + (int64_t)g * N.nparams + p] = acc;
}
__global__ __launch_bounds__(256) void k_train_reduce2(const TrainPlan* __restrict__ tp, TrainTiles tt, int tile0,
                                                       int tile1, const double* __restrict__ grp, int64_t gstride,
                                                       const int64_t* __restrict__ goff, double* __restrict__ grad,
                                                       int accumulate) {
    const int s = blockIdx.y;
    const TrainNet& N = tp->net[s];
    const int p = blockIdx.x * 256 + threadIdx.x;
    if (p >= N.nparams) return;
    const int t0 = max(tile0, tt.tile_start[s]), t1 = min(tile1, tt.tile_start[s + 1]);
    const int ng = t1 > t0 ? (t1 - t0 + kReduceGroup - 1) / kReduceGroup : 0;
    double acc = accumulate ? grad[goff[s] + p] : 0.0;
    for (int g = 0; g < ng; ++g) acc += grp[(int64_t)s * gstride + (int64_t)g * N.nparams + p];
    grad[goff[s] + p] = acc;
}

// ------------------------------------------------------------------ host side
template <int MODE>
static void launch_tile(bool gen, dim3 grid, size_t lds, hipStream_t st, const TrainPlan* tp, const double* Wm,
                        const double* par, const TrainTiles& tt, int tile0, const int* batom, const int* bslot,
                        const int* bstruct, const double* G, int ldg, double* out, const double* dcdo, double* partial,
                        double* Y) {
    if (gen)
        hipLaunchKernelGGL((k_train_tile<MODE, true>), grid, dim3(kTrainThreads), lds, st, tp, Wm, par, tt, tile0, batom,
                           bslot, bstruct, G, ldg, out, dcdo, partial, Y);
    else
        hipLaunchKernelGGL((k_train_tile<MODE, false>), grid, dim3(kTrainThreads), lds, st, tp, Wm, par, tt, tile0, batom,
                           bslot, bstruct, G, ldg, out, dcdo, partial, Y);
}

class TrainSet {
  public:
    TrainSet(Engine& owner, int n, const nnp_structure* ss, const double* energy) : owner_(owner) {
        if (n <= 0 || !ss || !energy) throw std::invalid_argument("nnp_train_create: invalid argument");
        const HostModel& hm = owner.host;
        const DevPlan& P = owner.pb.plan;
        T_ = hm.T;
        ldg_ = P.ldg;
        // network layout
        std::memset(&plan_, 0, sizeof(plan_));
        plan_.T = T_;
        int64_t pofs = 0;
        goff_.assign(T_ + 1, 0);
        for (int t = 0; t < T_; ++t) {
            const NetSpec& ns = hm.sp[t].net;
            const DevNet& dn = P.net[t];
            TrainNet& N = plan_.net[t];
            N.L = dn.L;
            N.nin = ns.nin;
            N.nin_pad = dn.nin_pad;
            N.act = dn.act;
            N.inpw_off = dn.inpw_off;
            N.inpb_off = dn.inpb_off;
            N.outw = dn.outw;
            N.outb = dn.outb;
            gen_ = gen_ || (N.L > 1 && N.act != NEU_TANH && N.act != NEU_LINEAR);
            if (ns.nodes.back() != 1) throw unsupported_error("nnp_train: networks with more than one output");
            int rb = 0, nb = 0;
            for (int l = 0; l < N.L; ++l) nb += ns.nodes[l];
            int rw = nb;
            for (int l = 0; l < N.L; ++l) {
                const int in_pad = l == 0 ? N.nin_pad : dn.wpad[l - 1];
                const int in_real = l == 0 ? ns.nin : ns.nodes[l - 1];
                N.nodes[l] = ns.nodes[l];
                N.wpad[l] = dn.wpad[l];
                N.woff[l] = pofs;
                pofs += (int64_t)dn.wpad[l] * in_pad;
                N.boff[l] = pofs;
                pofs += dn.wpad[l];
                pofs = (pofs + 1) & ~int64_t(1);
                N.rb[l] = rb;
                rb += ns.nodes[l];
                N.rw[l] = rw;
                rw += ns.nodes[l] * in_real;
            }
            N.nparams = rw;
            goff_[t + 1] = goff_[t] + N.nparams;
        }
        npar_dev_ = pofs;
        // parameter, gradient and staging memory (sizes known here, so that no pass allocates it); padding weights are zero
        d_par_.reserve(8 * (size_t)npar_dev_);
        d_res_.reserve(8 * (size_t)(total() + 3 * n));
        h_io_.reserve(8 * (size_t)(2 * total() + 3 * n));
        HIPCHK(hipMemcpy(d_par_.p, std::vector<double>(npar_dev_, 0.0).data(), 8 * (size_t)npar_dev_, hipMemcpyHostToDevice));
        d_plan_.reserve(sizeof(TrainPlan));
        HIPCHK(hipMemcpy(d_plan_.p, &plan_, sizeof(TrainPlan), hipMemcpyHostToDevice));
        d_goff_.reserve(sizeof(int64_t) * (T_ + 1));
        HIPCHK(hipMemcpy(d_goff_.p, goff_.data(), sizeof(int64_t) * (T_ + 1), hipMemcpyHostToDevice));
        // descriptors of the training set, computed once in chunks by a workspace of the model
        natoms_.resize(n);
        aoff_.assign(n + 1, 0);
        for (int k = 0; k < n; ++k) {
            if (ss[k].natoms <= 0) throw std::invalid_argument("nnp_train_create: empty structure");
            natoms_[k] = ss[k].natoms;
            aoff_[k + 1] = aoff_[k] + ss[k].natoms;
            for (int i = 0; i < ss[k].natoms; ++i) types_.push_back(ss[k].type[i]);
            if (!ss[k].pos || !ss[k].type) throw std::invalid_argument("nnp_train_create: null structure arrays");
            hpos_.insert(hpos_.end(), ss[k].pos, ss[k].pos + 3 * (size_t)ss[k].natoms);
            hopen_.push_back(ss[k].cell ? 0 : 1);
            for (int q = 0; q < 9; ++q) hcell_.push_back(ss[k].cell ? ss[k].cell[q] : 0.0);
        }
        eref_.assign(energy, energy + n);
        ntot_ = aoff_[n];
        d_G_.reserve((size_t)ntot_ * ldg_ * 8);
        Engine E(owner, 1000);
        int k0 = 0;
        while (k0 < n) {
            int k1 = k0;
            int64_t atoms = 0;
            while (k1 < n && (k1 == k0 || atoms + natoms_[k1] <= (1 << 18))) atoms += natoms_[k1++];
            std::vector<nnp_structure> chunk(ss + k0, ss + k1);
            E.upload(chunk);
            E.build_neighbors(false);
            E.descriptors<double>();
            HIPCHK(hipMemcpyAsync((double*)d_G_.p + (size_t)aoff_[k0] * ldg_, E.d_G.p, (size_t)atoms * ldg_ * 8,
                                  hipMemcpyDeviceToDevice, E.stream));
            HIPCHK(hipStreamSynchronize(E.stream));
            k0 = k1;
        }
        HIPCHK(hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking));
    }
    ~TrainSet() {
        if (stream_) (void)hipStreamSynchronize(stream_);
        if (ws_) (void)hipStreamSynchronize(ws_->stream);
        for (DevMem* m : {&d_plan_, &d_goff_, &d_G_, &d_par_, &d_out_, &d_dcdo_, &d_res_, &d_partial_, &d_grp_, &d_fref_,
                          &d_gF_, &d_V_, &d_tstruct_, &d_gtile_})
            m->release();
        h_io_.release();
        if (stream_) (void)hipStreamDestroy(stream_);
    }

    int64_t nparams(int t) const {
        if (t < 0 || t >= T_) throw std::invalid_argument("nnp_train_nparams: species out of range");
        return plan_.net[t].nparams;
    }
    int64_t total() const { return goff_[T_]; }

    // the model's current parameters in the reference order (operator>>)
    void get_params(double* x) const {
        for (int t = 0; t < T_; ++t) {
            const NetSpec& ns = owner_.host.sp[t].net;
            const TrainNet& N = plan_.net[t];
            double* y = x + goff_[t];
            for (int l = 0; l < N.L; ++l)
                for (int n = 0; n < N.nodes[l]; ++n) y[N.rb[l] + n] = ns.b[l][n];
            for (int l = 0; l < N.L; ++l) {
                const int in_real = l == 0 ? ns.nin : ns.nodes[l - 1];
                for (int m = 0; m < in_real; ++m)
                    for (int n = 0; n < N.nodes[l]; ++n) y[N.rw[l] + m * N.nodes[l] + n] = ns.W[l][(size_t)n * in_real + m];
            }
        }
    }

    struct Tiles {
        TrainTiles tt;
        int tiles = 0;
        int64_t pb = 0;  // partial elements of all tiles
    };

    // Groups of consecutive tiles of k_train_group: within each run of tiles (one structure's atoms of a species, or
    // with no struct_t a species), at most `gsize` tiles, gsize the smallest even number (a tile for each
    // team) that gives at most one group per CU (the kernel's residency, so one round) up to 32 tiles.  The groups'
    // rows take the tiles' places in `rows`.
    struct Groups {
        TrainTiles rows;  // group ranges of the species and their row bases
        int n = 0;
        int64_t pb = 0;
        std::vector<int> first;    // first tile of each group, then the tile count
        std::vector<int> structs;  // structure of each group (struct_t given)
    };
    Groups make_groups(const Tiles& tl, const std::vector<int>* struct_t) const {
        Groups r;
        const auto build = [&](int gsize) {
            std::memset(&r.rows, 0, sizeof(r.rows));
            r.first.clear();
            r.structs.clear();
            r.pb = 0;
            for (int t = 0; t <= kMaxSpecies; ++t) {
                r.rows.tile_start[t] = (int)r.first.size();
                r.rows.pbase[t] = r.pb;
                if (t >= T_) continue;
                for (int k = tl.tt.tile_start[t]; k < tl.tt.tile_start[t + 1];) {
                    int e = k + 1;
                    while (e < tl.tt.tile_start[t + 1] && e - k < gsize && (!struct_t || (*struct_t)[e] == (*struct_t)[k])) ++e;
                    r.first.push_back(k);
                    if (struct_t) r.structs.push_back((*struct_t)[k]);
                    r.pb += plan_.net[t].nparams;
                    k = e;
                }
            }
            r.n = (int)r.first.size();
        };
        for (int gsize = 2 * std::max(1, std::min(16, tl.tiles / (2 * owner_.num_cus))); gsize <= 32; gsize += 2) {
            build(gsize);
            if (r.n <= owner_.num_cus) break;
        }
        r.first.push_back(tl.tiles);
        return r;
    }

    void check_args(const char* fn, const double* x, int nbatch, const int* batch, int loss, double delta,
                    const double* err) const {
        if (!x || !err || nbatch <= 0 || !batch) throw std::invalid_argument(std::string(fn) + ": invalid argument");
        if (loss < NNP_LOSS_MSE || loss > NNP_LOSS_ASINH) throw std::invalid_argument(std::string(fn) + ": unknown loss");
        if ((loss == NNP_LOSS_HUBER || loss == NNP_LOSS_ASINH) && !(delta > 0))
            throw std::invalid_argument(std::string(fn) + ": delta must be positive");
        const int nst = (int)natoms_.size();
        for (int b = 0; b < nbatch; ++b)
            if (batch[b] < 0 || batch[b] >= nst) throw std::invalid_argument(std::string(fn) + ": structure out of range");
    }

    // Parameters from the reference's order to padded row-major layers, on stream st.
    // Staging of one call: [x, total][results: gradient, then three values a structure].  One kernel reads x in place and
    // one copy brings every result; with the parameters transposed on the host, four to fifteen pageable copies, and
    // the tiles and reference values of a chunk sent again on each call, a call waited more than it computed: 194 us
    // for 16 x 2048 atoms and 310 us for the force training of 24 structures of up to 700, now 121 and 180 us.
    void pack_params(const double* x, int nbatch, hipStream_t st) {
        h_io_.reserve(8 * (size_t)(2 * total() + 3 * (int64_t)nbatch));
        d_res_.reserve(8 * (size_t)(total() + 3 * (int64_t)nbatch));
        grad_started_ = false;
        std::memcpy(h_io_.p, x, 8 * (size_t)total());
        int maxnp = 1;
        for (int t = 0; t < T_; ++t) maxnp = std::max(maxnp, plan_.net[t].nparams);
        hipLaunchKernelGGL(k_train_params, dim3((maxnp + 255) / 256, T_), dim3(256), 0, st, (const TrainPlan*)d_plan_.p,
                           (const int64_t*)d_goff_.p, (const double*)h_io_.p, (double*)d_par_.p);
        HIPCHK(hipGetLastError());
    }
    // Values q (0: losses, 1: squared energy residuals, 2: squared force residuals) of the call's structures.
    double* res(int q, int nbatch) const { return (double*)d_res_.p + total() + (int64_t)q * nbatch; }
    // The results in host memory: the gradient at [0], res(q) at [total + q nbatch].
    const double* fetch_results(int nbatch, int nq, double* grad, hipStream_t st) {
        const int64_t o = grad ? 0 : total(), n = total() + (int64_t)nq * nbatch - o;
        double* h = (double*)h_io_.p + total();
        if (grad && !grad_started_) HIPCHK(hipMemsetAsync(d_res_.p, 0, 8 * (size_t)total(), st));
        HIPCHK(hipMemcpyAsync(h + o, (const double*)d_res_.p + o, 8 * (size_t)n, hipMemcpyDeviceToHost, st));
        HIPCHK(hipStreamSynchronize(st));
        if (grad) std::memcpy(grad, h, 8 * (size_t)total());
        return h + total();
    }
    // A call that ends by an exception leaves nothing in flight on its stream (the staging memory is written again
    // by the next call).
    struct Settle {
        hipStream_t st;
        ~Settle() {
            if (std::uncaught_exceptions() > 0) (void)hipStreamSynchronize(st);
        }
    };

    // What a batch's tiles read: atoms, slots and structures by species, first slots, reference energies, first
    // reference force of each structure (force training).
    struct TileArrays {
        DevMem atom, slot, strct, bstart, eref, fstart;
        TileArrays() = default;
        TileArrays(const TileArrays&) = delete;
        ~TileArrays() {
            for (DevMem* m : {&atom, &slot, &strct, &bstart, &eref, &fstart}) m->release();
        }
    };
    // Force training's state of a chunk of structures: workspace and tiles.
    struct Chunk {
        std::vector<int> key;
        std::unique_ptr<Engine> own;  // null: the scratch workspace
        Tiles tl;
        TileArrays ta;
        bool settled = false;  // its rows' reaction tables are known to miss nothing
    };

    // Species tiles of 16 atoms over the given (source row, slot, structure) lists per species,
    // uploaded into ta's tables on stream st.
    Tiles make_tiles(const std::vector<std::vector<int>>& atom_s, const std::vector<std::vector<int>>& slot_s,
                     const std::vector<std::vector<int>>& struct_s, hipStream_t st, TileArrays& ta) {
        Tiles r;
        std::memset(&r.tt, 0, sizeof(r.tt));
        hbatom_.clear();
        hbslot_.clear();
        hbstruct_.clear();
        for (int t = 0; t <= kMaxSpecies; ++t) {
            r.tt.tile_start[t] = r.tiles;
            r.tt.atom_start[t] = (int)hbatom_.size();
            r.tt.pbase[t] = r.pb;
            if (t < T_) {
                hbatom_.insert(hbatom_.end(), atom_s[t].begin(), atom_s[t].end());
                hbslot_.insert(hbslot_.end(), slot_s[t].begin(), slot_s[t].end());
                hbstruct_.insert(hbstruct_.end(), struct_s[t].begin(), struct_s[t].end());
                const int nt = ((int)atom_s[t].size() + 15) / 16;
                r.tiles += nt;
                r.pb += (int64_t)nt * plan_.net[t].nparams;
            }
        }
        const size_t nba = std::max<size_t>(hbatom_.size(), 1);
        ta.atom.reserve(4 * nba);
        ta.slot.reserve(4 * nba);
        ta.strct.reserve(4 * nba);
        HIPCHK(hipMemcpyAsync(ta.atom.p, hbatom_.data(), 4 * hbatom_.size(), hipMemcpyHostToDevice, st));
        HIPCHK(hipMemcpyAsync(ta.slot.p, hbslot_.data(), 4 * hbslot_.size(), hipMemcpyHostToDevice, st));
        HIPCHK(hipMemcpyAsync(ta.strct.p, hbstruct_.data(), 4 * hbstruct_.size(), hipMemcpyHostToDevice, st));
        return r;
    }

    // Gradient rows of every tile, in chunks of tiles (at most the model's train_chunk_elems row
    // elements at a time, 2^28 = 2 GB by default):
    // launch(tc, c0, c1) writes the rows of tiles [c0, c1) at the shifted bases of tc; the rows are
    // then added into the gradient in a fixed order (groups of consecutive tiles, then the groups).
    template <typename F>
    void sum_tiles(const Tiles& tl, hipStream_t st, F&& launch) {
        if (tl.tiles == 0) return;
        int64_t maxnp = 1;
        for (int t = 0; t < T_; ++t) maxnp = std::max<int64_t>(maxnp, plan_.net[t].nparams);
        const int chunk = (int)std::max<int64_t>(
            1, std::min<int64_t>({(int64_t)tl.tiles, owner_.train_chunk_elems / maxnp, (int64_t)kReduceGroup * 65535}));
        d_partial_.reserve(8 * (size_t)std::min<int64_t>(tl.pb, (int64_t)chunk * maxnp + maxnp));
        for (int c0 = 0; c0 < tl.tiles; c0 += chunk) {
            const int c1 = std::min(tl.tiles, c0 + chunk);
            // partial rows of this chunk start at element 0: shift each species' base
            TrainTiles tc = tl.tt;
            int64_t base = 0;
            for (int t = 0; t < T_; ++t) {
                const int t0 = std::max(c0, tl.tt.tile_start[t]), t1 = std::min(c1, tl.tt.tile_start[t + 1]);
                tc.pbase[t] = base - (int64_t)(t0 - tl.tt.tile_start[t]) * plan_.net[t].nparams;
                if (t1 > t0) base += (int64_t)(t1 - t0) * plan_.net[t].nparams;
            }
            launch(tc, c0, c1);
            HIPCHK(hipGetLastError());
            reduce_rows(tc, c0, c1, st, nullptr, nullptr);
        }
    }

    // The gradient (d_res_; set by a call's first rows) += the rows of tiles [c0, c1) (bases tc), optionally weighted by
    // dcdo[tstruct[tile]].
    void reduce_rows(const TrainTiles& tc, int c0, int c1, hipStream_t st, const int* tstruct,
                     const double* dcdo) {
        if (c1 <= c0) return;
        int64_t maxnp = 1;
        for (int t = 0; t < T_; ++t) maxnp = std::max<int64_t>(maxnp, plan_.net[t].nparams);
        const int gmax = (c1 - c0 + kReduceGroup - 1) / kReduceGroup;
        if (gmax > 65535) throw std::invalid_argument("nnp_train: too many tiles in one reduction");
        const int64_t gstride = (int64_t)gmax * maxnp;
        d_grp_.reserve(8 * (size_t)(T_ * gstride));
        const unsigned pblocks = (unsigned)((maxnp + 255) / 256);
        hipLaunchKernelGGL(k_train_reduce1, dim3(pblocks, gmax, T_), dim3(256), 0, st, (const TrainPlan*)d_plan_.p, tc, c0,
                           c1, (const double*)d_partial_.p, gmax, gstride, (double*)d_grp_.p, tstruct, dcdo);
        hipLaunchKernelGGL(k_train_reduce2, dim3(pblocks, T_), dim3(256), 0, st, (const TrainPlan*)d_plan_.p, tc, c0, c1,
                           (const double*)d_grp_.p, gstride, (const int64_t*)d_goff_.p, (double*)d_res_.p, grad_started_ ? 1 : 0);
        HIPCHK(hipGetLastError());
        grad_started_ = true;
    }

    // A tile kernel's dynamic LDS within the device's per-workgroup limit (above 64 KiB the kernel
    // is allowed the larger allocation first).
    void check_lds(size_t lds, const void* fn) {
        if (lds_limit_ == 0) {
            int dev = 0, v = 0;
            HIPCHK(hipGetDevice(&dev));
            HIPCHK(hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
            lds_limit_ = v > 0 ? (size_t)v : 65536;
        }
        if (lds > lds_limit_) throw unsupported_error("nnp_train: network too wide for the training kernels' LDS");
        if (lds > 65536) HIPCHK(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    }

    // Reference forces of every training atom (3 per atom, structures in creation order).
    void set_forces(const double* f) {
        if (!f) throw std::invalid_argument("nnp_train_set_forces: null argument");
        d_fref_.reserve(8 * 3 * (size_t)ntot_);
        HIPCHK(hipMemcpy(d_fref_.p, f, 8 * 3 * (size_t)ntot_, hipMemcpyHostToDevice));
        has_forces_ = true;
    }

    void error(const double* x, int nbatch, const int* batch, int loss, double delta, double* err, double* grad) {
        check_args("nnp_train_error", x, nbatch, batch, loss, delta, err);
        const Settle settle{stream_};
        pack_params(x, nbatch, stream_);
        int64_t maxnp = 1;
        for (int t = 0; t < T_; ++t) maxnp = std::max<int64_t>(maxnp, plan_.net[t].nparams);
        // Tiles: with the gradient, single-structure tiles (each structure's atoms of a species
        // padded to whole tiles) when that adds few tiles and every row fits in one buffer, so one
        // forward + backward pass per tile gives the outputs and the gradient rows of the outputs,
        // which the reduction weights by dcdo; otherwise species tiles across structures, a forward
        // pass for the energies and a second pass with the loss seeds.  The tiles of the previous
        // call are reused when the batch, mode and row buffer repeat.
        const int mode = grad ? (owner_.train_one_pass ? 2 : 1) : 0;
        std::vector<int> key(batch, batch + nbatch);
        key.push_back(mode);
        // (the rows that one buffer holds decide between the forms below)
        key.push_back((int)(owner_.train_chunk_elems >> 32));
        key.push_back((int)(owner_.train_chunk_elems & 0xffffffff));
        if (key != tiles_key_) {
            tiles_key_.clear();
            std::vector<int> bstart(nbatch + 1, 0);
            for (int b = 0; b < nbatch; ++b) bstart[b + 1] = bstart[b] + natoms_[batch[b]];
            std::vector<std::vector<int>> atom_s(T_), slot_s(T_), struct_s(T_);
            for (int b = 0; b < nbatch; ++b) {
                const int st = batch[b];
                for (int i = 0; i < natoms_[st]; ++i) {
                    const int g = (int)aoff_[st] + i, t = types_[g];
                    atom_s[t].push_back(g);
                    slot_s[t].push_back(bstart[b] + i);
                    struct_s[t].push_back(b);
                }
            }
            one_pass_ = false;
            if (grad) {
                int64_t tm = 0, th = 0;
                for (int t = 0; t < T_; ++t) {
                    tm += ((int64_t)atom_s[t].size() + 15) / 16;
                    for (size_t k = 0; k < atom_s[t].size();) {  // runs of one structure
                        size_t e = k;
                        while (e < atom_s[t].size() && struct_s[t][e] == struct_s[t][k]) ++e;
                        th += ((int64_t)(e - k) + 15) / 16;
                        k = e;
                    }
                }
                one_pass_ = mode == 2 && th <= tm + tm / 8 + 8 && th * maxnp <= owner_.train_chunk_elems;
            }
            if (one_pass_) {
                // pad each (structure, species) run to whole tiles with rows marked -1
                for (int t = 0; t < T_; ++t) {
                    std::vector<int> pa, ps, pst;
                    for (size_t k = 0; k < atom_s[t].size();) {
                        size_t e = k;
                        while (e < atom_s[t].size() && struct_s[t][e] == struct_s[t][k]) ++e;
                        for (size_t q = k; q < e; ++q) {
                            pa.push_back(atom_s[t][q]);
                            ps.push_back(slot_s[t][q]);
                            pst.push_back(struct_s[t][q]);
                        }
                        while (pa.size() % 16) {
                            pa.push_back(-1);
                            ps.push_back(0);
                            pst.push_back(struct_s[t][k]);
                        }
                        k = e;
                    }
                    atom_s[t].swap(pa);
                    slot_s[t].swap(ps);
                    struct_s[t].swap(pst);
                }
            }
            tiles_ = make_tiles(atom_s, slot_s, struct_s, stream_, ta_);
            std::vector<int> ts;
            if (one_pass_)
                for (int t = 0; t < T_; ++t)
                    for (size_t k = 0; k < struct_s[t].size(); k += 16) ts.push_back(struct_s[t][k]);
            grouped_ = grad && tiles_.tiles > 0 && train_group_shape(plan_, gshape_);
            if (grouped_) {
                groups_ = make_groups(tiles_, one_pass_ ? &ts : nullptr);
                // rows beyond one buffer: tile by tile, in chunks
                grouped_ = (int64_t)groups_.n * maxnp <= owner_.train_chunk_elems;
            }
            if (grouped_) {
                ts = groups_.structs;
                d_gtile_.reserve(4 * groups_.first.size());
                HIPCHK(hipMemcpyAsync(d_gtile_.p, groups_.first.data(), 4 * groups_.first.size(), hipMemcpyHostToDevice,
                                      stream_));
            }
            if (one_pass_) {
                d_tstruct_.reserve(4 * std::max<size_t>(ts.size(), 1));
                HIPCHK(hipMemcpyAsync(d_tstruct_.p, ts.data(), 4 * ts.size(), hipMemcpyHostToDevice, stream_));
            }
            std::vector<double> eb(nbatch);
            for (int b = 0; b < nbatch; ++b) eb[b] = eref_[batch[b]];
            ta_.eref.reserve(8 * (size_t)nbatch);
            HIPCHK(hipMemcpyAsync(ta_.eref.p, eb.data(), 8 * (size_t)nbatch, hipMemcpyHostToDevice, stream_));
            ta_.bstart.reserve(4 * (size_t)(nbatch + 1));
            natoms_batch_ = bstart[nbatch];
            HIPCHK(hipMemcpyAsync(ta_.bstart.p, bstart.data(), 4 * (size_t)(nbatch + 1), hipMemcpyHostToDevice, stream_));
            HIPCHK(hipStreamSynchronize(stream_));  // the host vectors above go out of scope
            tiles_key_ = key;
        }
        const Tiles& tl = tiles_;
        d_out_.reserve(8 * (size_t)std::max(natoms_batch_, 1));
        d_dcdo_.reserve(8 * (size_t)nbatch);
        size_t lds = 0;
        for (int t = 0; t < T_; ++t) lds = std::max(lds, train_lds_bytes(plan_.net[t]));
        for (int md = 0; md < 4; md += (md == 1 ? 2 : 1)) {  // modes 0, 1, 3
            const void* fn = md == 0 ? (gen_ ? (const void*)k_train_tile<0, true> : (const void*)k_train_tile<0, false>)
                             : md == 1 ? (gen_ ? (const void*)k_train_tile<1, true> : (const void*)k_train_tile<1, false>)
                                       : (gen_ ? (const void*)k_train_tile<3, true> : (const void*)k_train_tile<3, false>);
            check_lds(lds, fn);
        }
        const double* Wm = (const double*)owner_.d_w64.p;
        const TrainPlan* tpp = (const TrainPlan*)d_plan_.p;
        const double* par = (const double*)d_par_.p;
        const int *ba = (const int*)ta_.atom.p, *bsl = (const int*)ta_.slot.p, *bst = (const int*)ta_.strct.p;
        const double* Gp = (const double*)d_G_.p;
        GroupArgs ga{};
        if (grouped_) {
            d_partial_.reserve(8 * (size_t)groups_.pb);
            ga = GroupArgs{groups_.n, tpp, Wm,   par,  tl.tt,  groups_.rows, (const int*)d_gtile_.p,         ba,
                           bsl,       bst, Gp,   ldg_, (double*)d_out_.p,    (const double*)d_dcdo_.p,       (double*)d_partial_.p};
        }
        if (one_pass_ && grouped_) {
            HIPCHK(launch_group<false>(gshape_, ga, stream_));
        } else if (one_pass_) {
            d_partial_.reserve(8 * (size_t)std::max<int64_t>(tl.pb, 1));
            if (tl.tiles > 0)
                launch_tile<3>(gen_, dim3(tl.tiles), lds, stream_, tpp, Wm, par, tl.tt, 0, ba, bsl, bst, Gp, ldg_,
                               (double*)d_out_.p, nullptr, (double*)d_partial_.p, nullptr);
        } else if (tl.tiles > 0) {
            launch_tile<0>(gen_, dim3(tl.tiles), lds, stream_, tpp, Wm, par, tl.tt, 0, ba, bsl, bst, Gp, ldg_,
                           (double*)d_out_.p, nullptr, nullptr, nullptr);
        }
        hipLaunchKernelGGL(k_train_struct, dim3(nbatch), dim3(256), 0, stream_, (const double*)d_out_.p,
                           (const int*)ta_.bstart.p, (const double*)ta_.eref.p, loss, delta, (double*)d_dcdo_.p,
                           res(0, nbatch), res(1, nbatch));
        HIPCHK(hipGetLastError());
        if (grad) {
            if (grouped_) {
                if (!one_pass_) HIPCHK(launch_group<true>(gshape_, ga, stream_));
                reduce_rows(groups_.rows, 0, groups_.n, stream_, one_pass_ ? (const int*)d_tstruct_.p : nullptr,
                            (const double*)d_dcdo_.p);
            } else if (one_pass_) {
                reduce_rows(tl.tt, 0, tl.tiles, stream_, (const int*)d_tstruct_.p, (const double*)d_dcdo_.p);
            } else {
                sum_tiles(tl, stream_, [&](const TrainTiles& tc, int c0, int c1) {
                    launch_tile<1>(gen_, dim3(c1 - c0), lds, stream_, tpp, Wm, par, tc, c0, ba, bsl, bst, Gp, ldg_,
                                   nullptr, (const double*)d_dcdo_.p, (double*)d_partial_.p, nullptr);
                });
            }
        }
        const double* lv = fetch_results(nbatch, 2, grad, stream_);
        const double* e2 = lv + nbatch;
        err[0] = err[1] = 0.0;
        for (int b = 0; b < nbatch; ++b) {
            err[0] += lv[b];
            err[1] += e2[b];
        }
    }

    // Energy + force loss and its gradient (the training part of NNPTEF::error, nnptef.cpp:1040-1293,
    // with the exact derivative of the force term).  Per chunk of batch structures a workspace of the
    // model builds the neighbour list and descriptors; the networks at x give the atomic outputs and
    // dout/dG; the model's force kernels turn those into forces; the force residuals give gF = dL/dF,
    // the descriptor tangents V = dL/d(dout/dG), and the tile kernel the gradient.
    void error_force(const double* x, int nbatch, const int* batch, int loss, double delta, double beta, uint32_t flags,
                     double* err, double* grad) {
        check_args("nnp_train_error_force", x, nbatch, batch, loss, delta, err);
        if (!has_forces_) throw std::invalid_argument("nnp_train_error_force: reference forces not set");
        if (!(beta >= 0)) throw std::invalid_argument("nnp_train_error_force: beta must be non-negative");
        if (!ws_) ws_ = std::make_unique<Engine>(owner_, 1001);
        const hipStream_t st = ws_->stream;  // every chunk's work is ordered on this stream
        const bool all_images = flags & NNP_ALL_IMAGES;
        const Settle settle{st};
        pack_params(x, nbatch, st);
        size_t lds = 0, flds = 0;
        for (int t = 0; t < T_; ++t) {
            lds = std::max(lds, train_lds_bytes(plan_.net[t]));
            flds = std::max(flds, train_force_lds_bytes(plan_.net[t]));
        }
        check_lds(lds, gen_ ? (const void*)k_train_tile<2, true> : (const void*)k_train_tile<2, false>);
        if (grad) check_lds(flds, gen_ ? (const void*)k_train_force_tile<true> : (const void*)k_train_force_tile<false>);
        const double* Wm = (const double*)owner_.d_w64.p;
        int k0 = 0;
        while (k0 < nbatch) {
            // a chunk of whole structures, at most ~128k atoms (one structure if larger)
            int k1 = k0;
            int64_t atoms = 0;
            while (k1 < nbatch && (k1 == k0 || atoms + natoms_[batch[k1]] <= (1 << 17))) atoms += natoms_[batch[k1++]];
            const int nb = k1 - k0, n = (int)atoms;
            // The structures do not move between calls: a chunk seen before keeps its neighbour
            // rows, descriptors and tiles in a workspace of its own (up to the model's train_cache_atoms
            // option in all, 2^20 by default);
            // otherwise the scratch workspace builds them.
            std::vector<int> key(batch + k0, batch + k1);
            key.push_back(all_images ? 1 : 0);
            Chunk* C = nullptr;
            for (auto& c : fcache_)
                if (c->key == key) C = c.get();
            if (!C) {
                HIPCHK(hipStreamSynchronize(st));  // (the scratch workspace's last chunk)
                auto fresh = std::make_unique<Chunk>();
                const bool keep = fcache_atoms_ + atoms <= owner_.train_cache_atoms;
                if (keep) fresh->own = std::make_unique<Engine>(owner_, 1002);
                build_chunk(*fresh, batch + k0, nb, all_images, keep ? *fresh->own : *ws_, st);
                if (keep) {
                    fresh->key = key;
                    fcache_.push_back(std::move(fresh));
                    fcache_atoms_ += atoms;
                    C = fcache_.back().get();
                } else {
                    scratch_ = std::move(fresh);
                    C = scratch_.get();
                }
            }
            Engine& E = C->own ? *C->own : *ws_;
            const Tiles& tl = C->tl;
            const TileArrays& ta = C->ta;
            // the chunk's kernels, the workspace's force kernels included, run in order on st
            struct OnStream {
                Engine& e;
                hipStream_t own;
                OnStream(Engine& w, hipStream_t s) : e(w), own(w.stream) { e.stream = s; }
                ~OnStream() { e.stream = own; }
            } on_stream(E, st);
            d_out_.reserve(8 * (size_t)n);
            d_dcdo_.reserve(8 * (size_t)nb);
            d_gF_.reserve(8 * 3 * (size_t)n);
            d_V_.reserve(8 * (size_t)n * ldg_);
            E.d_dEdG.reserve(8 * (size_t)n * ldg_);
            // outputs and dout/dG at x, then the forces by the model's force kernels
            if (tl.tiles > 0)
                launch_tile<2>(gen_, dim3(tl.tiles), lds, st,
                                   (const TrainPlan*)d_plan_.p, Wm, (const double*)d_par_.p, tl.tt, 0,
                                   (const int*)ta.atom.p, (const int*)ta.slot.p, (const int*)ta.strct.p,
                                   (const double*)E.d_G.p, ldg_, (double*)d_out_.p, nullptr, nullptr,
                                   (double*)E.d_dEdG.p);
            HIPCHK(hipGetLastError());
            E.force_terms<double>();
            // reactions: the missed-reaction counter is cleared here (a cached chunk has no
            // neighbour launch in this call); a miss switches the chunk's workspace to receiver rows.  What is
            // missed depends on the rows alone, so a kept chunk is checked once.
            if (!C->settled) HIPCHK(hipMemsetAsync((int*)E.d_maxcnt.p + 1, 0, 4, st));
            E.assemble<double>();
            for (int attempt = 0; !C->settled; ++attempt) {
                int c[4] = {0, 0, 0, 0};
                HIPCHK(hipMemcpyAsync(c, E.d_maxcnt.p, 16, hipMemcpyDeviceToHost, st));
                HIPCHK(hipStreamSynchronize(st));
                if (!E.reactions_redo(c)) {
                    C->settled = true;
                    break;
                }
                if (attempt == 3) throw std::runtime_error("force assembly: receiver rows did not converge");
                E.assemble<double>();
            }
            hipLaunchKernelGGL(k_train_struct, dim3(nb), dim3(256), 0, st, (const double*)d_out_.p,
                               (const int*)ta.bstart.p, (const double*)ta.eref.p, loss, delta, (double*)d_dcdo_.p,
                               res(0, nbatch) + k0, res(1, nbatch) + k0);
            hipLaunchKernelGGL(k_train_fresid, dim3(nb), dim3(256), 0, st, (const double*)E.d_F.p,
                               (const double*)d_fref_.p, (const int*)ta.bstart.p, (const int64_t*)ta.fstart.p, beta,
                               (double*)d_gF_.p, res(2, nbatch) + k0);
            HIPCHK(hipGetLastError());
            if (grad) {
                HIPCHK(launch_symm_jvp(E.shape, owner_.pb.plan.generic, (const DevPlan*)E.d_plan.p,
                                       (const double*)E.d_rfe.p, (const double*)E.d_rfr.p, (const int*)E.d_type.p,
                                       (const DevStruc*)E.d_strucs.p, (const int*)E.d_astruc.p, n,
                                       (const int*)E.d_cnt.p, (const int*)E.d_nbrj.p, (const int*)E.d_meta.p,
                                       (const double4*)E.d_nbrr.p, E.maxp, E.lmaxp, (const double*)d_gF_.p,
                                       all_images ? 1 : 0, (double*)d_V_.p, ldg_, (E.moments & 1) ? 1 : 0, T_, st));
                sum_tiles(tl, st, [&](const TrainTiles& tc, int c0, int c1) {
                    const TrainPlan* tpp = (const TrainPlan*)d_plan_.p;
                    const double* par = (const double*)d_par_.p;
                    const int *ba = (const int*)ta.atom.p, *bs = (const int*)ta.strct.p;
                    const double *Gp = (const double*)E.d_G.p, *Vp = (const double*)d_V_.p, *dc = (const double*)d_dcdo_.p;
                    double* pp = (double*)d_partial_.p;
                    if (gen_)
                        hipLaunchKernelGGL(k_train_force_tile<true>, dim3(c1 - c0), dim3(kTrainThreads), flds, st, tpp, Wm,
                                           par, tc, c0, ba, bs, Gp, Vp, ldg_, dc, pp);
                    else
                        hipLaunchKernelGGL(k_train_force_tile<false>, dim3(c1 - c0), dim3(kTrainThreads), flds, st, tpp, Wm,
                                           par, tc, c0, ba, bs, Gp, Vp, ldg_, dc, pp);
                });
            }
            k0 = k1;
        }
        const double* lv = fetch_results(nbatch, 3, grad, st);
        const double *e2 = lv + nbatch, *f2 = e2 + nbatch;
        err[0] = err[1] = err[2] = 0.0;
        for (int b = 0; b < nbatch; ++b) {
            err[0] += lv[b] + 0.5 * beta * f2[b];
            err[1] += e2[b];
            err[2] += f2[b];
        }
    }

    // The chunk of nb structures: its neighbour rows and descriptors in B, its tiles and reference values on st.
    void build_chunk(Chunk& C, const int* batch, int nb, bool all_images, Engine& B, hipStream_t st) {
        std::vector<nnp_structure> cs(nb);
        std::vector<int> bstart(nb + 1, 0);
        std::vector<int64_t> fstart(nb);
        std::vector<double> eb(nb);
        // species tiles over the workspace atoms (source row = slot = workspace index)
        std::vector<std::vector<int>> atom_s(T_), struct_s(T_);
        for (int b = 0; b < nb; ++b) {
            const int sb = batch[b];
            cs[b].natoms = natoms_[sb];
            cs[b].type = types_.data() + aoff_[sb];
            cs[b].pos = hpos_.data() + 3 * aoff_[sb];
            cs[b].cell = hopen_[sb] ? nullptr : hcell_.data() + 9 * (size_t)sb;
            bstart[b + 1] = bstart[b] + natoms_[sb];
            fstart[b] = aoff_[sb];
            eb[b] = eref_[sb];
            for (int i = 0; i < natoms_[sb]; ++i) {
                const int t = types_[aoff_[sb] + i];
                atom_s[t].push_back(bstart[b] + i);
                struct_s[t].push_back(b);
            }
        }
        B.upload(cs);
        B.build_neighbors(all_images);
        B.descriptors<double>();
        C.tl = make_tiles(atom_s, atom_s, struct_s, st, C.ta);
        C.ta.bstart.reserve(4 * (size_t)(nb + 1));
        C.ta.fstart.reserve(8 * (size_t)nb);
        C.ta.eref.reserve(8 * (size_t)nb);
        HIPCHK(hipMemcpyAsync(C.ta.bstart.p, bstart.data(), 4 * (size_t)(nb + 1), hipMemcpyHostToDevice, st));
        HIPCHK(hipMemcpyAsync(C.ta.fstart.p, fstart.data(), 8 * (size_t)nb, hipMemcpyHostToDevice, st));
        HIPCHK(hipMemcpyAsync(C.ta.eref.p, eb.data(), 8 * (size_t)nb, hipMemcpyHostToDevice, st));
        HIPCHK(hipStreamSynchronize(st));  // the host vectors go out of scope
        if (B.stream != st) HIPCHK(hipStreamSynchronize(B.stream));
    }

  private:
    Engine& owner_;
    int T_ = 0, ldg_ = 0;
    int64_t ntot_ = 0, npar_dev_ = 0;
    TrainPlan plan_;
    std::vector<int64_t> goff_;
    std::vector<int> natoms_, types_;
    std::vector<int64_t> aoff_;
    std::vector<double> eref_;
    hipStream_t stream_ = nullptr;
    DevMem d_plan_, d_goff_, d_G_, d_par_, d_out_, d_dcdo_, d_res_, d_partial_, d_grp_, d_fref_, d_gF_, d_V_;
    HostPinned h_io_;
    bool grad_started_ = false;  // the call's gradient holds its first rows
    std::vector<double> hpos_, hcell_;
    std::vector<char> hopen_;
    std::vector<int> hbatom_, hbslot_, hbstruct_;
    bool has_forces_ = false;
    size_t lds_limit_ = 0;
    bool gen_ = false;  // some hidden layer is not tanh
    // tiles of the last energy-training call (batch + mode) and whether they are single-structure
    std::vector<int> tiles_key_;
    Tiles tiles_;
    TileArrays ta_;
    int natoms_batch_ = 0;
    bool one_pass_ = false;
    DevMem d_tstruct_;
    bool grouped_ = false;  // the tiles' rows by k_train_group
    GroupShape gshape_{};
    Groups groups_;
    DevMem d_gtile_;
    std::unique_ptr<Engine> ws_;  // workspace of the force passes
    // workspaces that keep the neighbour rows and descriptors of force-training chunks
    std::vector<std::unique_ptr<Chunk>> fcache_;
    std::unique_ptr<Chunk> scratch_;
    int64_t fcache_atoms_ = 0;
};

Engine& engine_of(nnp_model* m);

}  // namespace atomnn

using namespace atomnn;

struct nnp_train {
    std::unique_ptr<TrainSet> t;
};

template <typename F>
static int train_guard(F&& f) {
    try {
        set_error("");
        return f();
    } catch (const unsupported_error& e) {
        set_error(e.what());
        return NNP_EUNSUPPORTED;
    } catch (const hip_failure& e) {
        set_error(e.what());
        return NNP_EDEVICE;
    } catch (const std::bad_alloc&) {
        set_error("out of memory");
        return NNP_ENOMEM;
    } catch (const std::exception& e) {
        set_error(e.what());
        return NNP_EINVAL;
    }
}

extern "C" {

int nnp_train_create(nnp_model* m, int nstruc, const nnp_structure* s, const double* energy, nnp_train** out) {
    return train_guard([&]() {
        if (!m || !out) throw std::invalid_argument("nnp_train_create: null argument");
        *out = new nnp_train{std::make_unique<TrainSet>(engine_of(m), nstruc, s, energy)};
        return NNP_OK;
    });
}

int64_t nnp_train_nparams(nnp_train* t, int species) {
    int64_t n = -1;
    const int rc = train_guard([&]() {
        if (!t) throw std::invalid_argument("nnp_train_nparams: null argument");
        n = species < 0 ? t->t->total() : t->t->nparams(species);
        return NNP_OK;
    });
    return rc < 0 ? rc : n;
}

int nnp_train_get_params(nnp_train* t, double* x) {
    return train_guard([&]() {
        if (!t || !x) throw std::invalid_argument("nnp_train_get_params: null argument");
        t->t->get_params(x);
        return NNP_OK;
    });
}

int nnp_train_error(nnp_train* t, const double* x, int nbatch, const int* batch, int loss, double delta, double* err,
                    double* grad) {
    return train_guard([&]() {
        if (!t) throw std::invalid_argument("nnp_train_error: null argument");
        t->t->error(x, nbatch, batch, loss, delta, err, grad);
        return NNP_OK;
    });
}

int nnp_train_set_forces(nnp_train* t, const double* forces) {
    return train_guard([&]() {
        if (!t) throw std::invalid_argument("nnp_train_set_forces: null argument");
        t->t->set_forces(forces);
        return NNP_OK;
    });
}

int nnp_train_error_force(nnp_train* t, const double* x, int nbatch, const int* batch, int loss, double delta,
                          double beta, uint32_t flags, double* err, double* grad) {
    return train_guard([&]() {
        if (!t) throw std::invalid_argument("nnp_train_error_force: null argument");
        t->t->error_force(x, nbatch, batch, loss, delta, beta, flags, err, grad);
        return NNP_OK;
    });
}

void nnp_train_destroy(nnp_train* t) { delete t; }

}  // extern "C"
