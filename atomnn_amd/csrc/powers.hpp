// Angular sums and force terms for models whose G4 sets go beyond the moment expansion's zeta <= 4: every
// angular block has lambda = +-1, zeta in {1, 2, 4, 8, 16}, the GAUSS distance factor and one exponent table
// (the usual G4 sets: zeta = 1, 2, 4, 16).  The pairs are still visited one by one, but
//  * with x = |1 + lambda cos| / 2 the angular factors x^zeta come from four squarings and their
//    derivatives from D_(k+1) = 2 D_k x^(2^k), D_0 = lambda / 2, for both lambda: no selects, no pow;
//  * one lane owns a row entry j and sums over the other entry k, so R_e(j) and R_e'(j) leave the inner loop:
//      descriptors  sum_j R_e(j) [sum_k R_e(k) A_l(cos_jk)]
//      forces       dE/dd_j = sum_e R_e'(j) [sum_k S_e(cos_jk) R_e(k)],   S_e = sum_l w_el A_l
//                   v_j = sum_k dE/dcos_jk u_k,  X_j = -(dE/dd_j u_j + (v_j - (u_j . v_j) u_j) / d_j)
// Levels l: lambda = +1 in 0 .. 4 (zeta = 2^l), lambda = -1 in 5 .. 9.
#pragma once

#include "device.hpp"
#include "model.hpp"

namespace atomnn {

constexpr int kPowL = 10;           // levels
constexpr int kPowPad = kWave + 1;  // reduction row: consecutive rows start in different banks

// LDS, in elements of T: descriptors (reduction rows and their 64 partial sums), forces (weights per block)
constexpr int pow_red_elems() { return kPowL * kPowPad + kWave; }
template <int NE>
__host__ __device__ constexpr int pow_weight_elems(int ntypes) {
    return ntypes * (ntypes + 1) / 2 * NE * kPowL;
}

template <typename T>
__device__ __forceinline__ void pow_values(T cs, T (&A)[kPowL]) {
    A[0] = fabs(T(0.5) + T(0.5) * cs);
    A[5] = fabs(T(0.5) - T(0.5) * cs);
#pragma unroll
    for (int k = 1; k < 5; ++k) {
        A[k] = A[k - 1] * A[k - 1];
        A[5 + k] = A[4 + k] * A[4 + k];
    }
}

// Angular descriptors of the staged centre into Grow (zeroed by the caller).  Row entries j of a block's
// first species lie along the lanes, in parts when fewer than 33 (each part takes every parts-th k); within a
// species each unordered pair is visited once, k = j + s for s = 1 .. n / 2 around the segment.
template <typename T, int NE>
__device__ __forceinline__ void symm_angular_powers(const DevPlan* __restrict__ plan, int ti, int ntypes, const T* su,
                                                    const T* Rf, const int* seg, T* red, T* Grow, int lane) {
    const int nblk = ntypes * (ntypes + 1) / 2;
    T* psum = red + kPowL * kPowPad;
    for (int bb = 0; bb < ntypes; ++bb) {
        for (int a = 0; a <= bb; ++a) {
            const int blk = bb * (bb + 1) / 2 + a;
            const int sa = seg[a], na = seg[a + 1] - sa, sb = seg[bb], nb = seg[bb + 1] - sb;
            const bool same = a == bb;
            if (same ? na < 2 : (na == 0 || nb == 0)) continue;
            const T norm = T(plan->ang[ti][blk].norm);
            const int goff = plan->ang[ti][blk].goff;
            for (int r0 = 0; r0 < na; r0 += kWave) {
                const int nr = min(na - r0, kWave), parts = kWave / nr;
                const int part = lane / nr, j = r0 + lane - part * nr;
                const bool active = part < parts;
                T acc[NE][kPowL];
#pragma unroll
                for (int e = 0; e < NE; ++e)
#pragma unroll
                    for (int l = 0; l < kPowL; ++l) acc[e][l] = T(0);
                T rj[NE];
                if (active) {
                    const T ux = su[4 * (sa + j)], uy = su[4 * (sa + j) + 1], uz = su[4 * (sa + j) + 2];
#pragma unroll
                    for (int e = 0; e < NE; ++e) rj[e] = Rf[(sa + j) * NE + e];
                    const int hi = same ? na / 2 + 1 : nb;
                    for (int s = (same ? 1 : 0) + part; s < hi; s += parts) {
                        int k = s;
                        if (same) {
                            if (2 * s == na && j >= s) continue;  // opposite entries: once
                            k = j + s;
                            k = k >= na ? k - na : k;
                        }
                        const int pk = sb + k;
                        T A[kPowL];
                        pow_values<T>(ux * su[4 * pk] + uy * su[4 * pk + 1] + uz * su[4 * pk + 2], A);
#pragma unroll
                        for (int e = 0; e < NE; ++e) {
                            const T rk = Rf[pk * NE + e];
#pragma unroll
                            for (int l = 0; l < kPowL; ++l) acc[e][l] += A[l] * rk;
                        }
                    }
                }
                // sums over the lanes in a fixed order, one exponent at a time: 6 lanes of 11 addends per level
#pragma unroll
                for (int e = 0; e < NE; ++e) {
#pragma unroll
                    for (int l = 0; l < kPowL; ++l) red[l * kPowPad + lane] = active ? acc[e][l] * rj[e] : T(0);
                    __syncthreads();
                    const int l = lane / 6, q = lane - 6 * l;
                    T s = T(0);
                    if (l < kPowL)
                        for (int m = 11 * q; m < min(kWave, 11 * q + 11); ++m) s += red[l * kPowPad + m];
                    psum[lane] = s;
                    __syncthreads();
                    if (lane < kPowL) {
                        const int f = plan->pow_index[(((size_t)ti * nblk + blk) * NE + e) * kPowL + lane];
                        if (f >= 0) {
                            T t = T(0);
#pragma unroll
                            for (int m = 0; m < 6; ++m) t += psum[6 * lane + m];
                            Grow[goff + f] += t * norm;
                        }
                    }
                    __syncthreads();
                }
            }
        }
    }
}

// Block weights w[blk][e][l] = norm dE/dG[goff + f(e, l)] (0 where the block has no such function).
template <typename T, int NE>
__device__ __forceinline__ void pow_weights(const DevPlan* __restrict__ plan, int ti, int ntypes, const T* W, T* w,
                                            int lane) {
    const int nblk = ntypes * (ntypes + 1) / 2;
    for (int it = lane; it < nblk * NE * kPowL; it += kWave) {
        const DevAngular& A = plan->ang[ti][it / (NE * kPowL)];
        const int f = plan->pow_index[(size_t)ti * nblk * NE * kPowL + it];
        w[it] = f >= 0 ? W[A.goff + f] * T(A.norm) : T(0);
    }
}

// Angular part of dE/dr of entry p of species s (lanes own entries, k runs over the staged entries, the same
// for every lane): g += dE/dd u + (v - (u . v) u) / d.
template <typename T, int NE>
__device__ __forceinline__ void force_powers_entry(int ntypes, const T* su, const T* Rf, const T* Rd, const int* seg,
                                                   const T* wtab, int p, int s, T& gx, T& gy, T& gz) {
    const T ux = su[4 * p], uy = su[4 * p + 1], uz = su[4 * p + 2];
    T rj[NE], sd[NE];
#pragma unroll
    for (int e = 0; e < NE; ++e) {
        rj[e] = Rf[p * NE + e];
        sd[e] = T(0);
    }
    T vx = T(0), vy = T(0), vz = T(0);
    for (int b = 0; b < ntypes; ++b) {
        const int blk = b >= s ? b * (b + 1) / 2 + s : s * (s + 1) / 2 + b;
        T w[NE][kPowL];
#pragma unroll
        for (int e = 0; e < NE; ++e)
#pragma unroll
            for (int l = 0; l < kPowL; ++l) w[e][l] = wtab[(blk * NE + e) * kPowL + l];
        const int k1 = seg[b + 1];
        for (int k = seg[b]; k < k1; ++k) {
            const T kx = su[4 * k], ky = su[4 * k + 1], kz = su[4 * k + 2];
            const T cs = ux * kx + uy * ky + uz * kz;
            T A[kPowL], D[kPowL];
            pow_values<T>(cs, A);
            D[0] = T(0.5);
            D[5] = T(-0.5);
#pragma unroll
            for (int q = 1; q < 5; ++q) {
                D[q] = D[q - 1] * (A[q - 1] + A[q - 1]);
                D[5 + q] = D[4 + q] * (A[4 + q] + A[4 + q]);
            }
            T dc = T(0);
#pragma unroll
            for (int e = 0; e < NE; ++e) {
                const T rk = k == p ? T(0) : Rf[k * NE + e];  // the entry itself is no pair
                T S = T(0), dS = T(0);
#pragma unroll
                for (int l = 0; l < kPowL; ++l) {
                    S += w[e][l] * A[l];
                    dS += w[e][l] * D[l];
                }
                sd[e] += S * rk;
                dc += dS * (rj[e] * rk);
            }
            vx += dc * kx;
            vy += dc * ky;
            vz += dc * kz;
        }
    }
    T dd = T(0);
#pragma unroll
    for (int e = 0; e < NE; ++e) dd += sd[e] * Rd[p * NE + e];
    const T di = T(1) / su[4 * p + 3], uv = ux * vx + uy * vy + uz * vz;
    gx += dd * ux + di * (vx - uv * ux);
    gy += dd * uy + di * (vy - uv * uy);
    gz += dd * uz + di * (vz - uv * uz);
}

}  // namespace atomnn
