// Neighbour-list kernels.
//
// The list reproduces AtomNN's NeighborList::build (struc/neighbor.cpp:59-171) entry for
// entry: for centre i, neighbours j in ascending order; for each j the periodic images
// r_ij - R_n in the order of the image table (a-major over the norm-sorted lattice vectors,
// neighbor.cpp:87-95) relative to the minimum-image base Cell::diff(r_i, r_j)
// (struc/cell.cpp:103-128); inclusive cutoff d^2 <= rc^2; self images only when
// d^2 > 1e-6; the strictly closest image of each j != i (first on ties, and only below
// ||R||_F) carries the min flag (neighbor.cpp:131-141).  Open structures have no images
// and no min flags (neighbor.cpp:149-170).
//
// Two searches produce the same list:
//  * all-pairs: a centre's wavefronts sweep j in chunks of 64; the (j, image) pairs within
//    reach are spread over the lanes, prefix sums place the kept entries in order.  Used for
//    small cells (any image shell > 0) and small structures.
//  * cell list: for structures whose image shells are all 0 (every cell height > 2 rc) the
//    entry of j is exactly diff(r_i, r_j) when within rc; candidates come from the 27
//    neighbouring fractional bins as one flat list; each wavefront marks its kept candidates
//    in an LDS bitmap over the structure's atoms and reads them out in index order (very
//    large structures: a bitonic sort of the kept candidates instead), so the order is the
//    reference's.
// The partner of an entry (the mirrored pair that carries the Newton reaction) is found
// by the force-assembly kernel.
#include "device.hpp"

namespace atomnn {

// math/special.hpp:46-47 with z = 1: fmod(x, 1) = x - trunc(x) exactly for finite x.
__device__ __forceinline__ double fmod1(double x) { return x - trunc(x); }
__device__ __forceinline__ double wrap_half(double x) { return fmod1(fmod1(x + 0.5) + 1.0) - 0.5; }

// Cell::diff (cell.cpp:103-128)
__device__ __forceinline__ void cell_diff(const DevStruc& s, double dx, double dy, double dz, double& ox, double& oy,
                                          double& oz) {
    double f0 = s.RInv[0] * dx + s.RInv[1] * dy + s.RInv[2] * dz;
    double f1 = s.RInv[3] * dx + s.RInv[4] * dy + s.RInv[5] * dz;
    double f2 = s.RInv[6] * dx + s.RInv[7] * dy + s.RInv[8] * dz;
    f0 = wrap_half(f0);
    f1 = wrap_half(f1);
    f2 = wrap_half(f2);
    ox = s.R[0] * f0 + s.R[1] * f1 + s.R[2] * f2;
    oy = s.R[3] * f0 + s.R[4] * f1 + s.R[5] * f2;
    oz = s.R[6] * f0 + s.R[7] * f1 + s.R[8] * f2;
    const double d2 = ox * ox + oy * oy + oz * oz;
    if (d2 > s.dMax2) {
        double bx = ox, by = oy, bz = oz, best = d2;
#pragma unroll
        for (int q = 0; q < 6; ++q) {
            const int c = q >> 1;
            const double sg = (q & 1) ? -1.0 : 1.0;
            const double tx = ox + sg * s.R[c], ty = oy + sg * s.R[3 + c], tz = oz + sg * s.R[6 + c];
            const double t2 = tx * tx + ty * ty + tz * tz;
            if (t2 < best) {
                best = t2;
                bx = tx;
                by = ty;
                bz = tz;
            }
        }
        ox = bx;
        oy = by;
        oz = bz;
    }
}

// image vector R_n = a Rv0 + b Rv1 + c Rv2 (neighbor.cpp:87-95)
__device__ __forceinline__ void image_vec(const DevStruc& s, int a, int b, int c, double& x, double& y, double& z) {
    x = (double)a * s.Rv[0] + (double)b * s.Rv[3] + (double)c * s.Rv[6];
    y = (double)a * s.Rv[1] + (double)b * s.Rv[4] + (double)c * s.Rv[7];
    z = (double)a * s.Rv[2] + (double)b * s.Rv[5] + (double)c * s.Rv[8];
}

// Exclusive prefix sum over the wavefront in six DPP adds: shifts by 1, 2, 4 and 8 inside each row of 16
// lanes, then the last lane of row 0 (2) onto row 1 (3), then lane 31 onto rows 2 and 3.
__device__ __forceinline__ int wave_excl_scan(int v, int lane, int& total) {
    (void)lane;
    int x = v;
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);
    total = __builtin_amdgcn_readlane(x, kWave - 1);
    return x - v;
}

// Index table of a row from its ascending entries: entry p with index j opens every table entry after its
// predecessor's (index jp, -1 for the first entry) up to its own.
__device__ __forceinline__ void row_tab_open(unsigned short* tab, int width, int jp, int j, int p) {
    const int q0 = jp < 0 ? 0 : jp / width + 1, q1 = j / width;
    for (int q = q0; q <= q1; ++q) tab[q] = (unsigned short)p;
}
// the table entries after the last row entry (index j, -1 in an empty row) of a row of P entries
__device__ __forceinline__ void row_tab_close(unsigned short* tab, int width, int j, int P, int lane) {
    const int q0 = j < 0 ? 0 : j / width + 1;
    if (lane >= q0 && lane < kRowTab) tab[lane] = (unsigned short)P;
}

__device__ __forceinline__ void put_entry(int64_t slot, int j, int img, int typ, bool mn, double x, double y, double z,
                                          double d, int* nbr_j, unsigned short* nbr_key, int* nbr_meta,
                                          double4* nbr_r) {
    nbr_j[slot] = j;
    nbr_key[slot] = (unsigned short)j;
    nbr_meta[slot] = (img << 8) | (typ << 1) | (mn ? 1 : 0);
    nbr_r[slot] = make_double4(x, y, z, d);
}

// The last of the nb (<= 32) neighbouring bins whose first flat candidate is <= c: a binary
// search over the lanes' bin starts in five shuffles, executed by every lane.
__device__ __forceinline__ int owner_bin(int bfirst, int nb, int c) {
    int lo = 0;
#pragma unroll
    for (int step = 16; step > 0; step >>= 1) {
        const int mid = lo + step;
        const int fq = __shfl(bfirst, mid < nb ? mid : nb - 1, kWave);
        if (mid < nb && fq <= c) lo = mid;
    }
    return lo;
}

// Image index range that can hold r - R_n within rc along each norm-sorted lattice vector: with
// f_q = Gv_q . r, |f_q - n_q| = |(r - R_n) . Gv_q| <= rc |Gv_q|.  The ranges are sub-ranges of the
// image table, walked in its order, so the kept images and their order are unchanged.
struct ImgRange {
    int lo[3], hi[3];
};
__device__ __forceinline__ ImgRange img_range(const DevStruc& s, double bx, double by, double bz) {
    ImgRange g;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        const double f = s.Gv[3 * q] * bx + s.Gv[3 * q + 1] * by + s.Gv[3 * q + 2] * bz;
        g.lo[q] = max(-s.shell[q], (int)ceil(f - s.reach[q]));
        g.hi[q] = min(s.shell[q], (int)floor(f + s.reach[q]));
    }
    return g;
}

// The per-pass counters (neighbour maximum, missed reactions, work counter of the fused kernel), cleared by
// the first block of the neighbour kernels: nothing else touches them before the force assembly.
struct PassCounters {
    int* maxcnt;
    int* work;
};
__device__ __forceinline__ void clear_counters(const PassCounters& pc) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        pc.maxcnt[0] = 0;  // neighbour maximum
        pc.maxcnt[1] = 0;  // reactions missed by the force assembly's gather
        if (pc.work) *pc.work = 0;
    }
}

// ------------------------------------------------------------------ all-pairs search
// One centre a block.  Wavefront w takes the atoms 64 (W r + w) to 64 (W r + w) + 63 of round r, one a lane: difference
// vector and box of images within reach.  Where no atom has two images in its box (open structures, cells at least
// two cutoffs across) each lane takes its own.  Otherwise the images of all of them are spread over the lanes in (atom,
// image) order, twice: to count what each atom keeps and find its nearest image, and to write the entries, next to
// each other.  Places in the row come from scans inside the wavefront and the wavefronts' totals through LDS.
// A lane that walks its own atom's images costs the wavefront the longest walk, in a chain of FP64 latencies, twice:
// about 110 images are within reach of a centre, all of them on two lanes of a two-atom cell.  Walked so / now: 20 uneven
// cells of up to 512 atoms 24.5 / 9.1 us, one of 64 atoms 9.7 / 8.2, 600 of 20 atoms 51 / 29, 60 of 250 atoms 57 / 42, 512
// of up to 512 atoms 101 / 67, open structures of 2000 and 7000 atoms 46 / 26 and 234 / 163.
// W: four wavefronts a centre shorten the chain while the centres alone leave the chip idle; beyond kPairCentres one
// (34,700 centres: four 140 us, one 96, before the single-image path; 4,800: 24 against 17 us).
constexpr int kPairCentres = 2048;
struct PairChunk {  // a wavefront's 64 atoms
    double b[3][kWave];              // difference vector
    unsigned long long mind[kWave];  // bits of the smallest distance
    int off[kWave], lo[3][kWave], ext[2][kWave];  // first image, box of images (lowest indexes, last two extents)
    int type[kWave], kept[kWave], minn[kWave];
};
template <int W>
__global__ __launch_bounds__(kWave * W) void k_neigh_allpairs(const DevStruc* __restrict__ S, const int* __restrict__ atom_struc,
                                                          const double* __restrict__ pos, const int* __restrict__ type,
                                                          const int* __restrict__ centres, double rc2, int maxp,
                                                          int* __restrict__ cnt, int* __restrict__ nbr_j,
                                                          int* __restrict__ nbr_meta, double4* __restrict__ nbr_r,
                                                          unsigned short* __restrict__ row_tab, unsigned short* __restrict__ nbr_key, PassCounters pc) {
    clear_counters(pc);
    __shared__ PairChunk chunk[W];
    __shared__ int wtot[2][W];
    const int i = centres[blockIdx.x];
    const DevStruc& s = S[atom_struc[i]];
    const int lane = threadIdx.x % kWave, w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const bool one = W == 1 || s.natoms <= kWave;  // (uniform)
    if (one && w > 0) return;
    const int li = i - s.atom0;
    const double xi = pos[3 * i], yi = pos[3 * i + 1], zi = pos[3 * i + 2];
    const int64_t row = (int64_t)i * maxp;
    const int tw = row_tab_width(s.natoms);
    PairChunk& L = chunk[w];
    const int w1 = 2 * s.shell[1] + 1, w2 = 2 * s.shell[2] + 1;
    const bool periodic = s.periodic;
    const double fro = s.fro;
    const auto ordered = [] {  // LDS writes of some lanes before reads of others of the same wavefront
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
        __builtin_amdgcn_wave_barrier();
    };
    int written = 0;
    for (int j0 = 0, buf = 0; j0 < s.natoms; j0 += kWave * W, buf ^= 1) {
        const int jw = j0 + w * kWave, j = jw + lane;
        const bool valid = j < s.natoms;
        double bx = 0, by = 0, bz = 0;
        // images of this j that can be within rc (open structures: the single image 0)
        ImgRange g{{0, 0, 0}, {-1, -1, -1}};
        int tj = 0;
        if (valid) {
            const int gj = s.atom0 + j;
            tj = type[gj];
            const double dx = xi - pos[3 * gj], dy = yi - pos[3 * gj + 1], dz = zi - pos[3 * gj + 2];
            if (periodic) {
                cell_diff(s, dx, dy, dz, bx, by, bz);
                g = img_range(s, bx, by, bz);
            } else {
                bx = dx;
                by = dy;
                bz = dz;
                g = ImgRange{{0, 0, 0}, {0, 0, 0}};
            }
        }
        const int e0 = max(0, g.hi[0] - g.lo[0] + 1), e1 = max(0, g.hi[1] - g.lo[1] + 1), e2 = max(0, g.hi[2] - g.lo[2] + 1);
        const int mimg = e0 * e1 * e2;
        // no atom with two images (open structures, cells at least two cutoffs across): each lane takes its own
        const bool single = __all(mimg <= 1);
        int images = 0, mine = 0, n1 = 0;  // images of the wavefront's atoms; with `single` this lane's
        double rx1 = 0, ry1 = 0, rz1 = 0, d1 = 0;
        if (single) {
            if (mimg == 1) {
                n1 = ((g.lo[0] + s.shell[0]) * w1 + (g.lo[1] + s.shell[1])) * w2 + (g.lo[2] + s.shell[2]);
                double ix = 0, iy = 0, iz = 0;
                if (periodic) image_vec(s, g.lo[0], g.lo[1], g.lo[2], ix, iy, iz);
                rx1 = bx - ix;
                ry1 = by - iy;
                rz1 = bz - iz;
                const double d2 = rx1 * rx1 + ry1 * ry1 + rz1 * rz1;
                if (d2 <= rc2 && (j != li || 1e-6 < d2)) {
                    mine = 1;
                    d1 = sqrt(d2);
                }
            }
        } else {
            L.type[lane] = tj;
            L.off[lane] = wave_excl_scan(mimg, lane, images);
            L.b[0][lane] = bx;
            L.b[1][lane] = by;
            L.b[2][lane] = bz;
#pragma unroll
            for (int q = 0; q < 3; ++q) L.lo[q][lane] = g.lo[q];
            L.ext[0][lane] = e1;
            L.ext[1][lane] = e2;
            L.kept[lane] = 0;
            L.mind[lane] = __double_as_longlong(fro);  // (distances are positive: their bits order as they do)
            L.minn[lane] = INT_MAX;
            ordered();
        }
        // image q of the wavefront's: its atom (the last whose images begin at or before q), offset and vector
        const auto image = [&](int q, int& k, int& n, double& rx, double& ry, double& rz) {
            k = 0;
#pragma unroll
            for (int o = 32; o > 0; o >>= 1)
                if (L.off[k + o] <= q) k += o;
            const int t = q - L.off[k], f1 = L.ext[0][k], f2 = L.ext[1][k];
            const int u = t / f2, v = u / f1;
            const int a = L.lo[0][k] + v, b = L.lo[1][k] + u - v * f1, c = L.lo[2][k] + t - u * f2;
            n = ((a + s.shell[0]) * w1 + (b + s.shell[1])) * w2 + (c + s.shell[2]);
            double ix = 0, iy = 0, iz = 0;
            if (periodic) image_vec(s, a, b, c, ix, iy, iz);
            rx = L.b[0][k] - ix;
            ry = L.b[1][k] - iy;
            rz = L.b[2][k] - iz;
            const double d2 = rx * rx + ry * ry + rz * rz;
            return d2 <= rc2 && (jw + k != li || 1e-6 < d2) ? d2 : -1.0;  // -1: not kept
        };
        for (int q = lane; q < images; q += kWave) {
            int k, n;
            double rx, ry, rz;
            const double d2 = image(q, k, n, rx, ry, rz);
            if (d2 < 0) continue;
            atomicAdd(&L.kept[k], 1);
            if (periodic && jw + k != li) atomicMin(&L.mind[k], (unsigned long long)__double_as_longlong(sqrt(d2)));
        }
        if (!single) {
            ordered();
            mine = L.kept[lane];
        }
        int tot;
        int at = written + wave_excl_scan(mine, lane, tot);
        if (!one) {
            if (lane == 0) wtot[buf][w] = tot;
            __syncthreads();  // (the other buffer's readers passed the barrier before)
            tot = 0;
#pragma unroll
            for (int v = 0; v < W; ++v) {
                const int c = wtot[buf][v];
                if (v < w) at += c;
                tot += c;
            }
        }
        // the row's index table: atom j opens slot j / width when it is the slot's first
        if (valid && j % tw == 0) row_tab[(int64_t)i * kRowTab + j / tw] = (unsigned short)min(at, maxp);
        if (single && mine && at < maxp)
            put_entry(row + at, j, n1, tj, j != li && periodic && d1 < fro, rx1, ry1, rz1, d1, nbr_j, nbr_key, nbr_meta,
                      nbr_r);
        int put = __builtin_amdgcn_readfirstlane(at);  // (lane 0's: the wavefront's first entry)
        for (int q0 = 0; q0 < images; q0 += kWave) {
            int k = 0, n = 0;
            double rx = 0, ry = 0, rz = 0, d2 = -1.0;
            if (q0 + lane < images) d2 = image(q0 + lane, k, n, rx, ry, rz);
            const bool keep = d2 >= 0;
            const double d = keep ? sqrt(d2) : 0.0;
            // the nearest image, the first of equally near ones (images of an atom come in increasing n)
            const bool near = keep && periodic && jw + k != li && d < fro &&
                              (unsigned long long)__double_as_longlong(d) == L.mind[k];
            if (near) atomicMin(&L.minn[k], n);
            ordered();
            const uint64_t mask = __ballot(keep);
            const int e = put + __popcll(mask & ((1ull << lane) - 1));
            if (keep && e < maxp)
                put_entry(row + e, jw + k, n, L.type[k], near && n == L.minn[k], rx, ry, rz, d, nbr_j, nbr_key, nbr_meta,
                          nbr_r);
            put += __popcll(mask);
        }
        ordered();  // (before the next round's atoms are staged)
        written += tot;
    }
    if (w > 0) return;
    const int q0 = (s.natoms + tw - 1) / tw;  // slots past the last atom
    if (lane >= q0 && lane < kRowTab) row_tab[(int64_t)i * kRowTab + lane] = (unsigned short)min(written, maxp);
    if (lane == 0) {
        cnt[i] = written;
    }
}

// ------------------------------------------------------------------ cell list
// Bin of atom i (fractional coordinates wrapped into [0,1)), or -1 outside the cell list.
// The fields of a structure the binning reads (held in registers by the one-structure binning).
struct BinGeom {
    double RInv[9];
    int nbin[3];
    int bin0;
    int mode;
};
__device__ __forceinline__ BinGeom bin_geom(const DevStruc& s) {
    BinGeom g;
#pragma unroll
    for (int q = 0; q < 9; ++q) g.RInv[q] = s.RInv[q];
#pragma unroll
    for (int q = 0; q < 3; ++q) g.nbin[q] = s.nbin[q];
    g.bin0 = s.bin0;
    g.mode = s.mode;
    return g;
}
template <class SG>
__device__ __forceinline__ int bin_xyz(const SG& s, double x, double y, double z) {
    if (s.mode != 1) return -1;
    int b[3];
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        double f = s.RInv[3 * r] * x + s.RInv[3 * r + 1] * y + s.RInv[3 * r + 2] * z;
        f -= floor(f);
        int q = (int)(f * s.nbin[r]);
        q = q < 0 ? 0 : (q >= s.nbin[r] ? s.nbin[r] - 1 : q);
        b[r] = q;
    }
    return s.bin0 + (b[0] * s.nbin[1] + b[1]) * s.nbin[2] + b[2];
}
// An atom's entry in the bin-ordered candidate array: its fractional coordinates in [0, 1] rounded to
// FP32 and its index, what the cell-list search's distance filter reads.
template <class SG>
__device__ __forceinline__ float4 bin_entry(const SG& s, double x, double y, double z, int i) {
    float f[3];
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        const double v = s.RInv[3 * r] * x + s.RInv[3 * r + 1] * y + s.RInv[3 * r + 2] * z;
        f[r] = (float)(v - floor(v));
    }
    return make_float4(f[0], f[1], f[2], __int_as_float(i));
}
__device__ __forceinline__ int bin_of(const DevStruc* __restrict__ S, const int* __restrict__ atom_struc,
                                      const double* __restrict__ pos, int i) {
    return bin_xyz(S[atom_struc[i]], pos[3 * i], pos[3 * i + 1], pos[3 * i + 2]);
}

// Binning of the cell-list atoms: each atom's bin, every bin's first slot (nbins + 1 starts, so a bin ends
// where the next begins), and in bin order the atoms and their filter entries.  The order inside a bin is set by
// atomics and does not matter: the search places its entries by index.
//
// Up to kBinsSmallAtoms atoms of one structure (half as many of several, whose cells are looked up per atom)
// one workgroup does it all with the counters in LDS, each thread's atoms in registers between the count
// and the fill; larger batches take three launches (count with each atom's place in its bin, scan, fill).
// Kernel times, one workgroup against the three launches: 2048 atoms 7.8 / 10.1 us, 4096 atoms 9.4-11.5 / 10.9 us
// (and two launch gaps), 8192 atoms 18.8 / 11.2 us; 8192 atoms of 16 structures 25.9 / 11.6 us, 32768
// atoms of 16 structures 75 us / 14 us.
// ONE: a single structure, whose cell is read once per wavefront (scalar loads) instead of per atom.
__global__ void k_bin_atoms(const DevStruc* __restrict__ S, const int* __restrict__ atom_struc,
                            const double* __restrict__ pos, int natoms_total, int* __restrict__ atom_bin,
                            int* __restrict__ bin_count, int* __restrict__ bin_rank) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= natoms_total) return;
    const int bin = bin_of(S, atom_struc, pos, i);
    atom_bin[i] = bin;
    if (bin >= 0) bin_rank[i] = atomicAdd(&bin_count[bin], 1);
}

constexpr int kBinsSmallAtoms = 4096;
constexpr int kBinsSmallBins = 4096;
constexpr int kBinsPerThread = kBinsSmallAtoms / 1024;

// Exclusive scan of one value per thread over 1024 threads, and the block's total.
__device__ __forceinline__ int block_excl_scan(int v, int* part, int& total) {
    const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
    int wtot;
    int x = wave_excl_scan(v, lane, wtot);
    if (lane == 0) part[wv] = wtot;
    __syncthreads();
    total = 0;
#pragma unroll
    for (int k = 0; k < 1024 / kWave; ++k) {
        x += k < wv ? part[k] : 0;
        total += part[k];
    }
    return x;
}

template <bool ONE>
__global__ __launch_bounds__(1024) void k_bins_small(const DevStruc* __restrict__ S, const int* __restrict__ atom_struc,
                                                     const double* __restrict__ pos, int ntot, int nbins,
                                                     int* __restrict__ atom_bin, int* __restrict__ bin_start,
                                                     int* __restrict__ bin_atoms, float4* __restrict__ bin_pos) {
    __shared__ int cnt_l[kBinsSmallBins];
    __shared__ int part[1024 / kWave];
    const int t = threadIdx.x;
    for (int b = t; b < nbins; b += 1024) cnt_l[b] = 0;
    BinGeom g1{};
    if constexpr (ONE) g1 = bin_geom(S[0]);
    __syncthreads();
    // each thread's atoms i = t + 1024 k, in groups of four; the positions of a group are loaded
    // unconditionally at clamped (in-bounds) indices, so the four loads go out together (a guarded load
    // becomes a branch with a full wait after it); the exit test is the same for the whole block
    int mybin[kBinsPerThread], rank[kBinsPerThread];
    float4 entry[kBinsPerThread];
#pragma unroll
    for (int k0 = 0; k0 < kBinsPerThread; k0 += 4) {
        if (k0 * 1024 >= ntot) break;
        double px[4], py[4], pz[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int ic = min(t + 1024 * (k0 + q), ntot - 1);
            px[q] = pos[3 * ic];
            py[q] = pos[3 * ic + 1];
            pz[q] = pos[3 * ic + 2];
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int k = k0 + q, i = t + 1024 * k;
            mybin[k] = -1;
            if (i < ntot) {
                int bin;
                if constexpr (ONE) {
                    bin = bin_xyz(g1, px[q], py[q], pz[q]);
                    entry[k] = bin_entry(g1, px[q], py[q], pz[q], i);
                } else {
                    const DevStruc& s = S[atom_struc[i]];
                    bin = bin_xyz(s, px[q], py[q], pz[q]);
                    if (bin >= 0) entry[k] = bin_entry(s, px[q], py[q], pz[q], i);
                }
                atom_bin[i] = bin;
                mybin[k] = bin;
                if (bin >= 0) rank[k] = atomicAdd(&cnt_l[bin], 1);
            }
        }
    }
    __syncthreads();
    // exclusive scan in place: four consecutive bins per thread, then a scan of the 1024 thread sums
    int loc[4], sum = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int b = 4 * t + k;
        loc[k] = sum;
        sum += b < nbins ? cnt_l[b] : 0;
    }
    int total;
    const int excl = block_excl_scan(sum, part, total);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int b = 4 * t + k;
        if (b < nbins) {
            bin_start[b] = excl + loc[k];
            cnt_l[b] = excl + loc[k];
        }
    }
    if (t == 0) bin_start[nbins] = total;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kBinsPerThread; ++k) {
        if (k * 1024 >= ntot) break;
        const int b = mybin[k];
        if (b < 0) continue;
        const int slot = cnt_l[b] + rank[k];
        bin_atoms[slot] = t + 1024 * k;
        bin_pos[slot] = entry[k];
    }
}

// Bin starts (exclusive scan of the counts, the total last) by one block, four bins per thread and step; the
// counts are cleared behind it for the next pass.
__global__ __launch_bounds__(1024) void k_bin_scan(int* __restrict__ count, int* __restrict__ start, int nbins) {
    __shared__ int part[1024 / kWave];
    const int t = threadIdx.x;
    int carry = 0;
    for (int base = 0; base < nbins; base += 4096) {
        const int b0 = base + 4 * t;
        int v[4], sum = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = b0 + k < nbins ? count[b0 + k] : 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) sum += v[k];
        int total;
        int at = carry + block_excl_scan(sum, part, total);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (b0 + k < nbins) {
                start[b0 + k] = at;
                count[b0 + k] = 0;
            }
            at += v[k];
        }
        carry += total;
        __syncthreads();  // part is rewritten by the next step
    }
    if (t == 0) start[nbins] = carry;
}

// Scatter atoms into their bins.
__global__ void k_fill_bins(const DevStruc* __restrict__ S, const int* __restrict__ atom_struc,
                            const double* __restrict__ pos, const int* __restrict__ atom_bin, int natoms_total,
                            const int* __restrict__ bin_start, const int* __restrict__ bin_rank,
                            int* __restrict__ bin_atoms, float4* __restrict__ bin_pos) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= natoms_total) return;
    const int b = atom_bin[i];
    if (b < 0) return;
    const int slot = bin_start[b] + bin_rank[i];
    bin_atoms[slot] = i;
    bin_pos[slot] = bin_entry(S[atom_struc[i]], pos[3 * i], pos[3 * i + 1], pos[3 * i + 2], i);
}

// One wavefront per centre: gather candidates from the 27 neighbouring bins, keep those with
// |diff(r_i, r_j)| <= rc, sort the kept entries by j in LDS, write them in order.
// LDS: vals double[cap][4] | keys int[cap] | skey int[n2cap] | perm int[n2cap], n2cap = 2^k >= cap.
__global__ __launch_bounds__(kWave) void k_neigh_cells(const DevStruc* __restrict__ S, const int* __restrict__ atom_struc,
                                                       const double* __restrict__ pos, const int* __restrict__ type,
                                                       const int* __restrict__ centres, const int* __restrict__ atom_bin,
                                                       const int* __restrict__ bin_start,
                                                       const int* __restrict__ bin_atoms, double rc2, int maxp, int n2cap,
                                                       int* __restrict__ cnt, int* __restrict__ nbr_j,
                                                       int* __restrict__ nbr_meta, double4* __restrict__ nbr_r,
                                                       unsigned short* __restrict__ row_tab, unsigned short* __restrict__ nbr_key, PassCounters pc) {
    extern __shared__ double lds_cells[];
    clear_counters(pc);
    const int cap = maxp;
    double* vals = lds_cells;
    int* keys = (int*)(vals + 4 * cap);
    int* skey = keys + cap;
    int* perm = skey + n2cap;
    const int i = centres[blockIdx.x];
    const DevStruc& s = S[atom_struc[i]];
    const int lane = threadIdx.x;
    const double xi = pos[3 * i], yi = pos[3 * i + 1], zi = pos[3 * i + 2];
    const int myb = atom_bin[i] - s.bin0;
    const int bz = myb % s.nbin[2], by = (myb / s.nbin[2]) % s.nbin[1], bx = myb / (s.nbin[2] * s.nbin[1]);
    // neighbouring bins (along an axis with fewer than 3 bins every bin is visited once): lane o
    // owns bin o; a wave prefix sum over their counts gives one flat candidate list
    const int n0 = s.nbin[0] < 3 ? s.nbin[0] : 3, n1 = s.nbin[1] < 3 ? s.nbin[1] : 3, n2 = s.nbin[2] < 3 ? s.nbin[2] : 3;
    const int nb = n0 * n1 * n2;  // <= 27
    int bstart = 0, bcount = 0;
    if (lane < nb) {
        const int o2 = lane % n2, o1 = (lane / n2) % n1, o0 = lane / (n2 * n1);
        const int cx = s.nbin[0] < 3 ? o0 : (bx + o0 - 1 + s.nbin[0]) % s.nbin[0];
        const int cy = s.nbin[1] < 3 ? o1 : (by + o1 - 1 + s.nbin[1]) % s.nbin[1];
        const int cz = s.nbin[2] < 3 ? o2 : (bz + o2 - 1 + s.nbin[2]) % s.nbin[2];
        const int b = s.bin0 + (cx * s.nbin[1] + cy) * s.nbin[2] + cz;
        bstart = bin_start[b];
        bcount = bin_start[b + 1] - bstart;
    }
    int ncand;
    const int bfirst = wave_excl_scan(bcount, lane, ncand);  // first flat candidate of bin `lane`
    int kept = 0;
    for (int c0 = 0; c0 < ncand; c0 += kWave) {
        const int c = c0 + lane;
        const int ob = owner_bin(bfirst, nb, c);
        const int ostart = __shfl(bstart, ob, kWave), ofirst = __shfl(bfirst, ob, kWave);
        bool keep = false;
        double rx = 0, ry = 0, rz = 0, d2 = 0;
        int gj = 0;
        if (c < ncand) {
            gj = bin_atoms[ostart + (c - ofirst)];
            if (gj != i) {
                cell_diff(s, xi - pos[3 * gj], yi - pos[3 * gj + 1], zi - pos[3 * gj + 2], rx, ry, rz);
                d2 = rx * rx + ry * ry + rz * rz;
                keep = d2 <= rc2;
            }
        }
        int tot;
        const int at = kept + wave_excl_scan(keep ? 1 : 0, lane, tot);
        if (keep && at < cap) {
            keys[at] = gj - s.atom0;
            vals[4 * at] = rx;
            vals[4 * at + 1] = ry;
            vals[4 * at + 2] = rz;
            vals[4 * at + 3] = d2;
        }
        kept += tot;
    }
    __syncthreads();
    const int P = kept < cap ? kept : cap;
    int n2p = 1;
    while (n2p < P) n2p <<= 1;
    for (int q = lane; q < n2p; q += kWave) {
        skey[q] = q < P ? keys[q] : 0x7fffffff;
        perm[q] = q;
    }
    __syncthreads();
    // bitonic sort of (key, slot) by key; keys are distinct atoms
    for (int k = 2; k <= n2p; k <<= 1) {
        for (int jj = k >> 1; jj > 0; jj >>= 1) {
            for (int q = lane; q < n2p; q += kWave) {
                const int p = q ^ jj;
                if (p > q) {
                    const bool up = (q & k) == 0;
                    const int a = skey[q], b = skey[p];
                    if ((a > b) == up) {
                        skey[q] = b;
                        skey[p] = a;
                        const int t = perm[q];
                        perm[q] = perm[p];
                        perm[p] = t;
                    }
                }
            }
            __syncthreads();
        }
    }
    const int64_t row = (int64_t)i * maxp;
    for (int q = lane; q < P; q += kWave) {
        const int src = perm[q];
        const int j = keys[src];
        const double d = sqrt(vals[4 * src + 3]);
        // one image per j: it is the minimum image when below ||R||_F (neighbor.cpp:132-140)
        put_entry(row + q, j, 0, type[s.atom0 + j], d < s.fro, vals[4 * src], vals[4 * src + 1], vals[4 * src + 2], d,
                  nbr_j, nbr_key, nbr_meta, nbr_r);
        row_tab_open(row_tab + (int64_t)i * kRowTab, row_tab_width(s.natoms), q > 0 ? skey[q - 1] : -1, j, q);
    }
    row_tab_close(row_tab + (int64_t)i * kRowTab, row_tab_width(s.natoms), P > 0 ? skey[P - 1] : -1, P, lane);
    if (lane == 0) {
        cnt[i] = kept;
    }
}

// Cell list without a sort.  One wavefront per centre:
//  1. the 27 neighbouring bins are at most 18 runs of consecutive bins (three bins along the last
//     axis, two runs where they wrap), one flat candidate list;
//  2. filter: every candidate's distance from the bin-ordered FP32 fractional coordinates (one
//     coalesced 16-byte load), against rc plus a bound on the FP32 error; what may be within rc
//     (45-70 of some 320 candidates) goes to a short list in LDS;
//  3. the listed candidates take the reference's Cell::diff and its inclusive test in FP64; kept ones set
//     their bit in an LDS bitmap over the structure's atoms (an atomic OR, so the visiting order does
//     not matter) and stay in registers;
//  4. each kept entry's place in its row is the number of set bits before its own (a prefix count
//     per word, a popcount inside it): ascending index, the reference's order.
// Bound by the VALU instructions it issues and the latency of its loads.  Cell::diff is about 60 FP64
// operations; on every candidate and again on every set bit (a lane per bitmap word, most lanes idle) the
// search took 18.0 us on 4096 atoms (2 species, rc 6) and 205 us on 16 x 4096 atoms (rc 6.5); with the filter
// 11 us and 104 us (744 instead of 1516 VALU instructions per centre of the latter).
//
// The filter must keep everything Cell::diff would.  A cell-list structure has every height h > 2 rc: its last image
// shell is 0, so V / (|Rv0| |Rv1|) > 2 rc over the two longest vectors, and every height V / |Ri x Rj| is at least that.  An
// entry within rc then has fractional components |f| <= rc / h < 1/2 and is the image that rounding picks; the FP32
// coordinates (in [0, 1], error 2^-25) put the distance off by less than 4e-7 ||R||_F, and the filter adds
// 1e-6 ||R||_F.  Where some rc / h is within 1e-4 of 1/2 the rounding could take the other image, and
// where a row could hold more than the register batches (maxp > 192) or the filter lists more than they
// hold, every candidate takes Cell::diff and the kept set is read out of the bitmap instead.
// LDS: bitmap, one 32-bit word per 32 atoms of the largest cell-list structure (nwords_max); 16-bit prefix
// counts per word.
constexpr int kNeighList = 2 * kWave;  // two register batches
struct NeighEntry {  // a candidate's Cell::diff, j < 0 when it is not kept
    double x, y, z, d2;
    int j, t;
};
__global__ __launch_bounds__(kWave) void k_neigh_cells_bits(
    const DevStruc* __restrict__ S, const int* __restrict__ atom_struc, const double* __restrict__ pos,
    const int* __restrict__ type, int ncell, const int* __restrict__ atom_bin,
    const int* __restrict__ bin_start, const float4* __restrict__ bin_pos, int one_struc, double rc2, int maxp,
    int* __restrict__ cnt, int* __restrict__ nbr_j, int* __restrict__ nbr_meta, double4* __restrict__ nbr_r,
    unsigned short* __restrict__ row_tab, unsigned short* __restrict__ nbr_key, int nwords_max, PassCounters pc) {
    extern __shared__ unsigned int lds_bits[];
    clear_counters(pc);
    unsigned short* pre = reinterpret_cast<unsigned short*>(lds_bits + nwords_max);
    __shared__ int list[kNeighList];
    // centres in the XCD-local order of the cell-list atoms in bin order: the blocks of one XCD
    // cover one contiguous, spatially compact run of centres, whose candidates' coordinates and bin
    // lists they then share in that XCD's L2 (the centre a block computes does not change any row)
    const int slot = xcd_slot(ncell);
    if (slot < 0) return;
    const float4 own = bin_pos[slot];
    const int i = __builtin_amdgcn_readfirstlane(__float_as_int(own.w));
    const DevStruc& s = S[one_struc ? 0 : atom_struc[i]];
    const int lane = threadIdx.x;
    const int nwords = (s.natoms + 31) >> 5;
    for (int w = lane; w < nwords; w += kWave) lds_bits[w] = 0u;
    const double xi = pos[3 * i], yi = pos[3 * i + 1], zi = pos[3 * i + 2];
    const int nb0 = s.nbin[0], nb1 = s.nbin[1], nb2 = s.nbin[2];
    const unsigned myb = (unsigned)(atom_bin[i] - s.bin0), byx = myb / (unsigned)nb2, bx_ = byx / (unsigned)nb1;
    const int bz = (int)(myb - byx * nb2), by = (int)(byx - bx_ * nb1), bx = (int)bx_;
    // lane r owns run r: an (x, y) pair of neighbouring bins (an axis with fewer than 3 bins is covered
    // once) and one of the one or two stretches of bins along z
    const int n0 = min(nb0, 3), n1 = min(nb1, 3);
    const int nz = nb2 > 3 && (bz == 0 || bz == nb2 - 1) ? 2 : 1;
    const int nruns = n0 * n1 * nz;
    int first = 0, rcount = 0;
    if (lane < nruns) {
        const int hf = nz == 2 ? (lane & 1) : 0, xy = nz == 2 ? (lane >> 1) : lane;
        const int ox = (xy >= n1) + (xy >= 2 * n1), oy = xy - ox * n1;
        int cx = ox, cy = oy, z0, z1;
        if (nb0 >= 3) {
            cx = bx + ox - 1;
            cx = cx < 0 ? cx + nb0 : (cx >= nb0 ? cx - nb0 : cx);
        }
        if (nb1 >= 3) {
            cy = by + oy - 1;
            cy = cy < 0 ? cy + nb1 : (cy >= nb1 ? cy - nb1 : cy);
        }
        if (nb2 <= 3) {
            z0 = 0;
            z1 = nb2 - 1;
        } else if (nz == 1) {
            z0 = bz - 1;
            z1 = bz + 1;
        } else if (hf == 0) {  // the stretch at the low end
            z0 = 0;
            z1 = bz == 0 ? 1 : 0;
        } else {
            z0 = bz == 0 ? nb2 - 1 : nb2 - 2;
            z1 = nb2 - 1;
        }
        const int b = s.bin0 + (cx * nb1 + cy) * nb2;
        first = bin_start[b + z0];
        rcount = bin_start[b + z1 + 1] - first;
    }
    int ncand;
    const int rfirst = wave_excl_scan(rcount, lane, ncand);  // first flat candidate of run `lane`
    // The bin-order slot of flat candidate c = c0 + lane, for chunks c0 taken in order: the runs that start in
    // the chunk are walked (the same for every lane), each taking over the candidates from its start on;
    // empty runs are taken over by the next one.  run: the last run that starts at or before the chunk.
    const int shift = first - rfirst;
    int run = 0;
    auto chunk_slot = [&](int c0) {
        const int c = c0 + lane;
        int d = __builtin_amdgcn_readlane(shift, run);
        while (run + 1 < nruns) {
            const int f = __builtin_amdgcn_readlane(rfirst, run + 1);
            if (f > c0 + kWave - 1) break;
            ++run;
            d = c >= f ? __builtin_amdgcn_readlane(shift, run) : d;
        }
        return c < ncand ? c + d : slot;  // past the list: any valid slot
    };
    int nlist = 0;
    bool full = maxp > 192 || fmax(fmax(s.reach[0], s.reach[1]), s.reach[2]) > 0.4999;
    if (!full) {
        float R[9];
#pragma unroll
        for (int q = 0; q < 9; ++q) R[q] = (float)s.R[q];
        const double rlim = sqrt(rc2) + 1e-6 * s.fro;
        const float lim = (float)(rlim * rlim * (1.0 + 2e-6));
        for (int c0 = 0; c0 < ncand; c0 += kWave) {
            const int c = c0 + lane;
            const float4 v = bin_pos[chunk_slot(c0)];
            float dx = own.x - v.x, dy = own.y - v.y, dz = own.z - v.z;
            dx -= rintf(dx);
            dy -= rintf(dy);
            dz -= rintf(dz);
            const float x = R[0] * dx + R[1] * dy + R[2] * dz, y = R[3] * dx + R[4] * dy + R[5] * dz,
                        z = R[6] * dx + R[7] * dy + R[8] * dz;
            const int gj = __float_as_int(v.w);
            const bool near = c < ncand && gj != i && x * x + y * y + z * z <= lim;
            const unsigned long long m = __ballot(near);
            const int at = nlist + __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
            if (near && at < kNeighList) list[at] = gj;
            nlist += __popcll(m);
        }
        full = nlist > kNeighList;
    }
    __syncthreads();
    const int64_t row = (int64_t)i * maxp;
    const int per = (nwords + kWave - 1) / kWave;  // lanes own contiguous word ranges
    const int w0 = min(lane * per, nwords), w1 = min(w0 + per, nwords);
    if (!full) {
        auto take = [&](int p) {
            NeighEntry e{0.0, 0.0, 0.0, 0.0, -1, 0};
            if (p < nlist) {
                const int gj = list[p];
                e.t = type[gj];
                cell_diff(s, xi - pos[3 * gj], yi - pos[3 * gj + 1], zi - pos[3 * gj + 2], e.x, e.y, e.z);
                e.d2 = e.x * e.x + e.y * e.y + e.z * e.z;
                if (e.d2 <= rc2) {
                    e.j = gj - s.atom0;
                    atomicOr(&lds_bits[e.j >> 5], 1u << (e.j & 31));
                }
            }
            return e;
        };
        auto put = [&](const NeighEntry& e) {
            if (e.j < 0) return;
            const int w = e.j >> 5;
            const int p = pre[w] + __popc(lds_bits[w] & ((1u << (e.j & 31)) - 1u));
            const double d = sqrt(e.d2);
            // one image per j: it is the minimum image when below ||R||_F (neighbor.cpp:132-140)
            if (p < maxp)
                put_entry(row + p, e.j, 0, e.t, d < s.fro, e.x, e.y, e.z, d, nbr_j, nbr_key, nbr_meta, nbr_r);
        };
        const NeighEntry e0 = take(lane);
        NeighEntry e1{0.0, 0.0, 0.0, 0.0, -1, 0};
        if (nlist > kWave) e1 = take(kWave + lane);
        __syncthreads();
        int mine = 0;
        for (int w = w0; w < w1; ++w) mine += __popc(lds_bits[w]);
        int kept;
        int at = wave_excl_scan(mine, lane, kept);
        for (int w = w0; w < w1; ++w) {
            pre[w] = (unsigned short)at;
            at += __popc(lds_bits[w]);
        }
        __syncthreads();
        put(e0);
        if (nlist > kWave) put(e1);
        if (lane < kRowTab) {  // the row's index table: set bits before each slot's first atom
            const int j = lane * row_tab_width(s.natoms), w = j >> 5;
            const int p = j < s.natoms ? pre[w] + __popc(lds_bits[w] & ((1u << (j & 31)) - 1u)) : kept;
            row_tab[(int64_t)i * kRowTab + lane] = (unsigned short)min(p, maxp);
        }
        if (lane == 0) cnt[i] = kept;
        return;
    }
    run = 0;
    for (int c0 = 0; c0 < ncand; c0 += kWave) {
        const int c = c0 + lane, sl = chunk_slot(c0);
        if (c < ncand) {
            const int gj = __float_as_int(bin_pos[sl].w);
            if (gj != i) {
                double rx, ry, rz;
                cell_diff(s, xi - pos[3 * gj], yi - pos[3 * gj + 1], zi - pos[3 * gj + 2], rx, ry, rz);
                if (rx * rx + ry * ry + rz * rz <= rc2) {
                    const int lj = gj - s.atom0;
                    atomicOr(&lds_bits[lj >> 5], 1u << (lj & 31));
                }
            }
        }
    }
    __syncthreads();
    int mine = 0;
    for (int w = w0; w < w1; ++w) mine += __popc(lds_bits[w]);
    int kept;
    int at = wave_excl_scan(mine, lane, kept);
    const int tw = row_tab_width(s.natoms);
    for (int w = w0; w < w1; ++w) {
        unsigned int m = lds_bits[w];
        // slots of the row's index table whose first atom is among this word's 32 (the bits before it)
        for (int q = ((w << 5) + tw - 1) / tw; q < kRowTab && q * tw < (w << 5) + 32; ++q)
            row_tab[(int64_t)i * kRowTab + q] =
                (unsigned short)min(at + __popc(m & ((1u << (q * tw - (w << 5))) - 1u)), maxp);
        while (m) {
            const int bit = __ffs(m) - 1;
            m &= m - 1;
            if (at < maxp) {
                const int lj = (w << 5) + bit, gj = s.atom0 + lj;
                double rx, ry, rz;
                cell_diff(s, xi - pos[3 * gj], yi - pos[3 * gj + 1], zi - pos[3 * gj + 2], rx, ry, rz);
                const double d = sqrt(rx * rx + ry * ry + rz * rz);
                put_entry(row + at, lj, 0, type[gj], d < s.fro, rx, ry, rz, d, nbr_j, nbr_key, nbr_meta, nbr_r);
            }
            ++at;
        }
    }
    if (lane < kRowTab && lane * tw >= nwords * 32) row_tab[(int64_t)i * kRowTab + lane] = (unsigned short)min(kept, maxp);
    if (lane == 0) cnt[i] = kept;
}

// Largest neighbour count of the pass (the row-overflow check).  A few hundred blocks each
// fold a strided slice and issue one atomicMax: the per-centre kernels do not contend for
// one address.
__global__ __launch_bounds__(256) void k_count_max(const int* __restrict__ cnt, int n, int* __restrict__ maxcnt) {
    int m = 0;
    for (int t = blockIdx.x * 256 + threadIdx.x; t < n; t += gridDim.x * 256) m = max(m, cnt[t]);
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) m = max(m, __shfl_xor(m, o, kWave));
    __shared__ int wm[256 / kWave];
    if ((threadIdx.x & (kWave - 1)) == 0) wm[threadIdx.x / kWave] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 256 / kWave; ++w) m = max(m, wm[w]);
        atomicMax(maxcnt, m);
    }
}

}  // namespace atomnn

#include "engine.hpp"

namespace atomnn {

hipError_t launch_count_max(const int* cnt, int n, int* maxcnt, hipStream_t st);

hipError_t launch_neighbors(const NeighborArgs& a, hipStream_t st) {
    hipError_t e;
    const PassCounters pc{a.maxcnt, a.work};
    if (a.ncell > 0) {
        if (a.ntot <= (a.nstruc == 1 ? kBinsSmallAtoms : kBinsSmallAtoms / 2) && a.nbins <= kBinsSmallBins) {
            if (a.nstruc == 1)
                hipLaunchKernelGGL(k_bins_small<true>, dim3(1), dim3(1024), 0, st, a.S, a.atom_struc, a.pos, a.ntot,
                                   a.nbins, a.atom_bin, a.bin_start, a.bin_atoms, a.bin_pos);
            else
                hipLaunchKernelGGL(k_bins_small<false>, dim3(1), dim3(1024), 0, st, a.S, a.atom_struc, a.pos, a.ntot,
                                   a.nbins, a.atom_bin, a.bin_start, a.bin_atoms, a.bin_pos);
        } else {
            const dim3 grid((a.ntot + 255) / 256);
            hipLaunchKernelGGL(k_bin_atoms, grid, dim3(256), 0, st, a.S, a.atom_struc, a.pos, a.ntot, a.atom_bin,
                               a.bin_count, a.bin_rank);
            hipLaunchKernelGGL(k_bin_scan, dim3(1), dim3(1024), 0, st, a.bin_count, a.bin_start, a.nbins);
            hipLaunchKernelGGL(k_fill_bins, grid, dim3(256), 0, st, a.S, a.atom_struc, a.pos, a.atom_bin, a.ntot,
                               a.bin_start, a.bin_rank, a.bin_atoms, a.bin_pos);
        }
        const size_t bits_lds = (size_t)((a.cell_natoms_max + 31) / 32) * 4;
        if (bits_lds <= 32768) {  // the bitmap, then its prefix counts (16 bits per word)
            hipLaunchKernelGGL(k_neigh_cells_bits, dim3(xcd_grid(a.ncell)), dim3(kWave),
                               bits_lds + (bits_lds / 2 + 3) / 4 * 4, st, a.S, a.atom_struc, a.pos, a.type, a.ncell,
                               a.atom_bin, a.bin_start, a.bin_pos, a.nstruc == 1, a.rc2, a.maxp, a.cnt, a.nbr_j,
                               a.nbr_meta, a.nbr_r, a.row_tab, a.nbr_key, (int)(bits_lds / 4), pc);
        } else {  // very large structures: sort the kept candidates instead
            int n2cap = 1;
            while (n2cap < a.maxp) n2cap <<= 1;
            const size_t lds = (size_t)a.maxp * 32 + (size_t)a.maxp * 4 + (size_t)n2cap * 8;
            hipLaunchKernelGGL(k_neigh_cells, dim3(a.ncell), dim3(kWave), lds, st, a.S, a.atom_struc, a.pos, a.type,
                               a.cell_centres, a.atom_bin, a.bin_start, a.bin_atoms, a.rc2, a.maxp, n2cap, a.cnt,
                               a.nbr_j, a.nbr_meta, a.nbr_r, a.row_tab, a.nbr_key, pc);
        }
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    if (a.npair > 0) {
        if (a.npair <= kPairCentres)
            hipLaunchKernelGGL(k_neigh_allpairs<4>, dim3(a.npair), dim3(kWave * 4), 0, st, a.S, a.atom_struc, a.pos, a.type,
                               a.pair_centres, a.rc2, a.maxp, a.cnt, a.nbr_j, a.nbr_meta, a.nbr_r, a.row_tab, a.nbr_key, pc);
        else
            hipLaunchKernelGGL(k_neigh_allpairs<1>, dim3(a.npair), dim3(kWave), 0, st, a.S, a.atom_struc, a.pos, a.type,
                               a.pair_centres, a.rc2, a.maxp, a.cnt, a.nbr_j, a.nbr_meta, a.nbr_r, a.row_tab, a.nbr_key, pc);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    if (a.ntot > 0 && a.count_max) return launch_count_max(a.cnt, a.ntot, a.maxcnt, st);
    return hipGetLastError();
}

hipError_t launch_count_max(const int* cnt, int n, int* maxcnt, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_count_max, dim3(std::min((n + 255) / 256, 256)), dim3(256), 0, st, cnt, n, maxcnt);
    return hipGetLastError();
}

}  // namespace atomnn
