// Site-mode genetic relatedness matrix on the matrix cores (gfx950).
//
// For sites with at most two alleles the reference's
// genetic_relatedness_matrix(mode="site") (python/tskit/trees.py:8978-9102,
// from the divergence matrix of c/tskit/trees.c:8753-8826) reduces to
//     K = J C J / span,   C = G^T G,   J = I - 11^T / n,
// where G is the site x sample 0/1 matrix of derived alleles: the divergence
// matrix is D = a 1^T + 1 a^T - 2C (a = derived counts per sample) and the
// double centring -1/2 J D J removes the a terms exactly.  A site with more
// alleles differs between samples i and j iff d_i + d_j - d_i d_j -
// sum_a B_ai B_aj = 1 (d its any-derived row, B_a its row of allele a >= 1),
// so its rows d and B_a go into a second cross product C2 and, with
// P = 2C + C2, D = (P_ii + P_jj)/2 - P_ij and K = J P J / 2.  C and C2 are
// exact integer cross products (entries <= number of rows < 2^31), computed
// here on the matrix cores from the bits; the centring is FP64.
//
// Kernels:
//   k_geno_bits  one wavefront per chunk: the chunk sweep with a per-node
//                bitset of the samples below it (insert: OR, remove: AND-NOT);
//                each site's row is the bitset of its mutation's node.
//   k_site_bits  the same rows from the states of the state plan, whose bits
//                the plan's count kernel adds up (where the plan is usable).
//   k_sample_bits  bit rows by site -> by sample (each window's sites
//                zero-padded to a multiple of 128).
//   k_syrk       C = B B^T over the bits, upper-triangular 128x128 tiles,
//                mirrored on store.
//   k_centre     row sums, then K = (C - r_i/n - r_j/n + t/n^2) / span (FP64).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "tsg_common.h"
#include "tsg_kernels.h"
#include "tsg_launch.h"

#define WAVE 64

// --- genotype bitsets ------------------------------------------------------
// Word w of site s's bit rows from the bitsets of its mutations' nodes
// (below(node) = samples below it), following tsk_variant_decode's rule
// (genotypes.c:473-595): samples start at allele 0 and each mutation, in
// order, sets the samples below its node to its allele.  A site with at most
// two alleles gets one row, its derived allele; a site with three or more
// gets its any-derived row in gbits[s] and one row per derived allele at
// gbits[site_row2[s] + allele - 1].
template <typename Below>
__device__ __forceinline__ void site_rows(const TsgGenoArgs &a, int s, int w, int NW,
                                          Below below) {
    const int m0 = a.site_mut0[s], m1 = a.site_mut0[s + 1];
    const int r2 = a.site_row2 ? a.site_row2[s] : -1;
    if (r2 < 0) {
        uint32_t b1 = 0u;
        for (int m = m0; m < m1; m++) {
            const uint32_t b = below(a.mut_node[m]);
            b1 = (a.mut_allele[m] != 0) ? (b1 | b) : (b1 & ~b);
        }
        a.gbits[(int64_t) s * NW + w] = b1;
        return;
    }
    const int na = a.site_nalleles[s];
    uint32_t *rows = a.gbits + (int64_t) r2 * NW + w;
    for (int al = 1; al < na; al++) rows[(int64_t) (al - 1) * NW] = 0u;
    for (int m = m0; m < m1; m++) {
        const uint32_t b = below(a.mut_node[m]);
        const int al = a.mut_allele[m];
        for (int q = 1; q < na; q++) {
            uint32_t &r = rows[(int64_t) (q - 1) * NW];
            r = (q == al) ? (r | b) : (r & ~b);
        }
    }
    uint32_t d = 0u;
    for (int al = 1; al < na; al++) d |= rows[(int64_t) (al - 1) * NW];
    a.gbits[(int64_t) s * NW + w] = d;
}

__device__ void geno_bits_chunk(const TsgGenoArgs &a, int c, uint32_t *rec);

// Each workgroup owns one slab and loops over chunks blockIdx.x,
// blockIdx.x + gridDim.x, ... so the slab memory is bounded by the grid.
__global__ void __launch_bounds__(WAVE) k_geno_bits(const TsgGenoArgs a) {
    for (int c = blockIdx.x; c < a.num_chunks; c += gridDim.x) {
        __syncthreads();
        geno_bits_chunk(a, c, a.g_rec + (int64_t) blockIdx.x * a.g_stride);
    }
}

__device__ void geno_bits_chunk(const TsgGenoArgs &a, int c, uint32_t *rec) {
    const int lane = threadIdx.x;
    const int NW = a.NW;
    const int R = 1 + NW;  // parent, then NW bitset words
    const int64_t n0 = a.chunk_node0[c];
    const int nloc = (int) (a.chunk_node0[c + 1] - n0);
    auto par = [&](int u) -> int32_t & { return reinterpret_cast<int32_t &>(rec[(int64_t) u * R]); };
    auto word = [&](int u, int w) -> uint32_t & { return rec[(int64_t) u * R + 1 + w]; };

    for (int u = lane; u < nloc; u += WAVE) {
        par(u) = a.loc_parent0[n0 + u];
        for (int w = 0; w < NW; w++) word(u, w) = 0u;
    }
    __syncthreads();
    // every sample's bit, up its root path in the start tree
    for (int j = lane; j < a.num_samples; j += WAVE) {
        const uint32_t bit = 1u << (j & 31);
        const int w = j >> 5;
        for (int u = j; u >= 0; u = par(u)) atomicOr(&word(u, w), bit);
    }
    __syncthreads();
    const int t0 = a.chunk_tree0[c], t1 = a.chunk_tree0[c + 1];
    for (int t = t0; t < t1; t++) {
        if (t > t0) {
            const int64_t e0 = a.tr_off[t], e1 = a.tr_off[t + 1];
            const int64_t nrem = a.tr_nrem[t];
            for (int64_t e = e0; e < e1; e++) {
                const bool ins = (e - e0) >= nrem;
                const int u = a.ev_child[e], v = a.ev_parent[e];
                // lanes own words w = lane, lane + 64, ...; a chunk's child
                // bitset is re-read per ancestor from the same lane's word
                if (lane == 0) par(u) = ins ? v : TSG_NULL;
                __syncthreads();
                for (int w = lane; w < NW; w += WAVE) {
                    const uint32_t xc = word(u, w);
                    if (xc == 0u) continue;
                    for (int p = v; p >= 0; p = par(p)) {
                        word(p, w) = ins ? (word(p, w) | xc) : (word(p, w) & ~xc);
                    }
                }
                __syncthreads();
            }
        }
        const int s0 = a.tree_site0[t], s1 = a.tree_site0[t + 1];
        for (int s = s0; s < s1; s++) {
            for (int w = lane; w < NW; w += WAVE) {
                site_rows(a, s, w, NW, [&](int node) { return word(node, w); });
            }
        }
    }
}

// --- genotype bitsets on the hot plan ---------------------------------------
// One workgroup per (chunk, block of WB bitset words = 32*WB samples): the
// chunk's hot slots hold bitsets of the samples below them in LDS.  Seeding:
// each sample of the block sets its bit in its nearest hot ancestor-or-self,
// then the hot forest's levels OR upward, deepest first.  Events: lane w owns
// word w of every slot, so an edge insertion ORs the child's word into each
// node of its root path and a removal clears it (the child's samples lie
// below every path node and nowhere else among them) -- no lane reads
// another lane's words, so the event loop needs no barrier.  Each site's row
// rows come from its mutations' node bitsets (site_rows).  Grid: 8 * ceil(C / 8) x blocks.
//
// GENO: the genotype decode instead (tsk_variant_decode, genotypes.c:473-595):
// every sample starts at allele 0 and each mutation of the site, in order,
// sets the samples below its node to its allele index; lane w writes the 32
// int32 genotypes of its word.  Missing data is marked afterwards from the
// host's list of isolated samples (k_mark_missing).
template <bool GENO>
__global__ void __launch_bounds__(WAVE) k_geno_hot(const TsgGenoArgs a) {
    extern __shared__ uint32_t bits[];
    const int C = a.num_chunks;
    const int per = (C + 7) / 8;
    const int c = (blockIdx.x % 8) * per + blockIdx.x / 8;  // XCD-contiguous chunks
    if (c >= C) return;
    const int lane = threadIdx.x;
    const int WB = a.WB;
    const int w0 = blockIdx.y * WB;                // first word of the block
    const int nwb = min(WB, a.NW - w0);            // words in this block
    const int64_t s0 = a.chunk_node0[c];
    const int S = (int) (a.chunk_node0[c + 1] - s0);
    for (int i = lane; i < S * WB; i += WAVE) bits[i] = 0u;
    __syncthreads();
    const uint16_t *ss = a.sample_slot + (int64_t) (c / TSG_SS_CB) * a.num_samples * TSG_SS_CB +
                         c % TSG_SS_CB;
    const int j0 = w0 * 32, j1 = min(a.num_samples, (w0 + nwb) * 32);
    for (int j = j0 + lane; j < j1; j += WAVE) {
        const unsigned h = ss[(int64_t) j * TSG_SS_CB];
        if (h != TSG_NO_SLOT) atomicOr(&bits[h * WB + ((j >> 5) - w0)], 1u << (j & 31));
    }
    __syncthreads();
    const int32_t *lev = a.lev_slot0 + a.chunk_lev0[c];
    const int nlev = (int) (a.chunk_lev0[c + 1] - a.chunk_lev0[c]) - 1;
    for (int l = 0; l + 1 < nlev; l++) {
        const int h0 = lev[l], h1 = lev[l + 1];
        for (int idx = lane; idx < (h1 - h0) * nwb; idx += WAVE) {
            const int h = h0 + idx / nwb, w = idx % nwb;
            const int p = a.slot_par[s0 + h];
            const uint32_t v = bits[h * WB + w];
            if (p >= 0 && v != 0u) atomicOr(&bits[p * WB + w], v);
        }
        __syncthreads();
    }
    const int t0 = a.chunk_tree0[c], t1 = a.chunk_tree0[c + 1];
    for (int t = t0; t < t1; t++) {
        if (t > t0) {
            const int64_t e0 = a.tr_off[t], e1 = a.tr_off[t + 1];
            const int64_t nrem = a.tr_nrem[t];
            for (int64_t e = e0; e < e1; e++) {
                const bool ins = (e - e0) >= nrem;
                const int u = a.ev_child[e];
                const int64_t p0 = a.ev_path0[e], p1 = a.ev_path0[e + 1];
                if (lane < nwb) {
                    const uint32_t xc = bits[u * WB + lane];
                    if (xc != 0u) {
                        for (int64_t q = p0; q < p1; q++) {
                            uint32_t &b = bits[a.path[q] * WB + lane];
                            b = ins ? (b | xc) : (b & ~xc);
                        }
                    }
                }
            }
        }
        const int sa = a.tree_site0[t], sb = a.tree_site0[t + 1];
        for (int s = sa; s < sb; s++) {
            const int m0 = a.site_mut0[s], m1 = a.site_mut0[s + 1];
            if constexpr (GENO) {
                if (lane < nwb) {
                    int32_t g[32];
#pragma unroll
                    for (int b = 0; b < 32; b++) g[b] = 0;
                    for (int m = m0; m < m1; m++) {
                        const uint32_t mask = bits[a.mut_node[m] * WB + lane];
                        const int32_t al = a.mut_allele[m];
#pragma unroll
                        for (int b = 0; b < 32; b++) {
                            if ((mask >> b) & 1u) g[b] = al;
                        }
                    }
                    const int j0w = (w0 + lane) * 32;
                    int32_t *row = a.geno + (int64_t) s * a.num_samples + j0w;
                    const int nb = min(32, a.num_samples - j0w);
#pragma unroll
                    for (int b = 0; b < 32; b++) {
                        if (b < nb) row[b] = g[b];
                    }
                }
            } else {
                if (lane < nwb) {
                    site_rows(a, s, w0 + lane, a.NW,
                              [&](int node) { return bits[node * WB + lane]; });
                }
            }
        }
    }
}

// --- genotype bits on the state plan ----------------------------------------------
// The samples below a state as RW words: the states' counts (tsg_states.hip)
// with a word of 32 samples in place of a column, since the sets that a state
// sums are disjoint and so add up without carries.  All states of a level at
// once; the chunk walk (k_geno_hot) is a chain of dependent LDS updates per
// chunk.  (2500 samples, 177000 states of 79 words, 56000 sites: 383 us by
// chunks, 50 us of counts and 16 of rows here.)

// Rows 0 (no samples) and 1 + s (sample s), 4 words a thread.
__global__ void __launch_bounds__(256) k_bits_seed(uint32_t *x, int RW, int64_t n) {
    const int64_t i = (int64_t) blockIdx.x * 256 + threadIdx.x;
    const int64_t r = i / (RW / 4);
    const int w = (int) (i % (RW / 4)) * 4;
    if (r > n) return;
    uint32_t v[4] = {0, 0, 0, 0};
    if (r > 0 && (int) ((r - 1) >> 7) == w / 4) v[((r - 1) >> 5) & 3] = 1u << ((r - 1) & 31);
    *reinterpret_cast<uint4 *>(x + r * RW + w) = make_uint4(v[0], v[1], v[2], v[3]);
}

// Thread per (site, word): the site's bit rows from its mutations' states.
__global__ void __launch_bounds__(256) k_site_bits(const TsgGenoArgs a, int64_t b0) {
    const int64_t i = (b0 + blockIdx.x) * 256 + threadIdx.x;
    const int64_t site = i / a.NW;
    if (site >= a.num_sites) return;
    const int w = (int) (i % a.NW);
    site_rows(a, (int) site, w, a.NW, [&](int st) { return a.x[(int64_t) st * a.RW + w]; });
}

// Genotypes as G, site after site, 16 bytes a thread: cells q .. of one site
// or, at a site's end, of the next too.  A cell's value is the allele of the
// last of its site's mutations with the sample below it.
template <typename G>
__global__ void __launch_bounds__(256) k_genotypes(const TsgGenoArgs a, G *geno, int64_t cells) {
    constexpr int CELLS = 16 / (int) sizeof(G);
    const int64_t q = ((int64_t) blockIdx.x * 256 + threadIdx.x) * CELLS;
    if (q >= cells) return;
    const int n = a.num_samples;
    int64_t site = q / n;
    int j = (int) (q % n);
    uint32_t v[4] = {0, 0, 0, 0};
    for (int done = 0; done < CELLS && site < a.num_sites; site++, j = 0) {
        const int count = min(CELLS - done, n - j);
        const uint32_t here = ((1u << count) - 1u) << done;
        const int w = j >> 5;
        for (int m = a.site_mut0[site]; m < a.site_mut0[site + 1]; m++) {
            const uint32_t *row = a.x + (int64_t) a.mut_node[m] * a.RW;
            const uint32_t hi = w + 1 < a.NW ? row[w + 1] : 0u;
            // bits of samples j .. as cells done ..
            const uint32_t b = ((uint32_t) ((((uint64_t) hi << 32) | row[w]) >> (j & 31)) << done) & here;
            const uint32_t al = (uint32_t) a.mut_allele[m];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                if constexpr (sizeof(G) == 1) {
                    // 4 bits to 4 bytes of ones
                    const uint32_t on = ((((b >> (4 * k)) & 15u) * 0x00204081u) & 0x01010101u) * 255u;
                    v[k] = (v[k] & ~on) | (on & (al * 0x01010101u));
                } else {
                    if ((b >> k) & 1u) v[k] = al;
                }
            }
        }
        done += count;
    }
    *reinterpret_cast<uint4 *>(geno + q) = make_uint4(v[0], v[1], v[2], v[3]);
}

// --- bit rows by site -> by sample --------------------------------------------
// bits: [n_pad x KW] words, bit k of sample j's row its genotype at column k;
// site_of_col maps a padded column to its row of gbits (-1: zeros).  A wave
// takes 256 columns of 128 samples: per 64 columns each lane reads one site's
// 4 words and 128 ballots turn them; each lane then holds 32 bytes of two
// samples' rows.  Bound by its ballots, about 2 instructions a sample and 64
// sites (2500 samples x 56000 sites: 48 us; the int8 expansion this replaced
// wrote 143 MB, 66 us).
__global__ void __launch_bounds__(256) k_sample_bits(const uint32_t *gbits, int NW,
                                                     const int32_t *site_of_col, int64_t Kp,
                                                     uint32_t *bits) {
    const int lane = threadIdx.x % WAVE;
    const int64_t k0 = ((int64_t) blockIdx.x * 4 + threadIdx.x / WAVE) * 256;
    if (k0 >= Kp) return;
    const int w0 = blockIdx.y * 4;
    unsigned long long mine[2][4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int64_t k = k0 + q * 64 + lane;
        const int64_t site = k < Kp ? site_of_col[k] : -1;
#pragma unroll
        for (int h = 0; h < 4; h++) {
            const uint32_t v = (site >= 0 && w0 + h < NW) ? gbits[site * NW + w0 + h] : 0u;
            unsigned long long m = 0;
#pragma unroll
            for (int b = 0; b < 32; b++) {
                const unsigned long long all = __ballot((v >> b) & 1u);
                if (lane % 32 == b) m = all;
            }
            // word h's samples are 32 h + b: lanes 0-31 keep words 0 and 2,
            // lanes 32-63 words 1 and 3
            if (lane / 32 == h % 2) mine[h / 2][q] = m;
        }
    }
    const int64_t KW = Kp / 32;
#pragma unroll
    for (int r = 0; r < 2; r++) {
        uint32_t *row = bits + ((int64_t) blockIdx.y * 128 + r * 64 + lane) * KW + k0 / 32;
#pragma unroll
        for (int q = 0; q < 4; q += 2) {
            if (k0 + q * 64 < Kp) {  // (Kp is a multiple of 128)
                *reinterpret_cast<uint4 *>(row + 2 * q) =
                    make_uint4((uint32_t) mine[r][q], (uint32_t) (mine[r][q] >> 32),
                               (uint32_t) mine[r][q + 1], (uint32_t) (mine[r][q + 1] >> 32));
            }
        }
    }
}

// --- cross products of the bits ------------------------------------------------
typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));

#define BT 128  // output tile
// columns a wave may sum in FP32: whole numbers are exact below this
#define SYRK_MOST ((int64_t) 1 << 24)

// 32 bits as 32 FP4 values (E2M1: 1.0 is 0b0010).  The order of the values
// along k does not matter, being the same for both operands.
__device__ __forceinline__ v8i fp4(uint32_t b) {
    v8i r = {};
    r[0] = (int) ((b << 1) & 0x22222222u);
    r[1] = (int) (b & 0x22222222u);
    r[2] = (int) ((b >> 1) & 0x22222222u);
    r[3] = (int) ((b >> 2) & 0x22222222u);
    return r;
}

// One workgroup (4 waves) per upper-triangular 128x128 tile of one window and
// part of its columns.  A genotype is one bit, so the bits are what is read
// (a wave's 256 columns of 256 samples: 8 KB, straight into registers), and
// FP4 matrix instructions multiply them: products of 0 and 1, summed in FP32,
// are exact up to SYRK_MOST columns a wave.  Every wave computes the whole
// tile over a quarter of the columns, 4 x 4 tiles of 32 x 32, so that 8
// expansions (7 instructions each) feed 16 matrix instructions; the four
// waves' sums are added in LDS, as integers.
// (2500 samples x 56000 sites: 114 us; 721 with int8 operands staged in LDS,
// each wave a quarter of the tile.  5000 x 199000: 1322 us, 4693 before.)
__global__ void __launch_bounds__(256, 1) k_syrk(const uint32_t *bits, int64_t KW, int n_pad,
                                                 const int64_t *win_k0, const int64_t *win_k1,
                                                 int tiles_per_dim, bool add, int32_t *C) {
    extern __shared__ float part[];  // [4 waves][4 tiles][16][64]
    const int w = blockIdx.y;  // window
    // invert the upper-triangular tile index
    int t = blockIdx.x, ti = 0;
    int rowlen = tiles_per_dim;
    while (t >= rowlen) {
        t -= rowlen;
        ti++;
        rowlen--;
    }
    const int tj = ti + t;
    const int i0 = ti * BT, j0 = tj * BT;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    v16f acc[4][4];
#pragma unroll
    for (int a = 0; a < 4; a++)
#pragma unroll
        for (int b = 0; b < 4; b++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[a][b][r] = 0.0f;
    // this wave's chunks of 8 words (256 columns) of the window
    const int64_t kbeg = win_k0[w] / 32, kend = win_k1[w] / 32;
    const int64_t chunks = (kend - kbeg + 7) / 8;
    const int64_t parts = (int64_t) gridDim.z * 4, p = (int64_t) blockIdx.z * 4 + wave;
    const int64_t c0 = chunks * p / parts, c1 = chunks * (p + 1) / parts;
    const uint32_t *ra = bits + (int64_t) (i0 + (lane & 31)) * KW;
    const uint32_t *rb = bits + (int64_t) (j0 + (lane & 31)) * KW;
    uint4 na[4], nb[4];
    auto fetch = [&](int64_t c) {  // lanes 0-31 words 0-3 of the chunk, 32-63 words 4-7
        const int64_t k = kbeg + c * 8 + 4 * (lane >> 5);
        const bool in = c < c1 && k < kend;
#pragma unroll
        for (int a = 0; a < 4; a++) {
            na[a] = in ? *reinterpret_cast<const uint4 *>(ra + a * 32 * KW + k)
                       : make_uint4(0, 0, 0, 0);
            nb[a] = in ? *reinterpret_cast<const uint4 *>(rb + a * 32 * KW + k)
                       : make_uint4(0, 0, 0, 0);
        }
    };
    fetch(c0);
    for (int64_t c = c0; c < c1; c++) {
        uint4 ca[4], cb[4];
#pragma unroll
        for (int a = 0; a < 4; a++) ca[a] = na[a], cb[a] = nb[a];
        fetch(c + 1);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            v8i af[4], bf[4];
#pragma unroll
            for (int a = 0; a < 4; a++) {
                af[a] = fp4(q == 0 ? ca[a].x : q == 1 ? ca[a].y : q == 2 ? ca[a].z : ca[a].w);
                bf[a] = fp4(q == 0 ? cb[a].x : q == 1 ? cb[a].y : q == 2 ? cb[a].z : cb[a].w);
            }
#pragma unroll
            for (int a = 0; a < 4; a++)
#pragma unroll
                for (int b = 0; b < 4; b++)
                    // (formats 4: FP4; scales 0: unscaled)
                    acc[a][b] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
                        af[a], bf[b], acc[a][b], 4, 4, 0, 0, 0, 0);
        }
    }
    int32_t *Cw = C + (int64_t) w * n_pad * n_pad;
#pragma unroll
    for (int a = 0; a < 4; a++) {
        // row of tiles a: every wave's sums into LDS, wave b adds up tile b
        if (a > 0) __syncthreads();
#pragma unroll
        for (int b = 0; b < 4; b++)
#pragma unroll
            for (int r = 0; r < 16; r++)
                part[((wave * 4 + b) * 16 + r) * WAVE + lane] = acc[a][b][r];
        __syncthreads();
        const int col = j0 + wave * 32 + (lane & 31);
#pragma unroll
        for (int r4 = 0; r4 < 4; r4++) {
            const int row = i0 + a * 32 + r4 * 8 + (lane >> 5) * 4;
            int32_t v[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                v[r] = 0;
#pragma unroll
                for (int u = 0; u < 4; u++)
                    v[r] += (int32_t) part[((u * 4 + wave) * 16 + r4 * 4 + r) * WAVE + lane];
            }
            int32_t *down = Cw + (int64_t) row * n_pad + col;
            int32_t *across = Cw + (int64_t) col * n_pad + row;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                if (add) {
                    atomicAdd(down + (int64_t) r * n_pad, v[r]);
                    if (ti != tj) atomicAdd(across + r, v[r]);
                } else {
                    down[(int64_t) r * n_pad] = v[r];
                }
            }
            if (!add && ti != tj) {
                *reinterpret_cast<int4 *>(across) = make_int4(v[0], v[1], v[2], v[3]);
            }
        }
    }
}

// --- centring (FP64) ----------------------------------------------------------
// The n selected samples (sample indexes sel[0..n)) form the matrix.
// rowsum[w][a] = sum_b C[w][sel_a][sel_b] (exact in int64); block per (a, w).
// With sites of three or more alleles the matrices take P = 2 C + C2 (C
// over the rows of the other sites, C2 over the any-derived and per-allele
// rows of those sites, C2 null when there are none): two samples differ at
// a site in (P_ii + P_jj) / 2 - P_ij sites, and the relatedness is
// J P J / 2; without C2, P = 2C and these reduce to the biallelic forms.
__device__ __forceinline__ int64_t cross(const int32_t *C, const int32_t *C2, int64_t idx) {
    return C2 ? 2 * (int64_t) C[idx] + (int64_t) C2[idx] : (int64_t) C[idx];
}

__global__ void __launch_bounds__(256) k_rowsum(const int32_t *C, const int32_t *C2,
                                                const int32_t *sel, int n, int n_pad,
                                                int64_t *rowsum) {
    __shared__ long long part[256];
    const int i = blockIdx.x, w = blockIdx.y;
    const int64_t row = ((int64_t) w * n_pad + sel[i]) * n_pad;
    long long s = 0;
    for (int j = threadIdx.x; j < n; j += 256) s += cross(C, C2, row + sel[j]);
    part[threadIdx.x] = s;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if ((int) threadIdx.x < h) part[threadIdx.x] += part[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0) rowsum[(int64_t) w * n + i] = part[0];
}

// K[w][i][j] = (C_ij - r_i/n - r_j/n + t/n^2) * scale[w], t = sum_i r_i.
__global__ void __launch_bounds__(256) k_centre(const int32_t *C, const int32_t *C2,
                                                const int32_t *sel, const int64_t *rowsum, int n,
                                                int n_pad, const double *scale, double *K) {
    const int64_t gid = (int64_t) blockIdx.x * 256 + threadIdx.x;
    const int w = blockIdx.y;
    if (gid >= (int64_t) n * n) return;
    const int i = (int) (gid / n), j = (int) (gid % n);
    const int64_t *rs = rowsum + (int64_t) w * n;
    // grand total, recomputed per thread from the row sums would be O(n);
    // it is passed through rowsum[n * W + w] by the host-side launcher
    const double t = (double) rowsum[(int64_t) gridDim.y * n + w];
    const double dn = (double) n;
    const double cij = (double) cross(C, C2, ((int64_t) w * n_pad + sel[i]) * n_pad + sel[j]);
    const double v = cij - (double) rs[i] / dn - (double) rs[j] / dn + t / (dn * dn);
    K[(int64_t) w * n * n + gid] = (C2 ? 0.5 * v : v) * scale[w];
}

// Site divergence of singleton sets from the same cross products: samples i
// and j differ at a 0/1 site iff g_i + g_j - 2 g_i g_j = 1, so the count of
// differing sites is C_ii + C_jj - 2 C_ij (0 on the diagonal), times the
// window's span scale (trees.c:8753-8900 with sets of one sample).
__global__ void __launch_bounds__(256) k_divergence(const int32_t *C, const int32_t *C2,
                                                    const int32_t *sel, int n, int n_pad,
                                                    const double *scale, double *D) {
    const int64_t gid = (int64_t) blockIdx.x * 256 + threadIdx.x;
    const int w = blockIdx.y;
    if (gid >= (int64_t) n * n) return;
    const int i = (int) (gid / n), j = (int) (gid % n);
    const int64_t base = (int64_t) w * n_pad * n_pad;
    const int64_t si = sel[i], sj = sel[j];
    double v = 0.0;
    if (i != j) {
        const int64_t pii = cross(C, C2, base + si * n_pad + si);
        const int64_t pjj = cross(C, C2, base + sj * n_pad + sj);
        const int64_t pij = cross(C, C2, base + si * n_pad + sj);
        // without C2: C_ii + C_jj - 2 C_ij; with it (P_ii + P_jj) / 2 - P_ij
        // (P_ii is even: a site's any-derived row and its allele rows count
        // each carrier once each)
        v = C2 ? (double) ((pii + pjj) / 2 - pij) : (double) (pii + pjj - 2 * pij);
    }
    D[(int64_t) w * n * n + gid] = v * scale[w];
}

// Divergence between sample sets from the pairwise matrix D [W x n x n] of
// their samples (set k = rows off[k] .. off[k + 1]): one workgroup per
// (A, B, window) sums D over A x B in a fixed order, then divides by the
// number of pairs, |A||B| (A != B) or |A|(|A| - 1) when that is not zero
// (trees.c:8876-8899; the reference counts a pair within one set twice, as
// D's two triangles do).
__global__ void __launch_bounds__(256) k_set_divergence(const double *D, int n,
                                                        const int32_t *off, int nsets,
                                                        double *out) {
    __shared__ double part[256];
    const int A = blockIdx.x / nsets, B = blockIdx.x % nsets;
    const int w = blockIdx.y;
    const int a0 = off[A], a1 = off[A + 1], b0 = off[B], b1 = off[B + 1];
    const int nb = b1 - b0;
    const int64_t cnt = (int64_t) (a1 - a0) * nb;
    const double *Dw = D + (int64_t) w * n * n;
    double s = 0.0;
    for (int64_t t = threadIdx.x; t < cnt; t += 256) {
        const int i = a0 + (int) (t / nb), j = b0 + (int) (t % nb);
        s += Dw[(int64_t) i * n + j];
    }
    part[threadIdx.x] = s;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if ((int) threadIdx.x < h) part[threadIdx.x] += part[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const double na = (double) (a1 - a0), nbd = (double) nb;
        const double denom = (A == B) ? na * (na - 1) : na * nbd;
        const double v = part[0];
        out[((int64_t) w * nsets + A) * nsets + B] = (A == B && denom == 0) ? v : v / denom;
    }
}

// grand totals: one workgroup per window sums its n row sums (exact int64,
// so the order of the additions does not matter)
__global__ void __launch_bounds__(256) k_total(int64_t *rowsum, int n, int W) {
    __shared__ long long part[256];
    const int w = blockIdx.x;
    long long s = 0;
    for (int i = threadIdx.x; i < n; i += 256) s += rowsum[(int64_t) w * n + i];
    part[threadIdx.x] = s;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if ((int) threadIdx.x < h) part[threadIdx.x] += part[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0) rowsum[(int64_t) W * n + w] = part[0];
}

// --- launchers ------------------------------------------------------------------
hipError_t tsg_launch_geno_bits(const TsgGenoArgs &a, hipStream_t s) {
    hipLaunchKernelGGL(k_geno_bits, dim3(a.slots), dim3(WAVE), 0, s, a);
    return hipGetLastError();
}

template <bool GENO>
hipError_t launch_geno_hot(const TsgGenoArgs &a, size_t shmem, hipStream_t s) {
    if (shmem > 65536) {
        if ((int) shmem > tsg_lds_max()) return hipErrorInvalidValue;
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&k_geno_hot<GENO>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize,
                                           tsg_lds_max());
        if (e != hipSuccess) return e;
    }
    const dim3 grid(8u * (unsigned) ((a.num_chunks + 7) / 8),
                    (unsigned) ((a.NW + a.WB - 1) / a.WB));
    hipLaunchKernelGGL((k_geno_hot<GENO>), grid, dim3(WAVE), shmem, s, a);
    return hipGetLastError();
}

hipError_t tsg_launch_geno_hot(const TsgGenoArgs &a, size_t shmem, hipStream_t s) {
    return launch_geno_hot<false>(a, shmem, s);
}

// Missing data: geno[site * n + sample] = -1 for each listed pair.
template <typename G>
__global__ void k_mark_missing(G *geno, int n, const int32_t *site, const int32_t *sample,
                               int64_t npairs) {
    const int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (i < npairs) geno[(int64_t) site[i] * n + sample[i]] = (G) -1;
}
template <typename G>
hipError_t mark_missing(G *geno, int n, const int32_t *site, const int32_t *sample,
                        int64_t npairs, hipStream_t s) {
    if (npairs == 0) return hipGetLastError();
    hipLaunchKernelGGL(k_mark_missing<G>, dim3((unsigned) ((npairs + 255) / 256)), dim3(256), 0, s,
                       geno, n, site, sample, npairs);
    return hipGetLastError();
}

hipError_t tsg_launch_genotypes(const TsgGenoArgs &a, size_t shmem, const int32_t *miss_site,
                                const int32_t *miss_sample, int64_t nmiss, hipStream_t s) {
    hipError_t e = launch_geno_hot<true>(a, shmem, s);
    if (e != hipSuccess) return e;
    return mark_missing(a.geno, a.num_samples, miss_site, miss_sample, nmiss, s);
}

hipError_t tsg_launch_bits_seed(uint32_t *x, int RW, int n, hipStream_t s) {
    const int64_t threads = (int64_t) (n + 1) * (RW / 4);
    hipLaunchKernelGGL(k_bits_seed, dim3((unsigned) ((threads + 255) / 256)), dim3(256), 0, s, x, RW,
                       (int64_t) n);
    return hipGetLastError();
}

hipError_t tsg_launch_site_bits(const TsgGenoArgs &a, hipStream_t s) {
    const int64_t threads = (int64_t) a.num_sites * a.NW;
    return tsg_in_launches((threads + 255) / 256, [&](int64_t b, unsigned count) {
        hipLaunchKernelGGL(k_site_bits, dim3(count), dim3(256), 0, s, a, b);
    });
}

template <typename G>
hipError_t launch_states_genotypes(const TsgGenoArgs &a, G *geno, const int32_t *miss_site,
                                   const int32_t *miss_sample, int64_t nmiss, hipStream_t s) {
    constexpr int CELLS = 16 / (int) sizeof(G);
    const int64_t cells = (int64_t) a.num_sites * a.num_samples;
    const int64_t threads = (cells + CELLS - 1) / CELLS;
    hipLaunchKernelGGL(k_genotypes<G>, dim3((unsigned) ((threads + 255) / 256)), dim3(256), 0, s, a,
                       geno, cells);
    return mark_missing(geno, a.num_samples, miss_site, miss_sample, nmiss, s);
}

hipError_t tsg_launch_states_genotypes(const TsgGenoArgs &a, bool narrow, const int32_t *miss_site,
                                       const int32_t *miss_sample, int64_t nmiss, hipStream_t s) {
    return narrow ? launch_states_genotypes(a, (int8_t *) a.geno, miss_site, miss_sample, nmiss, s)
                  : launch_states_genotypes(a, a.geno, miss_site, miss_sample, nmiss, s);
}

hipError_t tsg_launch_sample_bits(const uint32_t *gbits, int NW, const int32_t *site_of_col,
                                  int64_t Kp, int n_pad, uint32_t *bits, hipStream_t s) {
    dim3 grid((unsigned) ((Kp + 1023) / 1024), (unsigned) (n_pad / 128));
    hipLaunchKernelGGL(k_sample_bits, grid, dim3(256), 0, s, gbits, NW, site_of_col, Kp, bits);
    return hipGetLastError();
}

// The columns of a window are split over workgroups, which then add into
// zeroed products, where its tiles alone leave compute units idle (one
// workgroup each: its registers), each wave keeping 8 chunks of 256 columns
// or more; and where a wave's share would reach SYRK_MOST.
hipError_t tsg_launch_syrk(const uint32_t *bits, int64_t Kp, int n_pad, const int64_t *win_k0,
                           const int64_t *win_k1, int64_t most_cols, int W, int32_t *C,
                           hipStream_t s) {
    const int tpd = n_pad / BT;
    const int64_t tiles = (int64_t) tpd * (tpd + 1) / 2 * W;
    const int64_t split = std::max<int64_t>(std::min<int64_t>(256 / tiles, most_cols / (4 * 8 * 256)),
                                            most_cols / (3 * SYRK_MOST) + 1);
    const size_t shmem = 4 * 4 * 16 * WAVE * sizeof(float);
    hipError_t e;
    if (split > 1) {
        const int64_t words = (int64_t) W * n_pad * n_pad / 2;
        if ((e = tsg_launch_fill_u64((unsigned long long *) C, words, s)) != hipSuccess) return e;
    }
    hipLaunchKernelGGL(k_syrk, dim3((unsigned) (tpd * (tpd + 1) / 2), (unsigned) W, (unsigned) split),
                       dim3(256), shmem, s, bits, Kp / 32, n_pad, win_k0, win_k1, tpd, split > 1, C);
    return hipGetLastError();
}

hipError_t tsg_launch_divergence(const int32_t *C, const int32_t *C2, const int32_t *sel, int n,
                                 int n_pad, int W, const double *scale, double *D,
                                 hipStream_t s) {
    const int64_t nn = (int64_t) n * n;
    hipLaunchKernelGGL(k_divergence, dim3((unsigned) ((nn + 255) / 256), (unsigned) W), dim3(256),
                       0, s, C, C2, sel, n, n_pad, scale, D);
    return hipGetLastError();
}

hipError_t tsg_launch_set_divergence(const double *D, int n, int W, const int32_t *off, int nsets,
                                     double *out, hipStream_t s) {
    hipLaunchKernelGGL(k_set_divergence, dim3((unsigned) nsets * (unsigned) nsets, (unsigned) W),
                       dim3(256), 0, s, D, n, off, nsets, out);
    return hipGetLastError();
}

hipError_t tsg_launch_centre(const int32_t *C, const int32_t *C2, const int32_t *sel,
                             int64_t *rowsum, int n, int n_pad, int W, const double *scale,
                             double *K, hipStream_t s) {
    hipLaunchKernelGGL(k_rowsum, dim3((unsigned) n, (unsigned) W), dim3(256), 0, s, C, C2, sel, n,
                       n_pad, rowsum);
    hipLaunchKernelGGL(k_total, dim3((unsigned) W), dim3(256), 0, s, rowsum, n, W);
    const int64_t nn = (int64_t) n * n;
    hipLaunchKernelGGL(k_centre, dim3((unsigned) ((nn + 255) / 256), (unsigned) W), dim3(256), 0, s,
                       C, C2, sel, rowsum, n, n_pad, scale, K);
    return hipGetLastError();
}
