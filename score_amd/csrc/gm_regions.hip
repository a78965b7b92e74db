/*
 * gm_regions.hip -- the growth step with several memory regions.
 *
 * SCORE run with OMP_NUM_THREADS = T > 1 splits the domain into T regions
 * (ompshar_ca2regions, SCORE_GridPartitioning.cpp:69-166), each with its own
 * Inside and Border lists, and runs their growth steps side by side
 * (SCORE_Kernel.cpp:6634-6654): each region sweeps its lists, lets its
 * completed Inside cells infect, then its completed Border cells.  An infection
 * aimed at a cell of another region is parked in a halo of the infecting
 * region, first come first served (omp_infect_OutOfRXFrontBorder, :4494-4555);
 * after the barrier each region takes up what its neighbours parked for it,
 * neighbour by neighbour in its mynborregions order and each halo in parking
 * order, into its Border list, with the weight looked up again
 * (ompshar_synchronize_haloregions_rx, :4777-4872).
 *
 * That outcome is one claim per target cell with a 32-bit key:
 *   attempt of the cell's own region    p*32 + r
 *   attempt parked in a halo            2^31 + n*2^28 + p*32 + r
 * p is the parent's position in the step's FullRX order (below 2^23), which
 * runs region by region, each Inside then Border, so that p orders one region's
 * parents as its serial loop does; r is the attempt's rank and n the rank of
 * the receiving region's neighbour index of the halo among the eight a halo can
 * have (3, 4, 5, 6, 15, 16, 17, 18).  Only a cell's own region attempts it directly,
 * so the smallest key is the serial winner: the own region's first attempt,
 * else the first parked one in the receiving region's order.  A halo cell,
 * once parked, is never parked again (its status is never reset, :4527-4531);
 * that can only matter for a cell that is no longer deformed, which no attempt
 * here reaches (it left the deformed bitmap).
 *
 * The 2T lists keep SCORE's slot numbering: a new record takes its list's k-th
 * recycled slot if there is one, else appends, k being its rank among the
 * list's new records in serial order (for a Border list: the region's own
 * infections, then the halo winners by neighbour).  Ranks come from prefix
 * counts over the parents, less the count at the region's first parent; the
 * infection passes give each block the parents of one region only, so that
 * count is the offset of the region's first block.
 *
 * At 160^3 in eight regions (477 steps of 8500 parents) a step of these passes went
 * from 135 to 62 us: compaction and propose pass 30 to 13, decide with the retirement and the recycled
 * slots 28 to 8.5, commit with the step's end 29 to 17, the two scans 27 to 13.4.
 *
 * Per step, in the profiling slots of the one-region kernels:
 *   k_reanchor (shared)   k_rg_sweep   k_rg_sweep_scan (+ per-list starts)
 *   k_rg_compact (+ the propose pass)   k_rg_decide (+ recycled slots)
 *   k_rg_decide_scan (+ per-region starts, list lengths)   k_rg_commit (+ the step's end)
 */
#include <algorithm>

#include "gm_device.h"

/* opposite neighbour direction (mynborregions order, ompshar_init_neighbortopology,
 * SCORE_Kernel.cpp:2028-2080) */
static __constant__ uint8_t c_opp[27] = {0, 2, 1, 4, 3, 6, 5, 10, 9, 8, 7, 14, 13, 12, 11, 18, 17, 16, 15,
                                         26, 25, 24, 23, 22, 21, 20, 19};
/* the halos an infection can be parked in, and each direction's index among them */
static __constant__ uint8_t c_hdir[GM_NHALO] = {3, 4, 5, 6, 15, 16, 17, 18};
static __device__ __forceinline__ constexpr uint32_t h_dir(int i) { return i < 4 ? 3u + i : 11u + i; }
/* the index among them of the opposite direction: 3 4 5 6 15 16 17 18 have 4 3 6 5 18 17 16 15 */
static __device__ __forceinline__ uint32_t h_opp(uint32_t i) { return i < 4u ? i ^ 1u : 11u - i; }
/* neighbour index of the direction (0, sy, sz), at [(sy+1)*3 + sz+1] */
static __constant__ uint8_t c_ydir_nb[9] = {15, 3, 16, 5, 0, 6, 17, 4, 18};
static __constant__ uint8_t c_hidx[27] = {0xFF, 0xFF, 0xFF, 0, 1, 2, 3, 0xFF, 0xFF, 0xFF, 0xFF, 0xFF, 0xFF, 0xFF,
                                          0xFF, 4, 5, 6, 7, 0xFF, 0xFF, 0xFF, 0xFF, 0xFF, 0xFF, 0xFF, 0xFF};

/* rows of the sweep's per-block counts, and where the infection pass's rows
 * start (after them: the recycling pass reads the sweep's offsets last) */
#define RS_F 0
#define RS_R 1
#define RS_UN 2
#define RW_ROW0 3
/* sweep blocks (of 2048 slots) up to which compaction blocks do the propose pass; runs in
 * eight regions, so and apart: 160^3 (0.8M slots at most) 29.9 and 31.2 ms, 200^3 (1.5M)
 * 34.5 and 34.6, 256^3 (3.1M) 49.7 and 42.2, 320^3 80.3 and 53.5 */
#define GM_RG_FUSE 1024u
/* and, after its own, the row of its parents in the grain that sets rhomax */
#define RW_TOP (RW_ROW0 + GM_RROWS)

/* the part_of block size for a grid of nb blocks, from any thread */
static __device__ __forceinline__ uint32_t part_per(uint32_t n, uint32_t nb, uint32_t q) {
    uint32_t per = (n + nb - 1u) / nb;
    return (per + q - 1u) / q * q;
}

/* Exclusive scan, in place, of `rows` <= 16 rows of nb <= GM_MAX_BLOCKS per-block
 * counts by one block of 1024 threads, a wave per row, eight consecutive entries per
 * lane; tot (shared) receives the totals.  (The whole block on one row after another
 * waited for memory twice a row: 17.6 us a step for eleven rows.) */
static __device__ void scan_rows(uint32_t *bcnt, uint32_t rows, uint32_t nb, uint32_t *tot) {
    const uint32_t lane = threadIdx.x & 63u, c = threadIdx.x >> 6;
    if (c < rows) {
        uint32_t carry = 0;
        for (uint32_t b0 = 0; b0 < nb; b0 += 512u) {
            const uint32_t i0 = b0 + 8u * lane;
            uint4 *q = reinterpret_cast<uint4 *>(bcnt + (size_t)c * GM_MAX_BLOCKS + i0);
            uint4 a = make_uint4(0u, 0u, 0u, 0u), b = a;
            if (i0 < nb) {
                a = q[0];
                b = q[1];
            }
            uint32_t v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w}, sum = 0;
#pragma unroll
            for (uint32_t j = 0; j < 8; j++) {
                const uint32_t x = i0 + j < nb ? v[j] : 0u;
                v[j] = sum;
                sum += x;
            }
            const uint32_t incl = wave_incl_scan(sum), run = carry + incl - sum;
            if (i0 < nb) {
                q[0] = make_uint4(run + v[0], run + v[1], run + v[2], run + v[3]);
                q[1] = make_uint4(run + v[4], run + v[5], run + v[6], run + v[7]);
            }
            carry += __shfl(incl, 63, 64);
        }
        if (lane == 0) tot[c] = carry;
    }
    __syncthreads();
}

/* grid of the infection passes: at least one block more than there are regions,
 * so that every region's parents fit in whole blocks of GM_PCHUNK multiples */
static uint32_t rg_infect_blocks(const GmDev &d, uint32_t parents_upper) {
    const uint32_t nb = grid_for(parents_upper, GM_PCHUNK);
    return nb > d.nreg ? nb : d.nreg + 1u;
}

/* The parents of infection-pass block b: blocks are handed out region by region
 * (L.bstart[r] is region r's first block), so a block holds one region's parents
 * only; r is that region (k_rg_sweep_scan; past the blocks in use: none). */
static __device__ __forceinline__ void rg_part(const GmDev &d, uint32_t b, uint32_t &lo, uint32_t &hi, uint32_t &r) {
    const uint4 v = d.L.breg[b];
    lo = v.x;
    hi = v.y;
    r = v.z;
}

/* sweep tiles of a list of n occupied slots: whole 8-tile chunks */
static __device__ __forceinline__ uint32_t list_tiles(uint32_t n) {
    return (n + 64u * GM_SW_TPC - 1u) / (64u * GM_SW_TPC) * GM_SW_TPC;
}

struct RgTarget {
    uint32_t x, y, z;
    uint32_t dl;                /* list the new record goes to */
    uint32_t hidx;              /* halo index among the GM_NHALO, for a parked attempt */
    uint32_t khi;               /* upper part of the claim key: 0 for the own region */
};

/* Target of attempt rank rk of a parent at (x,y,z) in list l, routed as the
 * reference does.  Inside parents (omp_infect_OutOfRXFrontInside,
 * SCORE_Kernel.cpp:4252-4344) stay in their region and send every target to its
 * Border list unless they lie more than one cell inside each face of the
 * region (:4606-4609).  Border parents (:4347-4556) wrap x and y, drop targets
 * outside z, send targets strictly inside the region to its Inside list and the
 * region's other targets to its Border list; a target in another region goes to
 * the first halo towards that region whose box, taken one cell beyond its
 * extent as the reference's test does (:4500-4512), holds it.  False: no
 * target. */
/* a region's box, loaded once by the caller for all attempts of its parents */
struct RgBox {
    int lo0, lo1, lo2, hi0, hi1, hi2;
};

/* region r's box from the region grid alone (as build_regions lays it out), so
 * that no load waits for it */
static __device__ __forceinline__ RgBox rg_box(const GmDev &d, uint32_t r) {
    const uint32_t iy = r % d.npy, iz = r / d.npy;
    const int lo1 = (int)(iy * d.nry), lo2 = (int)(iz * d.nrz);
    const int hi1 = iy + 1u == d.npy ? (int)d.ny - 1 : lo1 + (int)d.nry - 1;
    const int hi2 = iz + 1u == d.npz ? (int)d.nz - 1 : lo2 + (int)d.nrz - 1;
    return RgBox{0, lo1, lo2, (int)d.nx - 1, hi1, hi2};
}

static __device__ __forceinline__ bool rg_target(const GmDev &d, const RgBox &B, uint32_t l, uint32_t x, uint32_t y,
                                                  uint32_t z, int rk, RgTarget &o) {
    const uint32_t r = l >> 1;
    int tx = (int)x + dir_dx(rk), ty = (int)y + dir_dy(rk), tz = (int)z + dir_dz(rk);
    const int nx = (int)d.nx, ny = (int)d.ny, nz = (int)d.nz;
    const int lo0 = B.lo0, lo1 = B.lo1, lo2 = B.lo2, hi0 = B.hi0, hi1 = B.hi1, hi2 = B.hi2;
    o.khi = 0u;
    o.hidx = GM_NHALO;
    if (!(l & 1u)) {
        /* an Inside cell is strictly inside its region: this never fires, and
         * keeps a corrupted record from addressing outside the grid */
        if (tx < 0 || tx >= nx || ty < 0 || ty >= ny || tz < 0 || tz >= nz) return false;
        const bool deep = (int)x > lo0 + 1 && (int)x < hi0 - 1 && (int)y > lo1 + 1 && (int)y < hi1 - 1 &&
                          (int)z > lo2 + 1 && (int)z < hi2 - 1;
        o.dl = deep ? 2u * r : 2u * r + 1u;
    } else {
        if (tx < 0) tx += nx;
        if (tx >= nx) tx -= nx;
        if (ty < 0) ty += ny;
        if (ty >= ny) ty -= ny;
        if (tz < 0 || tz >= nz) return false;
        if (tx > lo0 && tx < hi0 && ty > lo1 && ty < hi1 && tz > lo2 && tz < hi2) {
            o.dl = 2u * r;
        } else {
            /* the target lies in the region or next to it: the neighbour in the
             * direction it left along y (none with one slab along y, whose
             * region spans every y) and z */
            const int uy = (int)y + dir_dy(rk), uz = (int)z + dir_dz(rk);
            const int sy = d.npy == 1u ? 0 : (uy < lo1 ? -1 : (uy > hi1 ? 1 : 0));
            const int sz = uz < lo2 ? -1 : (uz > hi2 ? 1 : 0);
            const GmRegion &R = d.reg[r];
            const uint32_t q = R.nbor[c_ydir_nb[(sy + 1) * 3 + (sz + 1)]];
            if (q == r) {
                o.dl = 2u * r + 1u;
            } else {
                /* the eight halos that can be, loaded together: a wave with one such
                 * attempt waits once, not once per halo (27 of them one after another
                 * made the propose, decide and commit passes 25, 23 and 25 us at 8500
                 * parents in eight regions) */
                uint4 hv[GM_NHALO];
#pragma unroll
                for (int i = 0; i < GM_NHALO; i++) hv[i] = *reinterpret_cast<const uint4 *>(&R.halo[h_dir(i)]);
                uint32_t hx = GM_NHALO;
#pragma unroll
                for (int i = GM_NHALO - 1; i >= 0; i--) {
                    const int ox = (int)(hv[i].y & 0xFFFFu), oy = (int)(hv[i].y >> 16), oz = (int)(hv[i].z & 0xFFFFu);
                    const int ex = (int)(hv[i].z >> 16), ey = (int)(hv[i].w & 0xFFFFu), ez = (int)(hv[i].w >> 16);
                    const bool in = tx >= ox && tx <= ox + ex && ty >= oy && ty <= oy + ey && tz >= oz && tz <= oz + ez;
                    if (hv[i].x == q && ex != 0 && in) hx = (uint32_t)i;
                }
                if (hx >= GM_NHALO) {
                    atomicOr(&d.st->err, GM_ERRF_HALO);
                    return false;
                }
                o.hidx = hx;
                o.dl = 2u * q + 1u;
                o.khi = (1u << 31) | (h_opp(hx) << 28);
            }
        }
    }
    o.x = (uint32_t)tx;
    o.y = (uint32_t)ty;
    o.z = (uint32_t)tz;
    return true;
}

/* ------------------------------------------------------------- list tables */

/* One block of 1024 threads: the lists' occupied and tile prefixes from their
 * lengths, and the lengths summed over Inside and Border lists; thread t takes
 * region t's two lists, of lengths nI and nB (at most 1024 regions). */
static __device__ __forceinline__ void rg_prefix_block(const GmDev &d, uint32_t nI, uint32_t nB) {
    __shared__ uint32_t ws[16][4];
    const uint32_t t = threadIdx.x, lane = t & 63u, w = t >> 6;
    const bool v = t < d.nreg;
    if (!v) nI = nB = 0;
    const uint32_t tI = list_tiles(nI), tB = list_tiles(nB);
    const uint32_t val[4] = {nI + nB, tI + tB, nI, nB};
    uint32_t incl[4];
#pragma unroll
    for (int c = 0; c < 4; c++) {
        incl[c] = wave_incl_scan(val[c]);
        if (lane == 63u) ws[w][c] = incl[c];
    }
    __syncthreads();
    uint32_t pre[4] = {0, 0, 0, 0}, tot[4] = {0, 0, 0, 0};
    for (uint32_t i = 0; i < 16u; i++)
#pragma unroll
        for (int c = 0; c < 4; c++) {
            if (i < w) pre[c] += ws[i][c];
            tot[c] += ws[i][c];
        }
    if (v) {
        const uint32_t o = pre[0] + incl[0] - val[0], ti = pre[1] + incl[1] - val[1];
        d.L.occ[2u * t] = o;
        d.L.occ[2u * t + 1u] = o + nI;
        d.L.tile[2u * t] = ti;
        d.L.tile[2u * t + 1u] = ti + tI;
    }
    if (t == 0) {
        d.L.occ[d.nlists] = tot[0];
        d.L.tile[d.nlists] = tot[1];
        d.st->nI = tot[2];
        d.st->nB = tot[3];
    }
    __syncthreads();
}

__global__ void __launch_bounds__(1024) k_rg_prefix(GmDev d) {
    const uint32_t t = threadIdx.x < d.nreg ? threadIdx.x : 0u;
    rg_prefix_block(d, d.L.n[2u * t], d.L.n[2u * t + 1u]);
}

hipError_t gm_launch_rg_prefix(const GmDev &d, hipStream_t s) {
    k_rg_prefix<<<1, 1024, 0, s>>>(d);
    return hipGetLastError();
}

/* nuclei placed by the host: records and codes scattered to their slots, and
 * their cells taken out of the deformed bitmap */
__global__ void k_rg_place(GmDev d, const uint32_t *slots, const GmRec *recs, uint32_t n) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const uint32_t s = slots[i];
        const GmRec r = recs[i];
        d.rec[s] = r;
        d.cstep[s] = (gm_cs_t)GM_CS_UNKNOWN;
        const uint32_t w = r.cell;
        const uint32_t z = w / d.nxy, rem = w - z * d.nxy, y = rem / d.nx, x = rem - y * d.nx;
        clear_deformed(d, x, y, z);
    }
}

hipError_t gm_launch_rg_place(const GmDev &d, const uint32_t *slots, const GmRec *recs, uint32_t n, hipStream_t s) {
    if (n) k_rg_place<<<fill_blocks(n), GM_BLOCK, 0, s>>>(d, slots, recs, n);
    return hipGetLastError();
}

/* ------------------------------------------------------------------- sweep */

/* Pass over the occupied slots of every list, as the one-region sweep does:
 * the lists' tiles follow one another, each list in whole 8-tile chunks, so a
 * chunk belongs to one list.  Completed and INACTIVE slots go into per-tile
 * masks, counted per block. */
__global__ void __launch_bounds__(GM_BLOCK) k_rg_sweep(GmDev d, GmSweepArgs A0) {
    __shared__ uint32_t red[GM_BLOCK / 64][3];
    __shared__ uint64_t sF[GM_BLOCK / 64][8], sR[GM_BLOCK / 64][8];
    if (d.st->halt) return;
    const GmSweepArgs A = step_args(d, A0);
    const uint32_t T = d.L.tile[d.nlists];
    const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t lo, hi;
    part_of(T, GM_SW_TPC, lo, hi);
    const uint32_t c_lo = lo / GM_SW_TPC, c_hi = hi / GM_SW_TPC; /* T is a whole number of chunks */
    const uint32_t kc = A.k & (GM_CS_MOD - 1u), horizon = d.horizon;
    uint32_t cF = 0, cR = 0, unknown = 0;
    for (uint32_t c = c_lo + w; c < c_hi; c += GM_BLOCK / 64) {
        const uint32_t tile0 = c * GM_SW_TPC;
        const uint32_t l = upper_index(d.L.tile, d.nlists, tile0);
        const uint32_t s0 = d.L.base[l] + (tile0 - d.L.tile[l]) * 64u;
        const uint32_t base = s0 + 8u * lane;
        const uint32_t lim = d.L.base[l] + d.L.n[l];
        const uint32_t nocc = lim > base ? (lim - base < 8u ? lim - base : 8u) : 0u;
        const uint4 cs = nocc ? *reinterpret_cast<const uint4 *>(d.cstep + base)
                              : make_uint4(0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu);
        const uint32_t pack = sweep_classify(cs, nocc, kc, horizon, unknown);
        cF += (uint32_t)__popc(pack & 0xFFu);
        cR += (uint32_t)__popc(pack >> 8);
        uint64_t myF, myR;
        sweep_masks(pack, sF[w], sR[w], myF, myR);
        if (lane < GM_SW_TPC) {
            d.mF[tile0 + lane] = myF;
            d.mR[tile0 + lane] = myR;
        }
    }
    for (int o = 32; o > 0; o >>= 1) {
        unknown += __shfl_down(unknown, o, 64);
        cF += __shfl_down(cF, o, 64);
        cR += __shfl_down(cR, o, 64);
    }
    if (lane == 0) {
        red[w][RS_F] = cF;
        red[w][RS_R] = cR;
        red[w][RS_UN] = unknown;
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        uint32_t t = 0;
        for (int i = 0; i < GM_BLOCK / 64; i++) t += red[i][threadIdx.x];
        d.bcnt[threadIdx.x * GM_MAX_BLOCKS + blockIdx.x] = t;
    }
}

/* One block: per-block offsets; then each list's first completed and first
 * INACTIVE position (the block offset of the tile where the list starts plus
 * the block's tiles before it), the per-list counts, and their sums over the
 * Inside and the Border lists.  The tiles are read beside the scan, and what the
 * lists' threads hand to each other stays in LDS. */
__global__ void __launch_bounds__(1024) k_rg_sweep_scan(GmDev d, uint32_t nb, uint32_t nbd) {
    __shared__ uint32_t acc[6], tot[3], ws[16], sF[2049], sR[2049], sS[1025];
    GmStats *st = d.st;
    if (st->halt) return;
    const uint32_t T = d.L.tile[d.nlists];
    const uint32_t per = T ? part_per(T, nb, GM_SW_TPC) : 1u;
    const uint32_t lane = threadIdx.x & 63u, wv = threadIdx.x >> 6;
    if (threadIdx.x < 6) acc[threadIdx.x] = 0;
    /* one wave per list, the lanes sharing the block's tiles before the list's first */
    if (threadIdx.x == 0) {
        d.L.tile_s[d.nlists] = T;
        sF[d.nlists] = sR[d.nlists] = 0;
    }
    for (uint32_t l = wv; l < d.nlists; l += 1024u / 64u) {
        const uint32_t t0 = d.L.tile[l];
        uint32_t ef = 0, er = 0;
        if (t0 < T)
            for (uint32_t t = t0 / per * per + lane; t < t0; t += 64) {
                ef += (uint32_t)__popcll(d.mF[t]);
                er += (uint32_t)__popcll(d.mR[t]);
            }
        for (int o = 32; o > 0; o >>= 1) {
            ef += __shfl_down(ef, o, 64);
            er += __shfl_down(er, o, 64);
        }
        if (lane == 0) {
            d.L.tile_s[l] = t0; /* this step's tiles, for the recycling pass after the lengths change */
            sF[l] = ef;
            sR[l] = er;
        }
    }
    if (nb <= GM_RG_FUSE) {
        scan_rows(d.bcnt, 3u, nb, tot);
    } else { /* sixteen rounds of a wave a row took 17 us, this 11 */
        uint32_t v[3];
        scan_block_counts<3>(d.bcnt, nb, v);
        if (threadIdx.x < 3u) tot[threadIdx.x] = threadIdx.x == 0u ? v[0] : threadIdx.x == 1u ? v[1] : v[2];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        if (tot[RS_UN]) st->err |= GM_ERRF_MISSED;
        /* infection keys are (halo, neighbour, p, rank) in 32 bits, p < 2^23 */
        if ((uint64_t)tot[RS_F] > (1ull << 23)) st->err |= GM_ERRF_KEYS;
    }
    for (uint32_t l = threadIdx.x; l <= d.nlists; l += 1024) {
        const uint32_t t0 = d.L.tile[l], b = t0 / per;
        const uint32_t f = t0 < T ? d.bcnt[RS_F * GM_MAX_BLOCKS + b] + sF[l] : tot[RS_F];
        const uint32_t r = t0 < T ? d.bcnt[RS_R * GM_MAX_BLOCKS + b] + sR[l] : tot[RS_R];
        d.L.par[l] = sF[l] = f;
        d.L.rst[l] = sR[l] = r;
    }
    __syncthreads();
    uint32_t a[6] = {0, 0, 0, 0, 0, 0};
    for (uint32_t l = threadIdx.x; l < d.nlists; l += 1024) {
        const uint32_t nf = sF[l + 1] - sF[l], nr = sR[l + 1] - sR[l], rc = d.L.rcap[l];
        const uint32_t rl = nr < rc ? nr : rc;
        d.L.rlen[l] = rl;
        const uint32_t k = (l & 1u) * 3u;
        a[k] += nf;
        a[k + 1] += nr;
        a[k + 2] += rl;
    }
#pragma unroll
    for (int c = 0; c < 6; c++)
        if (a[c]) atomicAdd(&acc[c], a[c]);
    /* the infection passes' blocks, region by region: pper parents each (a
     * multiple of GM_PCHUNK), few enough that all regions fit in nbd blocks */
    const uint32_t nfull = tot[RS_F];
    uint32_t pper = (nfull + (nbd - d.nreg) - 1u) / (nbd - d.nreg);
    pper = pper ? (pper + GM_PCHUNK - 1u) / GM_PCHUNK * GM_PCHUNK : GM_PCHUNK;
    const uint32_t r = threadIdx.x;
    const uint32_t nr = r < d.nreg ? sF[2u * r + 2u] - sF[2u * r] : 0u;
    const uint32_t blk = (nr + pper - 1u) / pper;
    const uint32_t incl = wave_incl_scan(blk);
    if (lane == 63u) ws[wv] = incl;
    __syncthreads();
    uint32_t pre = 0, totb = 0;
    for (uint32_t i = 0; i < 16u; i++) {
        if (i < wv) pre += ws[i];
        totb += ws[i];
    }
    if (r < d.nreg) d.L.bstart[r] = sS[r] = pre + incl - blk;
    if (threadIdx.x == 0) d.L.bstart[d.nreg] = sS[d.nreg] = totb;
    __syncthreads();
    /* each block's parents and region; blocks past the ones in use have none */
    for (uint32_t b = threadIdx.x; b < nbd; b += 1024) {
        uint4 v = make_uint4(0u, 0u, 0u, 0u);
        if (b < totb) {
            const uint32_t q = upper_index(sS, d.nreg, b), lo = sF[2u * q] + (b - sS[q]) * pper, end = sF[2u * q + 2u];
            v = make_uint4(lo, lo + pper < end ? lo + pper : end, q, 0u);
        }
        d.L.breg[b] = v;
    }
    if (threadIdx.x == 0) {
        st->ntried = 0;
        st->nfullI = acc[0];
        st->totRecI = acc[1];
        st->recLenI = acc[2];
        st->nfullB = acc[3];
        st->totRecB = acc[4];
        st->recLenB = acc[5];
    }
}

struct RgWave {
    uint4 q2[64];
    uint32_t bad[64];
    uint16_t wl[26 * 64];
};

/* Parents p0 .. p0+n-1 (n <= 64) by a wave, a lane each, as the one-region propose
 * pass: the parent's data into the dense array (with its list in place of the Border
 * flag), its value after the completing addition, its retirement into the log (rlog;
 * null: it does not fit); its deformed neighbours come from three 16-byte loads of the
 * bitmap.  Every attempt on one of them, routed to the region it lies in, claims it:
 * the parents' attempts are flattened into a list, a lane per attempt, so that a wave
 * waits for its attempts' halos at once.  Returns the attempts. */
static __device__ __forceinline__ uint32_t rg_propose(const GmDev &d, RgWave &W, uint32_t p0, uint32_t n, uint32_t k,
                                                      uint2 *rlog) {
    const uint32_t lane = threadIdx.x & 63u, p = p0 + lane;
    uint32_t am = 0;
    if (lane < n) {
        const uint32_t s = d.pslot[p], l = d.plist[p];
        const GmRec *r = d.rec + s;
        const RecC rc = rec_c(r);
        const RecA ra = rec_a(r);
        const double inc = r->inc;
        const uint32_t rxg = r->rxg, cell = rc.cell;
        const uint32_t z = cell / d.nxy, rem = cell - z * d.nxy, y = rem / d.nx, x = rem - y * d.nx;
        const bool interior = (x - 1u < d.nx - 2u) & (y - 1u < d.ny - 2u) & (z - 1u < d.nz - 2u);
        Neighbourhood nb;
        if (interior) nb.load(d, x, y, z);
        const double fin = advanced(ra.frac0, inc, k - ra.s0 + 1u);
        am = interior ? nb.mask() : face_attempts(d, x, y, z);
        const uint4 q2 = make_uint4(x, y, z, l);
        W.q2[lane] = q2;
        par_plane(d, GM_PAR_IDS)[p] = make_uint4(s, cell, rc.defg, rxg);
        reinterpret_cast<double2 *>(par_plane(d, GM_PAR_FP))[p] = make_double2(fin, rc.P);
        par_plane(d, GM_PAR_XYZ)[p] = q2;
        if (rlog) rlog[p] = make_uint2(cell, d.ndefg + rxg);
    }
    W.bad[lane] = 0;
    const uint32_t na = list_attempts(am, W.wl);
    for (uint32_t i = lane; i < na; i += 64u) {
        const uint32_t e = W.wl[i], q = e & 0xFFu, rk = e >> 8;
        const uint4 q2 = W.q2[q];
        RgTarget o;
        if (rg_target(d, rg_box(d, q2.w >> 1), q2.w, q2.x, q2.y, q2.z, (int)rk, o))
            atomicMin(&d.cell[cell_of(d, o.x, o.y, o.z)].x, o.khi | ((p0 + q) * 32u + rk));
        else
            atomicOr(&W.bad[q], 1u << rk);
    }
    wave_sync();
    if (lane < n) d.pmI[p] = am & ~W.bad[lane];
    wave_sync();
    return na;
}

/* The completed slots of tiles [lo, hi) in FullRX order (append_to_fullrx_*_list,
 * SCORE_Kernel.cpp:3994-4042, :4133-4180) from position `first` on, the lists one after
 * another, by one wave, a lane per tile; the position behind them. */
static __device__ __forceinline__ uint32_t rg_list(const GmDev &d, uint32_t lo, uint32_t hi, uint32_t first) {
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t runF = first;
    for (uint32_t batch = lo; batch < hi; batch += 64) {
        const uint32_t t = batch + lane;
        const uint64_t bf = t < hi ? d.mF[t] : 0ull;
        const uint32_t cf = (uint32_t)__popcll(bf);
        const uint32_t incf = wave_incl_scan(cf);
        uint32_t of = runF + incf - cf;
        runF += __shfl(incf, 63, 64);
        if (bf) {
            const uint32_t l = upper_index(d.L.tile, d.nlists, t);
            const uint32_t s0 = d.L.base[l] + (t - d.L.tile[l]) * 64u;
            for (uint64_t m = bf; m; m &= m - 1ull) {
                d.plist[of] = l;
                d.pslot[of++] = s0 + (uint32_t)__ffsll((long long)m) - 1u;
            }
        }
    }
    return runF;
}

/* Long fronts (more than GM_RG_FUSE sweep blocks): the list alone, a wave per block,
 * and the propose pass in a launch of its own, with full waves.  A sweep block has some
 * 30 parents, half a wave: on 512^3 in eight regions the two passes take less than the
 * fused one (81 us with four waves a block, 97 with one). */
__global__ void __launch_bounds__(64) k_rg_list(GmDev d) {
    if (d.st->halt) return;
    uint32_t lo, hi;
    part_of(d.L.tile[d.nlists], GM_SW_TPC, lo, hi);
    rg_list(d, lo, hi, d.bcnt[RS_F * GM_MAX_BLOCKS + blockIdx.x]);
}

/* Parents [p0, p1) by the block, 64 a wave, `step` parents on for the next; their
 * attempts are added to the step's. */
static __device__ __forceinline__ void rg_propose_block(const GmDev &d, uint32_t p0, uint32_t p1, uint32_t step) {
    __shared__ RgWave sw[GM_BLOCK / 64];
    __shared__ uint32_t satt[GM_BLOCK / 64];
    GmStats *st = d.st;
    const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
    const uint32_t nfull = st->nfullI + st->nfullB, k = st->kcur;
    const unsigned long long nret = st->nret;
    const bool logged = nret + nfull <= d.rlogCap;
    if (!logged && blockIdx.x == 0 && threadIdx.x == 0) atomicOr(&st->err, GM_ERRF_RLOG_FULL);
    uint32_t natt = 0;
    for (uint32_t p = p0 + w * 64u; p < p1; p += step)
        natt += rg_propose(d, sw[w], p, p1 - p < 64u ? p1 - p : 64u, k, logged ? d.rlog + nret : nullptr);
    if (lane == 0) satt[w] = natt;
    __syncthreads();
    natt = satt[0] + satt[1] + satt[2] + satt[3];
    if (threadIdx.x == 0 && natt) atomicAdd(&st->ntried, natt);
}

__global__ void __launch_bounds__(GM_BLOCK) k_rg_propose(GmDev d) {
    if (d.st->halt) return;
    rg_propose_block(d, blockIdx.x * GM_BLOCK, d.st->nfullI + d.st->nfullB, gridDim.x * GM_BLOCK);
}

/* The sweep's partition: a block's first wave lists its completed slots, then all its
 * waves take these parents through the propose pass, which in a launch of its own read
 * them back (5 us a step). */
__global__ void __launch_bounds__(GM_BLOCK) k_rg_compact(GmDev d) {
    __shared__ uint32_t send;
    if (d.st->halt) return;
    uint32_t lo, hi;
    part_of(d.L.tile[d.nlists], GM_SW_TPC, lo, hi);
    const uint32_t first = d.bcnt[RS_F * GM_MAX_BLOCKS + blockIdx.x];
    if (threadIdx.x < 64u) {
        const uint32_t end = rg_list(d, lo, hi, first);
        if (threadIdx.x == 0) send = end;
    }
    __syncthreads();
    rg_propose_block(d, first, send, GM_BLOCK);
}

/* Each list's INACTIVE slots in ascending order (append_to_recycling_*_list,
 * SCORE_Kernel.cpp:4037-4041, :4175-4179), as far as they can be handed out: at most
 * the recycled slots, and no more than the step's attempts.  Runs beside the decide
 * pass, before the new records per list are known (a pass of its own after that took
 * 5 us and a gap).  The sweep's partition and offsets; one wave per sweep block. */
static __device__ __forceinline__ void rg_recycle(const GmDev &d, uint32_t blk, uint32_t nblk) {
    const uint32_t lane = threadIdx.x, T = d.L.tile_s[d.nlists], per = part_per(T, nblk, GM_SW_TPC);
    uint32_t lo = blk * per, hi = lo + per;
    const uint32_t na = d.st->ntried;
    if (lo > T) lo = T;
    if (hi > T) hi = T;
    uint32_t runR = d.bcnt[RS_R * GM_MAX_BLOCKS + blk];
    for (uint32_t batch = lo; batch < hi; batch += 64) {
        const uint32_t t = batch + lane;
        const uint64_t br = t < hi ? d.mR[t] : 0ull;
        const uint32_t cr = (uint32_t)__popcll(br);
        const uint32_t incr = wave_incl_scan(cr);
        const uint32_t orr = runR + incr - cr;
        runR += __shfl(incr, 63, 64);
        if (br) {
            const uint32_t l = upper_index(d.L.tile_s, d.nlists, t);
            const uint32_t rl = d.L.rlen[l], lim = na < rl ? na : rl;
            uint32_t k = orr - d.L.rst[l];
            if (k < lim) {
                const uint32_t rel0 = (t - d.L.tile_s[l]) * 64u;
                uint32_t *rb = d.L.rbuf + d.L.rbase[l];
                for (uint64_t m = br; m && k < lim; m &= m - 1ull) rb[k++] = rel0 + (uint32_t)__ffsll((long long)m) - 1u;
            }
        }
    }
}

/* grid of the sweep, compaction and recycling passes for about nI + nB occupied slots */
static uint32_t rg_sweep_blocks(const GmDev &d, const GmSweepArgs &a) {
    const uint64_t tiles = (uint64_t)(a.nI + a.nB) / 64u + (uint64_t)GM_SW_TPC * (d.nlists + 1u);
    return grid_for((uint32_t)std::min<uint64_t>(tiles, 0xFFFFFFFFull), GM_SW_TPC * (GM_BLOCK / 64));
}

hipError_t gm_launch_rg_sweep(const GmDev &d, const GmSweepArgs &a, uint32_t parents_upper, hipStream_t s,
                              hipEvent_t *ev) {
    hipError_t e;
    GmSweepArgs A = a;
    A.reanchor = 0;
    if ((e = mark(ev, 0, s)) != hipSuccess) return e;
    if (a.reanchor && (e = gm_launch_reanchor(d, a, s)) != hipSuccess) return e;
    const uint32_t nb = rg_sweep_blocks(d, a);
    if ((e = mark(ev, 1, s)) != hipSuccess) return e;
    k_rg_sweep<<<nb, GM_BLOCK, 0, s>>>(d, A);
    if ((e = mark(ev, 2, s)) != hipSuccess) return e;
    k_rg_sweep_scan<<<1, 1024, 0, s>>>(d, nb, rg_infect_blocks(d, parents_upper));
    if ((e = mark(ev, 3, s)) != hipSuccess) return e;
    if (nb <= GM_RG_FUSE) {
        k_rg_compact<<<nb, GM_BLOCK, 0, s>>>(d);
    } else {
        k_rg_list<<<nb, 64, 0, s>>>(d);
        k_rg_propose<<<grid_for(parents_upper, GM_BLOCK), GM_BLOCK, 0, s>>>(d);
    }
    return hipGetLastError();
}

/* --------------------------------------------------------------- infection */

/* The attempts that hold their target's smallest key, as masks by destination (own
 * Inside, own Border, a halo), counted per block by row (GM_RW_*).  64 parents'
 * attempts are flattened into a list, a lane per attempt, so that all claims are
 * loaded together.  The parents retire here, beside the waiting for the claims.  The
 * partition into blocks (one region per block) is the commit pass's.  The launch's
 * first nrec blocks write the recycled slots. */
__global__ void __launch_bounds__(64) k_rg_decide(GmDev d, uint32_t nrec, uint32_t top_pos) {
    __shared__ uint4 sq2[64];
    __shared__ uint32_t sI[64], sB[64], sH[64], scnt[GM_RROWS];
    __shared__ uint16_t wl[26 * 64];
    if (d.st->halt) return;
    if (blockIdx.x < nrec) {
        rg_recycle(d, blockIdx.x, nrec);
        return;
    }
    const uint32_t lane = threadIdx.x, blk = blockIdx.x - nrec;
    uint32_t lo, hi, reg;
    rg_part(d, blk, lo, hi, reg);
    const RgBox box = rg_box(d, reg);
    if (lane < GM_RROWS) scnt[lane] = 0;
    uint32_t nI = 0, nB = 0, nA = 0, ntop = 0;
    bool wrapped = false;
    for (uint32_t batch = lo; batch < hi; batch += 64) {
        const uint32_t p = batch + lane;
        const bool valid = p < hi;
        const uint32_t am = valid ? d.pmI[p] : 0u;
        sq2[lane] = valid ? par_plane(d, GM_PAR_XYZ)[p] : make_uint4(0u, 0u, 0u, 0u);
        sI[lane] = sB[lane] = sH[lane] = 0;
        const uint4 q0 = valid ? par_plane(d, GM_PAR_IDS)[p] : make_uint4(0u, 0u, 0xFFFFFFFFu, 0xFFFFFFFFu);
        retire(d, q0.z, q0.w, valid, blk & (GM_SUBS - 1u));
        const uint32_t rp = valid ? d.rpos[q0.z] : 0xFFFFFFFFu;
        const uint32_t n = list_attempts(am, wl);
        for (uint32_t i = lane; i < n; i += 64u) {
            const uint32_t e = wl[i], q = e & 0xFFu, rk = e >> 8;
            const uint4 q2 = sq2[q];
            RgTarget o;
            rg_target(d, box, q2.w, q2.x, q2.y, q2.z, (int)rk, o);
            if (d.cell[cell_of(d, o.x, o.y, o.z)].x != (o.khi | ((batch + q) * 32u + rk))) continue;
            if (o.khi) {
                atomicOr(&sH[q], 1u << rk);
                atomicAdd(&scnt[GM_RW_H0 + o.hidx], 1u);
            } else {
                atomicOr((o.dl & 1u) ? &sB[q] : &sI[q], 1u << rk);
            }
        }
        wave_sync();
        ntop += rp == top_pos ? 1u : 0u;
        wrapped |= rp < top_pos;
        const uint32_t mI = sI[lane], mB = sB[lane];
        if (valid) {
            d.pmI[p] = mI;
            d.pmB[p] = mB;
            d.pmH[p] = sH[lane];
        }
        nI += (uint32_t)__popc(mI);
        nB += (uint32_t)__popc(mB);
        nA += (uint32_t)__popc(am);
        wave_sync();
    }
    for (int o = 32; o > 0; o >>= 1) {
        nI += __shfl_xor(nI, o, 64);
        nB += __shfl_xor(nB, o, 64);
        nA += __shfl_xor(nA, o, 64);
        ntop += __shfl_xor(ntop, o, 64);
    }
    wave_sync();
    if (__any(wrapped) && lane == 0) d.st->cwrap = 1u;
    if (lane == GM_RROWS) d.bcnt[RW_TOP * GM_MAX_BLOCKS + blk] = ntop;
    if (lane < GM_RROWS)
        d.bcnt[(RW_ROW0 + lane) * GM_MAX_BLOCKS + blk] =
            lane == GM_RW_I ? nI : lane == GM_RW_B ? nB : lane == GM_RW_A ? nA : scnt[lane];
}

/* One block: per-block offsets of every row; then, per region, the counts of
 * each row before its first parent (block offset plus the block's parents
 * before it); per region, where each neighbour's halo winners start in its
 * Border list (after its own winners, in its neighbour order: the infecting
 * region S = nbor[nb] parked them in its halo opp(nb)); the new records per
 * list, the lists' new lengths (recycled slots first, then appended) and their
 * prefixes for the next step.  A thread has a region: what it needs of the tables is
 * loaded beside the scan, and the regions' counts go through LDS (at most
 * 1025 x 11 of them). */
__global__ void __launch_bounds__(1024) k_rg_decide_scan(GmDev d, uint32_t nb) {
    __shared__ uint32_t acc[2], tot[GM_RROWS + 1], srs[(1024 + 1) * GM_RROWS];
    GmStats *st = d.st;
    const uint32_t q = threadIdx.x, r = q < d.nreg ? q : 0u;
    const uint32_t halt = st->halt, nused = d.L.bstart[d.nreg], b = d.L.bstart[r];
    const uint32_t oI = d.L.n[2u * r], oB = d.L.n[2u * r + 1u], rlI = d.L.rlen[2u * r], rlB = d.L.rlen[2u * r + 1u];
    const uint32_t left0 = d.win->left[0];
    uint32_t S[GM_NHALO];
#pragma unroll
    for (uint32_t j = 0; j < GM_NHALO; j++) S[j] = d.reg[r].nbor[c_hdir[j]];
    if (halt) return;
    /* (blocks past the ones in use counted nothing) */
    scan_rows(d.bcnt + RW_ROW0 * GM_MAX_BLOCKS, GM_RROWS + 1, nb, tot);
    if (q < 2) acc[q] = 0;
    if (q == 0) {
        st->nattempt = tot[GM_RW_A];
        if (tot[GM_RROWS]) { /* the cells left of the grain that sets rhomax */
            const uint32_t left = left0 - tot[GM_RROWS];
            d.win->left[0] = left;
            if (left == 0u) d.win->top_hit = 1u;
        }
    }
    /* each region's counts at its first parent: the offset of its first block
     * (the next region's, or the totals, for a region without parents) */
    if (q < d.nreg) {
        uint32_t v[GM_RROWS];
#pragma unroll
        for (int c = 0; c < GM_RROWS; c++) v[c] = b < nused ? d.bcnt[(RW_ROW0 + c) * GM_MAX_BLOCKS + b] : tot[c];
#pragma unroll
        for (int c = 0; c < GM_RROWS; c++) d.L.rs[q * GM_RROWS + c] = srs[q * GM_RROWS + c] = v[c];
    }
    if (q < GM_RROWS) d.L.rs[d.nreg * GM_RROWS + q] = srs[d.nreg * GM_RROWS + q] = tot[q];
    __syncthreads();
    uint32_t nI = 0, nB = 0, wI = 0, wB = 0;
    if (q < d.nreg) {
        const uint32_t *a = srs + q * GM_RROWS, *e = a + GM_RROWS;
        wI = e[GM_RW_I] - a[GM_RW_I];
        wB = e[GM_RW_B] - a[GM_RW_B];
#pragma unroll
        for (uint32_t j = 0; j < GM_NHALO; j++) {
            const uint32_t hs = GM_RW_H0 + c_hidx[c_opp[c_hdir[j]]];
            d.L.hoff[q * GM_NHALO + j] = wB;
            if (S[j] != q) wB += srs[(S[j] + 1u) * GM_RROWS + hs] - srs[S[j] * GM_RROWS + hs];
        }
        nI = wI > rlI ? oI + (wI - rlI) : oI;
        nB = wB > rlB ? oB + (wB - rlB) : oB;
        d.L.nold[2u * q] = oI;
        d.L.nold[2u * q + 1u] = oB;
        d.L.n[2u * q] = nI;
        d.L.n[2u * q + 1u] = nB;
    }
    if (wI) atomicAdd(&acc[0], wI);
    if (wB) atomicAdd(&acc[1], wB);
    __syncthreads();
    if (q == 0) {
        st->winI = acc[0];
        st->winB = acc[1];
    }
    rg_prefix_block(d, nI, nB);
}

/* New records as the one-region commit pass writes them;
 * a winner's slot is its rank in its list: own Inside and own Border winners
 * by the parents' prefix counts less the count at the region's first parent,
 * halo winners after the receiving region's own, by neighbour, then by the
 * infecting region's prefix count of that halo.  A halo winner's weight is
 * looked up again whatever its deformed grain (SCORE_Kernel.cpp:4853). */
static __device__ __forceinline__ void rg_commit_step(const GmDev &d, const GmPParams &pp, const GmSweepArgs &A, uint32_t need_one) {
    __shared__ uint32_t sI[64], sB[64], oI[64], oB[64];
    __shared__ uint4 sq0[64], sq2[64];
    __shared__ double sfin[64], sP[64];
    __shared__ uint16_t wl[26 * 64];
    GmStats *st = d.st;
    const uint32_t k = st->kcur;
    bool one = false;
    const uint32_t lane = threadIdx.x;
    __shared__ uint32_t srs[GM_RROWS], sL[2][5];
    uint32_t lo, hi, reg;
    rg_part(d, blockIdx.x, lo, hi, reg);
    if (lo >= hi) return; /* no parents: nothing to commit */
    const RgBox box = rg_box(d, reg);
    /* the block's region: its counts at its first parent, and its two lists' tables */
    if (lane < GM_RROWS) srs[lane] = d.L.rs[reg * GM_RROWS + lane];
    if (lane < 2u) {
        const uint32_t l = 2u * reg + lane;
        sL[lane][0] = d.L.rlen[l];
        sL[lane][1] = d.L.rbase[l];
        sL[lane][2] = d.L.nold[l];
        sL[lane][3] = d.L.cap[l];
        sL[lane][4] = d.L.base[l];
    }
    uint32_t run[GM_RROWS];
#pragma unroll
    for (int c = 0; c < GM_RROWS; c++) run[c] = d.bcnt[(RW_ROW0 + c) * GM_MAX_BLOCKS + blockIdx.x];
    for (uint32_t batch = lo; batch < hi; batch += 64) {
        const uint32_t pt = batch + lane;
        const bool valid = pt < hi;
        const uint32_t mI = valid ? d.pmI[pt] : 0u, mB = valid ? d.pmB[pt] : 0u, mH = valid ? d.pmH[pt] : 0u;
        uint4 q0 = make_uint4(0u, 0u, 0xFFFFFFFFu, 0xFFFFFFFFu), q2 = make_uint4(0u, 0u, 0u, 0u);
        double2 fp = make_double2(0.0, 0.0);
        if (valid) {
            q0 = par_plane(d, GM_PAR_IDS)[pt];
            fp = reinterpret_cast<const double2 *>(par_plane(d, GM_PAR_FP))[pt];
            q2 = par_plane(d, GM_PAR_XYZ)[pt];
        }
        /* one scan of both own lists' counts (a batch holds at most 64*26 of each) */
        const uint32_t packed = (uint32_t)__popc(mI) << 16 | (uint32_t)__popc(mB);
        const uint32_t inclIB = wave_incl_scan(packed), ex = inclIB - packed, bt = __shfl(inclIB, 63, 64);
        oI[lane] = run[GM_RW_I] + (ex >> 16);
        oB[lane] = run[GM_RW_B] + (ex & 0xFFFFu);
        sI[lane] = mI;
        sB[lane] = mB;
        sq0[lane] = q0;
        sq2[lane] = q2;
        sfin[lane] = fp.x;
        sP[lane] = fp.y;
        /* this parent's winners at their place in the flat list, by rank */
        const uint32_t nw = list_attempts(mI | mB | mH, wl);
        for (uint32_t w0 = 0; w0 < nw; w0 += 64) {
            const uint32_t w = w0 + lane;
            const bool on = w < nw;
            const uint32_t e = on ? wl[w] : 0u, j = e & 0xFFu, r = e >> 8, bit = 1u << r;
            const uint4 pq0 = sq0[j], pq2 = sq2[j];
            RgTarget o;
            o.khi = 0u;
            o.hidx = GM_NHALO;
            if (on) rg_target(d, box, pq2.w, pq2.x, pq2.y, pq2.z, (int)r, o);
            /* the list is in the order of the parents and ranks: a parked winner's rank
             * in its halo is those of the halo before it */
            uint32_t hrank = 0;
            if (__any(o.hidx < GM_NHALO)) {
#pragma unroll
                for (uint32_t h = 0; h < GM_NHALO; h++) {
                    const uint64_t m = __ballot(o.hidx == h);
                    if (o.hidx == h) hrank = run[GM_RW_H0 + h] + lanemask_lt_count(m);
                    run[GM_RW_H0 + h] += (uint32_t)__popcll(m);
                }
            }
            if (!on) continue;
            const uint32_t t = cell_of(d, o.x, o.y, o.z);
            const uint32_t g = d.cell[t].y;
            /* the rank in the destination list, and that list's tables: the block's
             * own two lists' from LDS, a halo's receiving list's from memory */
            uint32_t rank, ix;
            if (o.khi) {
                const uint32_t q = o.dl >> 1, nbi = (o.khi >> 28) & 7u;
                rank = d.L.hoff[q * GM_NHALO + nbi] + (hrank - srs[GM_RW_H0 + o.hidx]);
                ix = 2u;
            } else if (o.dl & 1u) {
                rank = oB[j] - srs[GM_RW_B] + (uint32_t)__popc(sB[j] & (bit - 1u));
                ix = 1u;
            } else {
                rank = oI[j] - srs[GM_RW_I] + (uint32_t)__popc(sI[j] & (bit - 1u));
                ix = 0u;
            }
            const uint32_t l = o.dl;
            uint32_t rl, rb, no, cp, bs;
            if (ix < 2u) {
                rl = sL[ix][0]; rb = sL[ix][1]; no = sL[ix][2]; cp = sL[ix][3]; bs = sL[ix][4];
            } else {
                rl = d.L.rlen[l]; rb = d.L.rbase[l]; no = d.L.nold[l]; cp = d.L.cap[l]; bs = d.L.base[l];
            }
            const uint32_t rel = rank < rl ? d.L.rbuf[rb + rank] : no + (rank - rl);
            if (rel >= cp) {
                atomicOr(&st->err, (l & 1u) ? GM_ERRF_BORDER_FULL : GM_ERRF_INSIDE_FULL);
                continue;
            }
            const NewCell nc = new_cell(d, pp, A, k, sfin[j], sP[j], pq0, r, g, o.khi != 0u);
            one |= nc.one;
            put_cell(d, k, nc, pq0, t, g, o.x, o.y, o.z, bs + rel);
        }
        run[GM_RW_I] += bt >> 16;
        run[GM_RW_B] += bt & 0xFFFFu;
        __syncthreads();
    }
    if (need_one && __any(one) && lane == 0) agent_store(&st->pone, 1u);
}

/* The block that finds the others in use done ends the step (step_tail), where a launch
 * of its own took 4 us and a gap, and with `out` the window.  What it needs of the
 * other blocks they change by device atomics alone. */
__global__ void __launch_bounds__(64) k_rg_commit(GmDev d, GmPParams pp, GmSweepArgs A, GmWindow w, uint32_t *out) {
    if (d.st->halt) {
        if (out && blockIdx.x == 0) stats_to_host(d, w.top_pos, out);
        return;
    }
    const uint32_t used = d.L.bstart[d.nreg], n = used ? used : 1u;
    if (blockIdx.x >= n) return;
    rg_commit_step(d, pp, A, w.need_one);
    __builtin_amdgcn_s_waitcnt(0);
    uint32_t t = 0;
    if (threadIdx.x == 0) t = atomicAdd(&d.st->ticket, 1u);
    if (rdlane(t, 0u) != n - 1u) return;
    if (threadIdx.x == 0) agent_store(&d.st->ticket, 0u);
    step_tail(d, w);
    if (!out) return;
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    stats_to_host(d, w.top_pos, out);
}

__global__ void __launch_bounds__(64) k_rg_window_end(GmDev d, uint32_t top_pos, uint32_t *out) { stats_to_host(d, top_pos, out); }

hipError_t gm_launch_rg_window_end(const GmDev &d, const GmWindow &w, GmStats *out, hipStream_t s) {
    k_rg_window_end<<<1, 64, 0, s>>>(d, w.top_pos, reinterpret_cast<uint32_t *>(out));
    return hipGetLastError();
}

hipError_t gm_launch_rg_infect(const GmDev &d, const GmPParams &pp, const GmSweepArgs &a, uint32_t parents_upper,
                               const GmWindow &w, GmStats *out, hipStream_t s, hipEvent_t *ev) {
    hipError_t e;
    if ((e = mark(ev, 4, s)) != hipSuccess) return e;
    const uint32_t nb = rg_infect_blocks(d, parents_upper), nrec = rg_sweep_blocks(d, a);
    if ((e = mark(ev, 5, s)) != hipSuccess) return e;
    k_rg_decide<<<nrec + nb, 64, 0, s>>>(d, nrec, w.top_pos);
    if ((e = mark(ev, 6, s)) != hipSuccess) return e;
    k_rg_decide_scan<<<1, 1024, 0, s>>>(d, nb);
    if ((e = mark(ev, 7, s)) != hipSuccess || (e = mark(ev, 8, s)) != hipSuccess) return e;
    GmSweepArgs A = a;
    A.reanchor = 0;
    k_rg_commit<<<nb, 64, 0, s>>>(d, pp, A, w, reinterpret_cast<uint32_t *>(out));
    if ((e = mark(ev, 9, s)) != hipSuccess) return e;
    return hipGetLastError();
}
